// The reconstruction's geometry: the image, its pixel tiles and what follows
// from them in counts.  Compiled by hipcc into the kernels and their launchers
// and by g++ into the CPU library of the tests, which hold the counts at sizes
// whose tables no test would want to fill.
#pragma once

#if defined(__HIPCC__)
#define MDAS_GEO __host__ __device__ inline
#else
#define MDAS_GEO inline
#endif

namespace mdas {

struct ReconGeo {
    int W, H;
    float fW, fH, sX, sY;
    float stepX, stepY;   // scale / width (kdgrid.cu:501-503)
    float invPixArea;     // 1 / ((sX*sY) / float(W*H)) (kdgrid.cu:532, vec_math.h:483-487)
    int TW, TH, tilesX, tilesY;
    int lw, lh;           // TW = 2^lw, TH = 2^lh (a tile holds 16 or 64 pixels)
    int tbits;            // Morton bits per tile axis
};

inline ReconGeo recon_geo(int W, int H, float sX, float sY, int TW, int TH) {
    ReconGeo G;
    G.W = W;
    G.H = H;
    G.fW = (float)W;
    G.fH = (float)H;
    G.sX = sX;
    G.sY = sY;
    G.stepX = sX / (float)W;
    G.stepY = sY / (float)H;
    const float pixArea = (sX * sY) / (float)(W * H);
    G.invPixArea = 1.0f / pixArea;
    G.TW = TW;
    G.TH = TH;
    G.lw = __builtin_ctz(TW);
    G.lh = __builtin_ctz(TH);
    G.tilesX = (W + TW - 1) / TW;
    G.tilesY = (H + TH - 1) / TH;
    const int m = G.tilesX > G.tilesY ? G.tilesX : G.tilesY;
    int bits = 0;
    while ((1 << bits) < m) ++bits;
    G.tbits = bits;
    return G;
}

// Entries of the tables of the tiles' key ranges, which Morton codes index:
// up to 2^32 (more than 32768 tiles along an axis), beyond an int.
MDAS_GEO long long tile_entries(const ReconGeo& G) { return 1ll << (2 * G.tbits); }

MDAS_GEO int geo_clamp(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// kdgrid.cu:524-529: pixel span [x0, x1) x [y0, y1) of a leaf box, its start
// held to the image: a tree's boxes lie inside, an uploaded state's may begin
// before the first pixel, whose tiles the span must not index (a span that
// starts past the image or ends before it is empty).
MDAS_GEO void pixel_span(float mn0, float mx0, float mn1, float mx1, const ReconGeo& G, int& x0, int& x1,
                         int& y0, int& y1) {
    x0 = geo_clamp((int)(mn0 * G.fW / G.sX), 0, G.W);
    y0 = geo_clamp((int)(mn1 * G.fH / G.sY), 0, G.H);
    const int xx = (int)(mx0 * G.fW / G.sX) + 1, yy = (int)(mx1 * G.fH / G.sY) + 1;
    x1 = xx < G.W ? xx : G.W;
    y1 = yy < G.H ? yy : G.H;
}

// Tiles that a span touches.
MDAS_GEO int tiles_of(int x0, int x1, int y0, int y1, const ReconGeo& G) {
    if (x0 >= x1 || y0 >= y1) return 0;
    return (((x1 - 1) >> G.lw) - (x0 >> G.lw) + 1) * (((y1 - 1) >> G.lh) - (y0 >> G.lh) + 1);
}

// Keys (leaves, once for each tile they touch) that a tree of `leaves` leaves
// gives, from what the host knows: the initial cells' extents and number.  A
// leaf is split along its longest axis, so one of a tree grown by 2^s has s
// halvings behind it, taken in that order; one of p by q pixels touches
// (1 + p / TW) (1 + q / TH) tiles on average.  Over 3 to 6 dimensions, sample
// spaces of the unit square and of pixels, 1 .. 8192 initial cells and 100 to
// 70000 leaves the count was 0.4 to 2.0 of this.  The keys per leaf run from 1.1
// to thousands, since at a unit square x and y are halved no sooner than time
// and lens: 354 leaves with 1.1 M keys at 1920x1080 took 7.05 ms with the sort
// launched for 1.5 keys per leaf (one workgroup), 4.75 with 1024 workgroups
// always and 0.90 with this; a 640x360 image of 314 thousand leaves is the same
// in 8 x 8 and 4 x 4 tiles.
inline double expected_keys(const ReconGeo& G, double leaves, double initial, int D, const double* extent) {
    double e[8];
    for (int d = 0; d < D; ++d) e[d] = extent[d];
    for (double n = 2.0 * initial; n <= leaves; n *= 2.0) {
        int k = 0;
        for (int d = 1; d < D; ++d)
            if (e[d] > e[k]) k = d;
        e[k] *= 0.5;
    }
    const double x = 1.0 + e[0] * G.W / G.sX / G.TW, y = 1.0 + e[1] * G.H / G.sY / G.TH;
    return leaves * (x < G.tilesX ? x : G.tilesX) * (y < G.tilesY ? y : G.tilesY);
}

// The sort's digits: ceil(bits / 10) passes of equal width, at least 4 bits.
static const int kSortMaxBits = 10;  // histograms of 1024 bins
inline int sort_digit(int bits) {
    const int passes = (bits + kSortMaxBits - 1) / kSortMaxBits, d = (bits + passes - 1) / passes;
    return d > 4 ? d : 4;
}
// Its workgroups for that many keys, at most 1024 (its kernels take any number
// of keys): half a tile of 4096 each, up to a whole one for 10-bit digits where
// every CU has one, since each brings counters for all its digits' values (a
// 640x360 image in 1 x 64 tiles, 925 thousand keys: 561 workgroups 180 us, 281
// 166 us).
static const int kSortBlocks = 1024;
inline int sort_blocks(double keys, int digit) {
    double n = keys / 2048.0;
    if (digit > 9 && n > 256.0) n = n > 512.0 ? 0.5 * n : 256.0;
    return n >= kSortBlocks ? kSortBlocks : (n <= 1.0 ? 1 : (int)n + 1);
}

// f(t) for the entries t of a table of n that thread `tid` of `threads` takes.
template <typename F>
MDAS_GEO void each_entry(long long n, long long tid, long long threads, F f) {
    for (long long t = tid; t < n; t += threads) f(t);
}

}  // namespace mdas
