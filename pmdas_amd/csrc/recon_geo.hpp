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

// f(t) for the entries t of a table of n that thread `tid` of `threads` takes.
template <typename F>
MDAS_GEO void each_entry(long long n, long long tid, long long threads, F f) {
    for (long long t = tid; t < n; t += threads) f(t);
}

}  // namespace mdas
