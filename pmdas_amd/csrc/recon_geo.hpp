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

// f(t) for the entries t of a table of n that thread `tid` of `threads` takes.
template <typename F>
MDAS_GEO void each_entry(long long n, long long tid, long long threads, F f) {
    for (long long t = tid; t < n; t += threads) f(t);
}

}  // namespace mdas
