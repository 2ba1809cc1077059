// Reconstruction: box-filter of the leaves into pixels (kdgrid.cu:483-582),
// done as a deterministic gather instead of the reference's float atomics.
//
//  1. k_recon_prep: one coalesced pass over the leaves writes a 32-byte
//     record per leaf (xy box, mean value, volume) and counts the pixel tiles
//     each leaf's span touches.
//  2. k_recon_emit: every leaf emits one 64-bit key per tile,
//         key = morton2(tile_x, tile_y) << 32 | leaf index,
//     in leaf order (offsets from the chunks' counts).
//  3. radix_sort_keys: stable LSD radix sort (digits of up to 10 bits,
//     LDS-staged scatter) on the Morton bits only; since keys are emitted in leaf order
//     the result is the total 64-bit order.
//  4. k_tile_ranges: start / end of every tile's key segment.
//  5. k_gather: a group of 16 or 64 lanes owns a tile of 16 or 64 pixels,
//     walks the tile's leaf records in index order (staged in LDS) and every
//     lane accumulates its pixel.  Each contribution is computed with the
//     reference's own expressions, including its accumulated pixel bounds
//     (pMax += step), so a pixel is the sum of its contributions in leaf
//     index order.
#include <algorithm>
#include <cmath>

#include "mdas_leaf.hpp"
#include "recon_geo.hpp"

#pragma clang fp contract(off)

namespace mdas {

static const int kReconChunks = 4096;  // most leaf chunks of the record and key kernels
static int recon_chunks(const Grid& g) { return std::min(g.chunks(), kReconChunks); }
static const int kSortKeysPerThread = 16;  // scatter tile: 4096 keys staged in LDS (8192: slower)

__device__ __forceinline__ void record_span(const float4& q0, const ReconGeo& G, int& x0, int& x1,
                                            int& y0, int& y1) {
    pixel_span(q0.x, q0.y, q0.z, q0.w, G, x0, x1, y0, y1);
}

// Keys counted by each of the reconstruction's chunks (the passes' partials are
// free between passes).
__device__ __forceinline__ int* key_counts(const DevGrid& a) { return reinterpret_cast<int*>(a.part); }

// Record of leaf i: q0 = (mn0, mx0, mn1, mx1), q1 = (mean value, volume).
// The mean is the slot-order sum times 1/n (kdgrid.cu:510-518,
// vec_math.h:492-496); the pixel span and the xy area are recomputed from q0
// by whoever needs them, with the same operations.
template <int D>
__global__ __launch_bounds__(256) void k_recon_prep(DevGrid a, ReconGeo G, float4* rrec) {
    __shared__ int red[4];
    const int L = leaf_total(a);
    int beg, end;
    chunk_range(L, gridDim.x, blockIdx.x, beg, end);
    int c = 0;
    for (int i = beg + threadIdx.x; i < end; i += 256) {
        int4 id4;
        float mn[D], mx[D];
        load_leaf<D>(a, i, leaf_count(a, i), id4, mn, mx);
        const int ids[4] = {id4.x, id4.y, id4.z, id4.w};
        // all four loads in flight at once; an empty slot reads sample 0
        float vx[4], vy[4], vz[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float* v = a.values + (size_t)(ids[q] >= 0 ? ids[q] : 0) * 3;
            vx[q] = v[0];
            vy[q] = v[1];
            vz[q] = v[2];
        }
        float sx = 0.0f, sy = 0.0f, sz = 0.0f;
        int n = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (ids[q] >= 0) {
                sx += vx[q];
                sy += vy[q];
                sz += vz[q];
                ++n;
            }
        const float inv = 1.0f / (float)n;
        float vol = 1.0f;
#pragma unroll
        for (int d = 0; d < D; ++d) vol *= (mx[d] - mn[d]);
        const float4 q0 = make_float4(mn[0], mx[0], mn[1], mx[1]);
        int x0, x1, y0, y1;
        record_span(q0, G, x0, x1, y0, y1);
        c += tiles_of(x0, x1, y0, y1, G);
        float4* r = rrec + (size_t)i * 2;
        r[0] = q0;
        r[1] = make_float4(sx * inv, sy * inv, sz * inv, vol);
    }
    c = wave_sum(c);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) key_counts(a)[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// Total of the counted keys -> n_keys.  A total beyond the key buffer
// (cap_keys) is recorded in recon_overflow and leaves n_keys = 0, so that no
// later kernel reads or writes past the buffer.
__device__ __forceinline__ bool keys_fit(const DevGrid& a, int total, long long cap_keys, bool lead) {
    const bool over = (long long)total > cap_keys;
    if (lead) {
        a.cnt->n_keys = over ? 0 : total;
        a.cnt->recon_overflow = over ? total : 0;
    }
    return !over;
}
// For a host that sizes the buffers from the count.
__global__ __launch_bounds__(256) void k_count_keys(DevGrid a, int chunks) {
    __shared__ int lds[4];
    int c = 0, total;
    for (int k = threadIdx.x; k < chunks; k += 256) c += key_counts(a)[k];
    block_exscan(c, lds, total);
    keys_fit(a, total, 0x7fffffff, threadIdx.x == 0);
}

// Every workgroup sums the chunks' counts for itself (at most kReconChunks, 16
// coalesced loads a thread: about 1 us in place of a scan kernel of 7 and its
// launch).  Also clears the tiles' ranges for k_tile_ranges.
__global__ __launch_bounds__(256) void k_recon_emit(DevGrid a, ReconGeo G, const float4* rrec,
                                                    unsigned long long* keys, long long cap_keys,
                                                    int* tstart, int* tend) {
    __shared__ int lds[4];
    each_entry(tile_entries(G), blockIdx.x * 256ll + threadIdx.x, gridDim.x * 256ll,
               [&](long long t) { tstart[t] = tend[t] = 0; });
    const int L = leaf_total(a);
    int beg, end, base, first_end;
    chunk_range(L, gridDim.x, blockIdx.x, beg, end);
    if (beg >= end && blockIdx.x > 0) return;
    chunk_range(L, gridDim.x, 0, base, first_end);
    const int chunks = first_end > 0 ? (L + first_end - 1) / first_end : 0;  // those that hold leaves
    int before = 0, after = 0, total;
    for (int k = threadIdx.x; k < chunks; k += 256) {
        const int c = key_counts(a)[k];
        before += k < (int)blockIdx.x ? c : 0;
        after += k < (int)blockIdx.x ? 0 : c;
    }
    block_exscan(before, lds, base);
    block_exscan(after, lds, total);
    if (!keys_fit(a, base + total, cap_keys, blockIdx.x == 0 && threadIdx.x == 0)) return;
    for (int t0 = beg; t0 < end; t0 += 256) {
        const int i = t0 + threadIdx.x;
        int x0 = 0, x1 = 0, y0 = 0, y1 = 0, c = 0;
        if (i < end) {
            record_span(rrec[(size_t)i * 2], G, x0, x1, y0, y1);
            c = tiles_of(x0, x1, y0, y1, G);
        }
        int off = base + block_exscan(c, lds, total);
        if (c > 0) {
            for (int ty = y0 >> G.lh; ty <= (y1 - 1) >> G.lh; ++ty)
                for (int tx = x0 >> G.lw; tx <= (x1 - 1) >> G.lw; ++tx)
                    keys[off++] = ((unsigned long long)morton2(tx, ty) << 32) | (unsigned)i;
        }
        base += total;
    }
}

// ---------------------------------------------------------- device scan --
// Exclusive scan of n <= 1024*1024 unsigned ints in place: block sums, then the
// block-local scans with their offsets.
__device__ __forceinline__ unsigned block_scan_u32(unsigned v, unsigned* ls, unsigned& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    unsigned x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        unsigned y = (unsigned)__shfl_up((int)x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) ls[w] = x;
    __syncthreads();
    unsigned pre = 0;
    total = 0;
    for (int k = 0; k < 16; ++k) {
        if (k < w) pre += ls[k];
        total += ls[k];
    }
    __syncthreads();
    return pre + x - v;
}

__global__ __launch_bounds__(1024) void k_scan_reduce(const unsigned* data, int n, unsigned* sums) {
    __shared__ unsigned ls[16];
    const int i = blockIdx.x * 1024 + threadIdx.x;
    unsigned total;
    (void)block_scan_u32(i < n ? data[i] : 0u, ls, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Every workgroup adds up the block sums before its own (at most 1024, one
// load a thread).
__global__ __launch_bounds__(1024) void k_scan_down(unsigned* data, int n, const unsigned* sums) {
    __shared__ unsigned ls[16];
    const int i = blockIdx.x * 1024 + threadIdx.x;
    unsigned before, total;
    (void)block_scan_u32(threadIdx.x < blockIdx.x ? sums[threadIdx.x] : 0u, ls, before);
    const unsigned ex = block_scan_u32(i < n ? data[i] : 0u, ls, total);
    if (i < n) data[i] = before + ex;
}

// ------------------------------------------------------------ radix sort --
// Stable LSD radix sort of 64-bit keys over bits [shift, shift+BITS) per
// pass, BITS chosen per sort so the Morton bits take as few passes as
// possible (at most 10 bits a pass).  Reduce-then-scan: per-workgroup digit
// histograms, one exclusive scan over (digit, workgroup), then a scatter in
// which every workgroup ranks a tile of up to 4096 keys by digit, stages it in
// LDS in digit order and writes each digit run contiguously -- runs of 8 keys
// on average at 512 digits, where a 256-key tile would leave most keys alone
// in their line.  A wave ranks its quarter of the tile, 64 keys at a time, by
// ballots against counters of its own; the waves meet once per tile (meeting
// three times per 256 keys, as before, made the ranking the larger part:
// 26 M keys in 8-bit passes 139 -> 115 us each, 1 M keys 16.8 -> 9.0).
template <int BITS>
__global__ __launch_bounds__(256) void k_rs_hist(const unsigned long long* keys, const int* n_ptr,
                                                 int shift, unsigned* hist) {
    constexpr int NB = 1 << BITS;
    __shared__ unsigned h[NB];
    const int n = *n_ptr;
    for (int d = threadIdx.x; d < NB; d += 256) h[d] = 0;
    __syncthreads();
    int beg, end;
    chunk_range(n, gridDim.x, blockIdx.x, beg, end);
    for (int i = beg + threadIdx.x; i < end; i += 256)
        atomicAdd(&h[(unsigned)(keys[i] >> shift) & (unsigned)(NB - 1)], 1u);
    __syncthreads();
    for (int d = threadIdx.x; d < NB; d += 256) hist[d * gridDim.x + blockIdx.x] = h[d];
}

template <int BITS>
__global__ __launch_bounds__(256) void k_rs_scatter(const unsigned long long* in,
                                                    unsigned long long* out, const int* n_ptr,
                                                    int shift, const unsigned* hist) {
    constexpr int NB = 1 << BITS;
    constexpr int R = NB > 256 ? NB / 256 : 1;  // digits per thread in the tile scan
    constexpr int KPT = kSortKeysPerThread;
    constexpr int TILE = 256 * KPT;
    __shared__ unsigned base[NB];   // where the workgroup's next key of a digit goes
    __shared__ int wcnt[4][NB];     // keys of a digit per wave, then its offset in the tile
    __shared__ int toff[NB];        // the digit's offset in the tile
    __shared__ int scr[4];
    __shared__ unsigned long long stage[TILE];
    const int n = *n_ptr;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int beg, end;
    chunk_range(n, gridDim.x, blockIdx.x, beg, end);
    if (beg >= end) return;
    for (int d = threadIdx.x; d < NB; d += 256) base[d] = hist[d * gridDim.x + blockIdx.x];
    for (int t0 = beg; t0 < end; t0 += TILE) {
        const int nvalid = min(TILE, end - t0);
        const int subs = (nvalid + 255) / 256;      // rounds of 64 keys per wave
        const int first = w * subs * 64 + lane;     // this lane's key of round s: first + 64 s
        unsigned long long k[KPT];
#pragma unroll
        for (int s = 0; s < KPT; ++s)
            k[s] = s < subs && first + 64 * s < nvalid ? in[t0 + first + 64 * s] : 0ull;
        for (int q = 0; q < 4; ++q)
            for (int d = threadIdx.x; d < NB; d += 256) wcnt[q][d] = 0;
        __syncthreads();
        // rank of each key among the wave's keys of its digit, in input order
        int rk[KPT];
#pragma unroll
        for (int s = 0; s < KPT; ++s) {
            if (s < subs) {  // uniform
                const bool valid = first + 64 * s < nvalid;
                const unsigned d = (unsigned)(k[s] >> shift) & (unsigned)(NB - 1);
                unsigned long long m = __ballot(valid);
#pragma unroll
                for (int b = 0; b < BITS; ++b) {
                    const bool bit = (d >> b) & 1u;
                    const unsigned long long bal = __ballot(bit);
                    m &= bit ? bal : ~bal;
                }
                const int below = lanes_below(m), before = wcnt[w][d];
                rk[s] = before + below;
                wave_sync_lds();
                if (valid && below == 0) wcnt[w][d] = before + __popcll(m);
                wave_sync_lds();
            }
        }
        __syncthreads();
        // offsets of the digits in the tile, then of each wave's keys
        {
            int loc[R], sum = 0;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int dd = (int)threadIdx.x * R + r;
                loc[r] = dd < NB ? wcnt[0][dd] + wcnt[1][dd] + wcnt[2][dd] + wcnt[3][dd] : 0;
                sum += loc[r];
            }
            int all;
            int ex = block_exscan(sum, scr, all);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int dd = (int)threadIdx.x * R + r;
                if (dd < NB) {
                    toff[dd] = ex;
                    int o = ex;
                    for (int q = 0; q < 4; ++q) {
                        const int c = wcnt[q][dd];
                        wcnt[q][dd] = o;
                        o += c;
                    }
                    ex += loc[r];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KPT; ++s) {
            if (s < subs && first + 64 * s < nvalid) {
                const unsigned d = (unsigned)(k[s] >> shift) & (unsigned)(NB - 1);
                stage[wcnt[w][d] + rk[s]] = k[s];
            }
        }
        __syncthreads();
        // the tile in digit order: each digit's run goes to its own range
        for (int p = threadIdx.x; p < nvalid; p += 256) {
            const unsigned long long kk = stage[p];
            const unsigned dd = (unsigned)(kk >> shift) & (unsigned)(NB - 1);
            out[base[dd] + (p - toff[dd])] = kk;
        }
        __syncthreads();
        for (int dd = threadIdx.x; dd < NB; dd += 256)
            base[dd] += (dd + 1 < NB ? toff[dd + 1] : nvalid) - toff[dd];
        __syncthreads();
    }
}

static void scan_u32(unsigned* data, int n, unsigned* sums, hipStream_t st) {
    const int nb = (n + 1023) / 1024;
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(1024), 0, st, data, n, sums);
    hipLaunchKernelGGL(k_scan_down, dim3(nb), dim3(1024), 0, st, data, n, sums);
}

template <int BITS>
static void sort_pass(Grid& g, unsigned* rs_hist, const unsigned long long* a, unsigned long long* b,
                      int sh, int blocks, hipStream_t st) {
    const int* n_ptr = &g.dev.cnt->n_keys;
    const int nh = (1 << BITS) * blocks;
    kbeg(g, st, "k_rs_hist");
    hipLaunchKernelGGL(k_rs_hist<BITS>, dim3(blocks), dim3(256), 0, st, a, n_ptr, sh, rs_hist);
    kend(g, st);
    kbeg(g, st, "k_rs_scan");
    scan_u32(rs_hist, nh, rs_hist + nh, st);
    kend(g, st);
    kbeg(g, st, "k_rs_scatter");
    hipLaunchKernelGGL(k_rs_scatter<BITS>, dim3(blocks), dim3(256), 0, st, a, b, n_ptr, sh,
                       rs_hist);
    kend(g, st);
}

// Sorts keys[0, n) by bits [lo, hi) in ceil((hi - lo) / 10) passes of equal
// digit width; returns the buffer holding the result.
static unsigned long long* radix_sort_keys(Grid& g, ReconBufs& rb, int lo, int hi, double expected,
                                           hipStream_t st) {
    unsigned long long* a = rb.keys;
    unsigned long long* b = rb.keys_alt;
    g.recon_sort_passes = 0;
    const int total = hi - lo;
    if (total <= 0) return a;
    const int bits = sort_digit(total), blocks = sort_blocks(expected, bits);
    g.recon_sort_blocks = blocks;
    for (int sh = lo; sh < hi; sh += bits) {
        switch (bits) {
        case 4: sort_pass<4>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        case 5: sort_pass<5>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        case 6: sort_pass<6>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        case 7: sort_pass<7>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        case 8: sort_pass<8>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        case 9: sort_pass<9>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        default: sort_pass<10>(g, rb.rs_hist, a, b, sh, blocks, st); break;
        }
        g.recon_sort_passes++;
        g.recon_sort_bits = bits;
        unsigned long long* t = a;
        a = b;
        b = t;
    }
    return a;
}

__global__ __launch_bounds__(256) void k_tile_ranges(const unsigned long long* keys,
                                                     const int* n_ptr, int* start, int* end) {
    const int n = *n_ptr;
    for (int p = blockIdx.x * 256 + threadIdx.x; p < n; p += gridDim.x * 256) {
        const unsigned t = (unsigned)(keys[p] >> 32);
        if (p == 0 || (unsigned)(keys[p - 1] >> 32) != t) start[t] = p;
        if (p == n - 1 || (unsigned)(keys[p + 1] >> 32) != t) end[t] = p + 1;
    }
}

// ---------------------------------------------------------------- gather --
// GS = pixels per tile (16 or 64); a wave holds 64/GS tiles and takes GS
// records of each at a time, a record per lane, then a pixel per lane.  What
// bounds it is arithmetic (a record covers 2 to 5 pixels of a tile), so all
// that depends on the record and a column or a row only is done once, by the
// record's lane: the walk of the accumulated pixel bounds (kdgrid.cu:532-576)
// and the overlap with each of its columns and rows, kept in LDS (a pixel's
// lane did both for itself, per record: 920 us at 1080p for 26 M records, now
// 525; 640x360 48 -> 25 us), and the lanes of the
// pixels it overlaps get its bit with LDS atomics.  Where a record overlaps more
// than kOrPixels (7) the atomics of the busiest lane cost more than a ballot
// for each column and each row: a pixel's records are its column's that are
// also its row's (up to kBallots columns and rows: 640x360 27 -> 22.7 us, 6D
// 960x540 181 -> 169; ballots everywhere made 3D 256x256 27 -> 34 us, and 64x1
// tiles 540 -> 690).  A pixel then adds its records'
// contributions in index order: two overlaps, a product and a quotient each.
static const int kOrPixels = 7, kBallots = 24;
// Dynamic LDS of one wave: means and volumes, coverage words, xy areas, and
// the overlaps, TW + TH per record (an odd stride spreads them over the banks).
__host__ __device__ constexpr int gather_stride(int TW, int TH) { return (TW + TH) | 1; }
__host__ __device__ constexpr int gather_lds(int TW, int TH) { return 64 * (16 + 8 + 4 + 4 * gather_stride(TW, TH)); }

// Overlap of [mn, mx] with the pixels [p0, p1) of an axis, of which the span
// starts at s0 (at coordinate lo), into ov[p - base]; a bit per positive one.
__device__ __forceinline__ unsigned long long axis_overlaps(float mn, float mx, int s0, float lo, float step,
                                                            int p0, int p1, int base, float* ov) {
    float pMin = lo, pMax = lo + step;
    for (int q = s0; q < p0; ++q) {  // exactly as kdgrid.cu:536-576 walks them
        pMin = pMax;
        pMax += step;
    }
    unsigned long long bits = 0ull;
    for (int q = p0; q < p1; ++q) {
        const float d = fminf(pMax, mx) - fmaxf(pMin, mn);
        ov[q - base] = d;
        if (d > 0.0f) bits |= 1ull << (q - base);
        pMin = pMax;
        pMax += step;
    }
    return bits;
}

template <int GS>
__global__ __launch_bounds__(256) void k_gather(ReconGeo G, const float4* __restrict__ rrec,
                                                const unsigned long long* __restrict__ keys,
                                                const int* __restrict__ tstart,
                                                const int* __restrict__ tend, float4* pixels) {
    extern __shared__ float4 gather_mem[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int stride = gather_stride(G.TW, G.TH);
    char* mem = reinterpret_cast<char*>(gather_mem) + w * gather_lds(G.TW, G.TH);
    float4* mean = reinterpret_cast<float4*>(mem);
    unsigned long long* covers = reinterpret_cast<unsigned long long*>(mem + 64 * 16);
    float* area = reinterpret_cast<float*>(mem + 64 * 24);
    float* ov = area + 64;
    const int grp = lane / GS, gl = lane % GS;      // tile within the wave, lane within the tile
    const int tile = (blockIdx.x * (blockDim.x >> 6) + w) * (64 / GS) + grp;
    const int ntiles = G.tilesX * G.tilesY;
    const bool live = tile < ntiles;
    const int tx = live ? tile % G.tilesX : 0, ty = live ? tile / G.tilesX : 0;
    const int pc = gl & (G.TW - 1), pr = gl >> G.lw;       // this lane's pixel in the tile
    const int ox = tx * G.TW, oy = ty * G.TH;
    int s0 = 0, s1 = 0;
    if (live) {
        const unsigned code = morton2(tx, ty);
        s0 = tstart[code];
        s1 = tend[code];
    }
    // rounds of GS records until the longest tile of the wave is done; the
    // records of round rd + 1 and the keys of round rd + 2 are loaded while
    // round rd is accumulated
    int rounds = (s1 - s0 + GS - 1) / GS;
#pragma unroll
    for (int o = GS; o < 64; o <<= 1) rounds = max(rounds, __shfl_xor(rounds, o, 64));
    float accx = 0.0f, accy = 0.0f, accz = 0.0f;
    const int gbase = grp * GS;
    auto nrec_of = [&](int rd) { return max(0, min(GS, s1 - (s0 + rd * GS))); };
    float4 c0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), c1 = c0;  // records of the round to stage
    if (gl < nrec_of(0)) {
        const int i = (int)(unsigned)(keys[s0 + gl] & 0xffffffffull);
        c0 = rrec[(size_t)i * 2];
        c1 = rrec[(size_t)i * 2 + 1];
    }
    unsigned long long knext = gl < nrec_of(1) ? keys[s0 + GS + gl] : 0ull;
    for (int rd = 0; rd < rounds; ++rd) {
        unsigned long long cols = 0ull, rows = 0ull;  // of the tile that this lane's record overlaps
        if (gl < nrec_of(rd)) {
            int x0, x1, y0, y1;
            record_span(c0, G, x0, x1, y0, y1);
            float* o = ov + lane * stride;
            cols = axis_overlaps(c0.x, c0.y, x0, (float)x0 * G.sX / G.fW, G.stepX, max(x0, ox),
                                 min(x1, ox + G.TW), ox, o);
            rows = axis_overlaps(c0.z, c0.w, y0, (float)y0 * G.sY / G.fH, G.stepY, max(y0, oy),
                                 min(y1, oy + G.TH), oy, o + G.TW);
            mean[lane] = c1;
            area[lane] = (c0.y - c0.x) * (c0.w - c0.z);
        }
        wave_sync_lds();
        if (gl < nrec_of(rd + 1)) {
            const int i = (int)(unsigned)(knext & 0xffffffffull);
            c0 = rrec[(size_t)i * 2];
            c1 = rrec[(size_t)i * 2 + 1];
        }
        knext = gl < nrec_of(rd + 2) ? keys[s0 + (rd + 2) * GS + gl] : 0ull;
        // the round's records that overlap this lane's pixel, bit j for the
        // tile's record j
        unsigned long long cov = 0ull;
        if (G.TW + G.TH <= kBallots && __any(__popcll(cols) * __popcll(rows) > kOrPixels)) {
            // the records of the pixel's column and those of its row
            unsigned long long rcov = 0ull;
            for (int c = 0; c < G.TW; ++c) {
                const unsigned long long b = __ballot((cols >> c) & 1ull);
                cov = pc == c ? b : cov;
            }
            for (int r = 0; r < G.TH; ++r) {
                const unsigned long long b = __ballot((rows >> r) & 1ull);
                rcov = pr == r ? b : rcov;
            }
            cov &= rcov;
            if (GS < 64) cov = (cov >> gbase) & ((1ull << (GS & 63)) - 1ull);
        } else {
            unsigned long long own = 0ull;  // the tile's pixels this lane's record overlaps
            while (rows != 0ull) {
                own |= cols << (__builtin_ctzll(rows) << G.lw);
                rows &= rows - 1ull;
            }
            covers[lane] = 0ull;
            wave_sync_lds();
            while (own != 0ull) {
                atomicOr(&covers[gbase + __builtin_ctzll(own)], 1ull << gl);
                own &= own - 1ull;
            }
            wave_sync_lds();
            cov = covers[lane];
        }
        // in index order (the other records add nothing): the loop runs as
        // often as the most-covered pixel of the wave needs
        while (cov != 0ull) {
            const int j = gbase + __builtin_ctzll(cov);
            cov &= cov - 1ull;
            const float dx = ov[j * stride + pc], dy = ov[j * stride + G.TW + pr];
            const float4 m = mean[j];
            const float v = dx * dy * m.w / area[j];
            accx += (m.x * v) * G.invPixArea;
            accy += (m.y * v) * G.invPixArea;
            accz += (m.z * v) * G.invPixArea;
        }
        wave_sync_lds();
    }
    const int px = ox + pc, py = oy + pr;
    if (live && px < G.W && py < G.H) pixels[(size_t)py * G.W + px] = make_float4(accx, accy, accz, 0.0f);
}

// -------------------------------------------------------- scatter (atomics) --
// kdgrid.cu:483-582 as written: one thread per leaf, float atomics per pixel.
template <int D>
__global__ __launch_bounds__(256) void k_scatter(DevGrid a, ReconGeo G, float4* pixels) {
    const int L = leaf_total(a);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < L; i += gridDim.x * 256) {
        int4 id4;
        float mn[D], mx[D];
        load_leaf<D>(a, i, leaf_count(a, i), id4, mn, mx);
        const int ids[4] = {id4.x, id4.y, id4.z, id4.w};
        float sx = 0.0f, sy = 0.0f, sz = 0.0f;
        int n = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (ids[q] >= 0) {
                const float* v = a.values + (size_t)ids[q] * 3;
                sx += v[0];
                sy += v[1];
                sz += v[2];
                ++n;
            }
        const float inv = 1.0f / (float)n;
        sx *= inv;
        sy *= inv;
        sz *= inv;
        float vol = 1.0f;
#pragma unroll
        for (int d = 0; d < D; ++d) vol *= (mx[d] - mn[d]);
        int x0, x1, y0, y1;
        pixel_span(mn[0], mx[0], mn[1], mx[1], G, x0, x1, y0, y1);
        float pMinY = (float)y0 * G.sY / G.fH;
        float pMaxY = pMinY + G.stepY;
        for (int y = y0; y < y1; ++y) {
            float pMinX = (float)x0 * G.sX / G.fW;
            float pMaxX = pMinX + G.stepX;
            for (int x = x0; x < x1; ++x) {
                const float clox = fmaxf(pMinX, mn[0]);
                const float chix = fminf(pMaxX, mx[0]);
                const float cloy = fmaxf(pMinY, mn[1]);
                const float chiy = fminf(pMaxY, mx[1]);
                if (clox < chix && cloy < chiy) {
                    const float v = (chix - clox) * (chiy - cloy) * vol / ((mx[0] - mn[0]) * (mx[1] - mn[1]));
                    float* p = (float*)(pixels + (size_t)y * G.W + x);
                    atomicAdd(p, (sx * v) * G.invPixArea);
                    atomicAdd(p + 1, (sy * v) * G.invPixArea);
                    atomicAdd(p + 2, (sz * v) * G.invPixArea);
                }
                pMinX = pMaxX;
                pMaxX += G.stepX;
            }
            pMinY = pMaxY;
            pMaxY += G.stepY;
        }
    }
}

// ----------------------------------------------------------------- bytes --
// helpers.h:35-66: clamp, sRGB (pow with exponent 1/2.4), 8-bit quantise.
__device__ __forceinline__ unsigned char quantize8(float x) {
    x = fmaxf(0.0f, fminf(x, 1.0f));
    unsigned v = (unsigned)(x * 256.0f);
    return (unsigned char)min(v, 255u);
}

__global__ __launch_bounds__(256) void k_bytes(const float4* px, uchar4* out, long long n) {
    const float invGamma = 1.0f / 2.4f;
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float4 c = px[i];
        const float in[3] = {c.x, c.y, c.z};
        unsigned char o[3];
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
            const float x = fmaxf(0.0f, fminf(in[ch], 1.0f));
            const float p = powf_mdas(x, invGamma);
            const float s = x < 0.0031308f ? 12.92f * x : 1.055f * p - 0.055f;
            o[ch] = quantize8(s);
        }
        out[i] = make_uchar4(o[0], o[1], o[2], 255);
    }
}

// ------------------------------------------------------------ launchers --
static ReconGeo make_geo(const Grid& g, int W, int H) {
    return recon_geo(W, H, g.sX, g.sY, g.tile_w, g.tile_h);
}

#define MDAS_DISPATCH_D(D_, STMT)                      \
    switch (D_) {                                      \
    case 3: { constexpr int DD = 3; STMT; } break;     \
    case 4: { constexpr int DD = 4; STMT; } break;     \
    case 5: { constexpr int DD = 5; STMT; } break;     \
    case 6: { constexpr int DD = 6; STMT; } break;     \
    default: return hipErrorInvalidValue;              \
    }

static hipError_t grow_keys(ReconBufs& rb, long long cap) {
    if (rb.keys) (void)hipFree(rb.keys);
    if (rb.keys_alt) (void)hipFree(rb.keys_alt);
    rb.keys = rb.keys_alt = nullptr;
    rb.keys_cap = 0;
    hipError_t e = hipMalloc(&rb.keys, sizeof(unsigned long long) * (size_t)cap);
    if (e == hipSuccess) e = hipMalloc(&rb.keys_alt, sizeof(unsigned long long) * (size_t)cap);
    if (e != hipSuccess) return e;
    rb.keys_cap = cap;
    return hipSuccess;
}

// Upper bound on the keys one leaf emits: the tiles its pixel span can touch.
// A leaf's box is at most g.ext_x by g.ext_y in x and y (splits only shrink
// boxes), and a span of extent ext over n pixels of a sample space of size s
// holds at most floor(ext n / s) + 2 pixels (floor(mx n/s) - floor(mn n/s) + 1,
// with a margin for the rounding of the float products); p pixels starting
// anywhere in a tile of T touch at most (p + T - 2) / T + 1 tiles.
static long long tiles_per_leaf(const Grid& g, const ReconGeo& G) {
    auto axis = [](double ext, int n, double s, int T, int tiles) {
        long long p = (long long)std::floor(ext * (double)n / s * (1.0 + 1e-6) + 1e-3) + 2;
        p = std::min<long long>(p, n);
        return std::min<long long>((p + T - 2) / T + 1, tiles);
    };
    return axis(g.ext_x, G.W, G.sX, G.TW, G.tilesX) * axis(g.ext_y, G.H, G.sY, G.TH, G.tilesY);
}

static long long key_bound(const Grid& g, const ReconGeo& G) {
    return tiles_per_leaf(g, G) * std::max<long long>(g.host.n_leaves, 1);
}

// Key buffers of at most this many bytes are sized from the bound up front
// (no host round trip in the reconstruction); larger bounds (tiny initial
// grids, whose leaves span many tiles) size them from the counted keys.
static const long long kKeyBoundBytes = 8ll << 30;

static long long align256(long long b) { return (b + 255) / 256 * 256; }

long long recon_key_bound(const Grid& g, int W, int H) { return key_bound(g, make_geo(g, W, H)); }
long long recon_tiles_cap(const Grid& g, int W, int H) { return tile_entries(make_geo(g, W, H)); }

long long recon_bytes_needed(const Grid& g, int W, int H) {
    const ReconGeo G = make_geo(g, W, H);
    const long long kb = key_bound(g, G);
    if (kb > 0x7fffffffLL) return -1;
    const long long L = std::max<long long>(g.host.n_leaves, 1);
    return align256(sizeof(unsigned) * kSortHistWords) + 2 * align256(sizeof(int) * tile_entries(G)) +
           align256(sizeof(float4) * 2 * L) + 2 * align256(sizeof(unsigned long long) * kb);
}

// Sizes the grid's reconstruction buffers for the current leaf count (g.host
// is current after every call that changes the tree) and image; allocates
// only when they grow.  Sets g.recon_bounded when the key buffers hold the
// bound, i.e. the reconstruction needs no host round trip.
hipError_t recon_reserve(Grid& g, int W, int H) {
    ReconGeo G = make_geo(g, W, H);
    ReconBufs& rb = g.rb;
    const long long L = g.host.n_leaves;
    if (L > rb.rrec_cap) {
        if (rb.rrec) (void)hipFree(rb.rrec);
        rb.rrec = nullptr;
        rb.rrec_cap = 0;
        const long long cap = std::min<long long>((long long)g.cap_l, L + L / 4 + 1024);
        hipError_t e = hipMalloc(&rb.rrec, sizeof(float4) * 2 * (size_t)cap);
        if (e != hipSuccess) return e;
        rb.rrec_cap = cap;
    }
    const long long kb = key_bound(g, G);
    g.recon_bounded = kb <= 0x7fffffffLL && kb * 16 <= kKeyBoundBytes;
    if (g.recon_bounded && kb > rb.keys_cap) {
        hipError_t e = grow_keys(rb, kb);
        if (e != hipSuccess) return e;
    }
    const long long tiles = tile_entries(G);
    if (tiles > rb.tiles_cap) {
        if (rb.tile_start) (void)hipFree(rb.tile_start);
        if (rb.tile_end) (void)hipFree(rb.tile_end);
        rb.tile_start = rb.tile_end = nullptr;
        rb.tiles_cap = 0;
        hipError_t e = hipMalloc(&rb.tile_start, sizeof(int) * tiles);
        if (e == hipSuccess) e = hipMalloc(&rb.tile_end, sizeof(int) * tiles);
        if (e != hipSuccess) return e;
        rb.tiles_cap = tiles;
    }
    if (!rb.rs_hist) {
        hipError_t e = hipMalloc(&rb.rs_hist, sizeof(unsigned) * kSortHistWords);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Per-leaf records and tile counts.  Stream-ordered when the key
// buffers hold the bound; otherwise the key count is read back (a
// synchronisation) and the buffers grown to it.
hipError_t recon_prepare(Grid& g, int W, int H, hipStream_t st) {
    hipError_t e = recon_reserve(g, W, H);
    if (e != hipSuccess) return e;
    ReconGeo G = make_geo(g, W, H);
    g.recon_pixels = (long long)W * H;
    kbeg(g, st, "k_recon_prep");
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_recon_prep<DD>, dim3(recon_chunks(g)), dim3(256), 0, st,
                                            g.dev, G, g.rb.rrec));
    kend(g, st);
    if (!g.recon_bounded) {
        int nk = 0;
        hipLaunchKernelGGL(k_count_keys, dim3(1), dim3(256), 0, st, g.dev, recon_chunks(g));
        e = hipMemcpyAsync(&nk, &g.dev.cnt->n_keys, sizeof(int), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
        if (nk > g.rb.keys_cap) {
            e = grow_keys(g.rb, (long long)nk + nk / 4 + 1024);
            if (e != hipSuccess) return e;
        }
    }
    return hipGetLastError();
}

double recon_expected_keys(const Grid& g, long long leaves, int W, int H) {
    const ReconGeo G = make_geo(g, W, H);
    double e[6] = {g.ext_x, g.ext_y};
    for (int d = 2; d < g.D; ++d) e[d] = 1.0 / (double)(1 << g.b);
    return expected_keys(G, (double)leaves, (double)(1ll << (g.b * g.D + 2 * g.e)), g.D, e);
}

static bool capturing(hipStream_t st) {
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;  // the null stream cannot be captured
    return st != nullptr && hipStreamIsCapturing(st, &s) == hipSuccess && s != hipStreamCaptureStatusNone;
}

// Keys in leaf order, their sort, the tiles' key ranges and the gather, on
// the buffers of rb (records already written by k_recon_prep).
static hipError_t recon_finish(Grid& g, ReconBufs& rb, float* pixels, int W, int H, hipStream_t st,
                               hipEvent_t ev_sort0, hipEvent_t ev_sort1) {
    ReconGeo G = make_geo(g, W, H);
    kbeg(g, st, "k_recon_emit");
    hipLaunchKernelGGL(k_recon_emit, dim3(recon_chunks(g)), dim3(256), 0, st, g.dev, G, rb.rrec, rb.keys, rb.keys_cap,
                       rb.tile_start, rb.tile_end);
    kend(g, st);
    // a graph is replayed for any tree that the buffers hold; the kernels take
    // any number of keys, but few workgroups for many would take turns (captured
    // over 2048 leaves, replayed for 11 M at 1080p: 44 ms, now 1.53)
    const bool graph = capturing(st);
    // keys there can be: the bound, or the buffers where they were sized from
    // the count
    const long long bound = graph ? rb.keys_cap : std::min(key_bound(g, G), rb.keys_cap);
    if (ev_sort0) (void)hipEventRecord(ev_sort0, st);
    // the sorted keys end in keys or keys_alt by the parity of the pass
    // count; the buffers keep their roles, so a captured graph stays valid
    const double expected = recon_expected_keys(g, graph ? rb.rrec_cap : g.host.n_leaves, W, H);
    unsigned long long* sorted = radix_sort_keys(g, rb, 32, 32 + 2 * G.tbits, expected, st);
    g.keys_sorted = sorted;
    if (ev_sort1) (void)hipEventRecord(ev_sort1, st);
    kbeg(g, st, "k_tile_ranges");
    int blocks = (int)std::min<long long>((bound + 255) / 256, 8192);  // grid-stride over
    if (blocks < 1) blocks = 1;                                        // the device count
    hipLaunchKernelGGL(k_tile_ranges, dim3(blocks), dim3(256), 0, st, sorted, &g.dev.cnt->n_keys,
                       rb.tile_start, rb.tile_end);
    kend(g, st);
    const int ntiles = G.tilesX * G.tilesY;
    const int gs = G.TW * G.TH;
    // four waves a workgroup; one where their LDS would exceed 64 KB (tiles
    // of more than 48 pixels along an axis)
    const int lds = gather_lds(G.TW, G.TH), waves = 4 * lds <= 65536 ? 4 : 1;
    const int per = waves * (64 / gs);  // tiles of a workgroup
    const dim3 grid((ntiles + per - 1) / per), block(64 * waves);
    kbeg(g, st, "k_gather");
    if (gs == 64)
        hipLaunchKernelGGL(k_gather<64>, grid, block, waves * lds, st, G, rb.rrec, sorted, rb.tile_start, rb.tile_end,
                           (float4*)pixels);
    else
        hipLaunchKernelGGL(k_gather<16>, grid, block, waves * lds, st, G, rb.rrec, sorted, rb.tile_start, rb.tile_end,
                           (float4*)pixels);
    kend(g, st);
    return hipGetLastError();
}

hipError_t launch_integrate_gather(Grid& g, float* pixels, int W, int H, hipStream_t st,
                                   hipEvent_t ev_sort0, hipEvent_t ev_sort1) {
    return recon_finish(g, g.rb, pixels, W, H, st, ev_sort0, ev_sort1);
}

hipError_t recon_on_buffers(Grid& g, ReconBufs& rb, float* pixels, int W, int H, hipStream_t st) {
    ReconGeo G = make_geo(g, W, H);
    g.recon_pixels = (long long)W * H;
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_recon_prep<DD>, dim3(recon_chunks(g)), dim3(256), 0, st,
                                            g.dev, G, rb.rrec));
    return recon_finish(g, rb, pixels, W, H, st, nullptr, nullptr);
}

hipError_t launch_integrate_scatter(Grid& g, float* pixels, int W, int H, hipStream_t st) {
    ReconGeo G = make_geo(g, W, H);
    launch_fill_f32(pixels, 0.0f, 4ll * W * H, st);
    int blocks = (int)std::min<long long>(((long long)g.cap_l + 255) / 256, 8192);
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_scatter<DD>, dim3(blocks), dim3(256), 0, st, g.dev,
                                            G, (float4*)pixels));
    return hipGetLastError();
}

hipError_t launch_bytes(const float* pixels, unsigned char* out, long long n, hipStream_t st) {
    int blocks = (int)std::min<long long>((n + 255) / 256, 8192);
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_bytes, dim3(blocks), dim3(256), 0, st, (const float4*)pixels,
                       (uchar4*)out, n);
    return hipGetLastError();
}

}  // namespace mdas
