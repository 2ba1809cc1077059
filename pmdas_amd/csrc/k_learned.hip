// Learned proposal: per-leaf features and labels, MLP scoring fused into the
// error pass, and the MLP's training kernels (forward on MFMA, FP32
// backward, Adam).
//
// Features of a leaf (computed whenever its plain error is, from the same
// reads): log2 extent per dimension relative to the domain (6, zero above
// D), sample count, mean / variance / min / max luminance of its samples,
// depth (splits since the initial grid), log2 error, log2 error per volume,
// log2 volume, D.  Label of a split leaf: log2 of its relative error
// reduction, r = max(e_parent - e_left - e_right, 2^-10 e_parent) / e_parent,
// measured by the plain error estimate of the two children one pass later.
// Score used for selection: e * 2^clamp(y), y the network's prediction of
// log2 r; the plain error e is the fallback when the network is absent or its
// output is not finite.  Second label form: log2 of the squared image change
// the split makes (image_label below), scored as 2^clamp(y).  In general the
// score is e^kappa_e * 2^(kappa_y y) -- (1, 1) for the first form, (0, 1)
// for the second; equal exponents kappa scale the selection test
// pow(score / max, alpha) to the effective exponent kappa * alpha.
#include "mdas_leaf.hpp"
#include "mlp_device.hpp"

#pragma clang fp contract(off)

namespace mdas {

__device__ __forceinline__ float log2_floor(float x) { return __log2f(fmaxf(x, 1.0e-30f)); }

template <int D>
__device__ __forceinline__ void leaf_features_ext(const LeafSamples& ls, const float* ext, float e,
                                                  float depth, float sX, float sY, float* f) {
#pragma unroll
    for (int d = 0; d < 6; ++d) {
        if (d < D) {
            const float dom = d == 0 ? sX : (d == 1 ? sY : 1.0f);
            f[d] = log2_floor(ext[d] / dom);
        } else {
            f[d] = 0.0f;
        }
    }
    const int n = ls.n;
    float lum[4], s = 0.0f, lo = 3.402823466e+38f, hi = -3.402823466e+38f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        lum[q] = 0.2126f * ls.vx[q] + 0.7152f * ls.vy[q] + 0.0722f * ls.vz[q];
        if (q < n) {
            s += lum[q];
            lo = fminf(lo, lum[q]);
            hi = fmaxf(hi, lum[q]);
        }
    }
    const float mean = s / (float)n;
    float var = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (q < n) var += (lum[q] - mean) * (lum[q] - mean);
    var /= (float)n;
    f[6] = (float)n;
    f[7] = mean;
    f[8] = var;
    f[9] = lo;
    f[10] = hi;
    f[11] = depth;
    f[12] = log2_floor(e);
    f[13] = log2_floor(e / ls.vol);
    f[14] = log2_floor(ls.vol);
    f[15] = (float)D;
}

// The same from the leaf's box (extents mx - mn).
template <int D>
__device__ __forceinline__ void leaf_features(const LeafSamples& ls, const float* mn,
                                              const float* mx, float e, float depth, float sX,
                                              float sY, float* f) {
    float ext[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) ext[d] = d < D ? mx[d] - mn[d] : 1.0f;
    leaf_features_ext<D>(ls, ext, e, depth, sX, sY, f);
}

__device__ __forceinline__ float split_label(float ep, float el, float er) {
    if (!(ep > 0.0f)) return -10.0f;
    float d = ep - el;
    d = d - er;
    const float r = fmaxf(d, ep * 0.0009765625f) / ep;
    return __log2f(r);
}

// Image-change label: the reconstruction spreads a leaf's mean times its
// volume over its xy footprint, so refining parent p into children c moves
// the image by (m_c - m_p) v_c / a_c over each child's footprint a_c; the
// label is log2 of the squared change integrated over the footprints,
// sum_c (m_c - m_p)^2 v_c^2 / a_c (m = mean luminance, v = volume).
__device__ __forceinline__ float image_label(float mp, const float* mc, const float* vc,
                                             const float* ac) {
    float s = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const float d = mc[h] - mp;
        const float w = vc[h] * vc[h] / ac[h];
        s += d * d * w;
    }
    return __log2f(s + 1.0e-30f);
}

// ---------------------------------------------------- fused error pass --
// Same leaves as the plain stale-error pass (every leaf on the first pass,
// afterwards the two children of each split, handled here as one item so the
// split's label sees both), same plain error.  Writes perr and the features;
// with collection on, the label row of each split (parent features, which
// are still at the left child's slot); err receives the score and the
// workgroup max of the scores feeds the selection's global max.
template <int D>
__device__ __forceinline__ void errors_learned_body(const DevGrid& a, const LearnDev& l, int blk,
                                                    int nblk, int par) {
    __shared__ unsigned short xsb[4][128 * kMlpIn];  // a wave's staged rows (bf16)
    __shared__ unsigned short actb[4][16 * kMlpH];   // layer-1 activations (bf16)
    __shared__ float ys[4][16];
    __shared__ __align__(16) unsigned short w1s[64 * 32], w2s[64 * 64];  // the bf16 weights
    __shared__ float bl[3 * 64 + 1];  // b1, b2, bf16-rounded w3, b3
    const TreeCounts counts = a.cnt->slot[par];
    if (a.cnt->done || loop_limit_reached(a.cnt, counts.N, counts.L)) return;
    const bool first = a.cnt->passes == 0;
    const int n_items = first ? counts.L : counts.new_n;
    if (blk * 256 >= n_items) return;
    const int L_old = counts.L_old;
    const long long rows_base = (first || l.X == nullptr) ? 0 : *l.rows;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const bool feats = l.feat != nullptr;  // false: a plain member of a batch
    const bool model = feats && l.mlp.p != nullptr;
    if (model) {  // the weights once per workgroup, for every wave's tiles
        for (int k = threadIdx.x; k < 64 * 32 / 8; k += 256)
            ((u16x8*)w1s)[k] = ((const u16x8*)l.mlp.w1p)[k];
        for (int k = threadIdx.x; k < 64 * 64 / 8; k += 256)
            ((u16x8*)w2s)[k] = ((const u16x8*)l.mlp.w2p)[k];
        if (threadIdx.x < 64) {
            bl[threadIdx.x] = l.mlp.p[kOffB1 + threadIdx.x];
            bl[64 + threadIdx.x] = l.mlp.p[kOffB2 + threadIdx.x];
            bl[128 + threadIdx.x] = l.mlp.w3r[threadIdx.x];
        }
        if (threadIdx.x == 0) bl[192] = l.mlp.p[kOffB3];
        __syncthreads();
    }
    float m = 0.0f;
    for (int t0 = blk * 256; t0 < n_items; t0 += nblk * 256) {
        const int t = t0 + threadIdx.x;
        const bool act = t < n_items;
        int c[2] = {-1, -1};
        if (act) {
            c[0] = first ? t : a.split_list[t];
            c[1] = first ? -1 : L_old + t;
        }
        // the parent's row is still in the left child's slot; a collected
        // row takes it now, the label later needs only its error and mean
        float depth = 0.0f, pe = 0.0f, pm = 0.0f;
        if (act && !first && feats) {
            const float* prow = l.feat + (size_t)c[0] * kFeat;
            if (l.keep) {
                pe = l.perr[c[0]];
                pm = prow[7];
                if (l.X != nullptr && rows_base + t < l.cap_rows) {
                    const float4* pr = (const float4*)prow;
                    float4* xo = (float4*)(l.X + (rows_base + t) * kFeat);
#pragma unroll
                    for (int k = 0; k < 4; ++k) xo[k] = pr[k];
                }
            }
            depth = prow[11] + 1.0f;  // scoring only: all a split carries over
        }
        float e[2] = {0.0f, 0.0f}, vol[2] = {1.0f, 1.0f}, axy[2] = {1.0f, 1.0f}, mc[2] = {0.0f, 0.0f};
        const int hmax = first ? 1 : 2;
        // one child at a time: its features are stored and staged as the
        // network's input row (row 64 h + lane) as soon as they exist, so a
        // single feature row is live
        auto finish = [&](int h, const float* f) {
            mc[h] = f[7];
            if (c[h] >= 0 && feats) {
                if (l.keep) {
                    float4* fo = (float4*)(l.feat + (size_t)c[h] * kFeat);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        fo[k] = make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
                    l.perr[c[h]] = e[h];
                } else {
                    l.feat[(size_t)c[h] * kFeat + 11] = f[11];
                }
            }
            if (model && h < hmax) {
                unsigned short* xr = &xsb[w][(64 * h + lane) * kMlpIn];
#pragma unroll
                for (int k = 0; k < kMlpIn; ++k)
                    xr[k] = f2bf((f[k] - l.mlp.p[kOffMu + k]) * l.mlp.p[kOffIsd + k]);
            }
        };
        if (act && !first && a.sext != nullptr) {
            // both children from the split's entries: sample indices, volumes
            // and extents (the parent's, the axis's two halves), not records
            // (a plain member of a batch has no extents and reads records)
            const int4 s0 = a.sdat[2 * t], s1 = a.sdat[2 * t + 1];
            const int4 x0 = a.sext[2 * t], x1 = a.sext[2 * t + 1];
            const int ids[2][4] = {{s0.x, s0.y, -1, -1}, {s0.z, s0.w, s1.x, -1}};
            LeafSamples ls[2];
            load_values(a, ids[0], ls[0]);  // the five value loads together
            load_values(a, ids[1], ls[1]);
            vol[0] = __int_as_float(s1.y);
            vol[1] = __int_as_float(s1.z);
            const float exl[6] = {__int_as_float(x0.x), __int_as_float(x0.y), __int_as_float(x0.z),
                                  __int_as_float(x0.w), __int_as_float(x1.x), __int_as_float(x1.y)};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float ex[6];
#pragma unroll
                for (int d = 0; d < 6; ++d) ex[d] = (h == 1 && d == x1.w) ? __int_as_float(x1.z) : exl[d];
                float f[kFeat];
                e[h] = error_of_values(ids[h], vol[h], ls[h]);
                leaf_features_ext<D>(ls[h], ex, e[h], depth, a.sX, a.sY, f);
                axy[h] = ex[0] * ex[1];
                finish(h, f);
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float f[kFeat];
                if (c[h] >= 0) {
                    LeafSamples ls;
                    float mn[D], mx[D];
                    e[h] = leaf_error_s<D>(a, c[h], ls, mn, mx);
                    leaf_features<D>(ls, mn, mx, e[h], depth, a.sX, a.sY, f);
                    vol[h] = ls.vol;
                    axy[h] = (mx[0] - mn[0]) * (mx[1] - mn[1]);
                } else {
#pragma unroll
                    for (int k = 0; k < kFeat; ++k) f[k] = 0.0f;
                }
                finish(h, f);
            }
        }
        if (act && !first && feats && l.X != nullptr && rows_base + t < l.cap_rows)
            l.Y[rows_base + t] = l.label_mode == 0 ? split_label(pe, e[0], e[1])
                                                   : image_label(pm, mc, vol, axy);
        // scores: the wave's (up to) 128 leaves as 8 tiles of 16 rows
        float q[2] = {e[0], e[1]};
        if (model) {
            for (int tile = 0; tile < 4 * hmax; ++tile) {
                float y[4];
                mlp16_bf(w1s, w2s, bl, &xsb[w][16 * tile * kMlpIn], actb[w], y);
                if ((lane & 15) == 0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) ys[w][4 * (lane >> 4) + i] = y[i];
                }
                wave_sync_lds();
                const int h = tile >> 2;
                if ((lane >> 4) == (tile & 3)) {
#pragma unroll
                    for (int hh = 0; hh < 2; ++hh) {
                        if (hh != h || c[hh] < 0) continue;
                        const float yv = ys[w][lane & 15];
                        if (fabsf(yv) < 3.0e38f) {  // false for NaN and +-inf
                            const float yc = fminf(fmaxf(yv, l.ylo), l.yhi);
                            float s;
                            if (l.kappa_e == 1.0f && l.kappa_y == 1.0f)
                                s = e[hh] * exp2f(yc);
                            else if (l.kappa_e == 0.0f && l.kappa_y == 1.0f)
                                s = exp2f(yc);
                            else  // e^kappa_e * 2^(kappa_y y)
                                s = exp2f(l.kappa_e * log2_floor(e[hh]) + l.kappa_y * yc);
                            if (s < 3.0e38f) q[hh] = s;
                        }
                    }
                }
                wave_sync_lds();
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (c[h] >= 0) {
                a.err[c[h]] = q[h];
                m = fmaxf(m, q[h]);
            }
        }
    }
    super_max(a.smax + par * kSuper, m, blk);
}

// 4 waves per SIMD: the feature phase and the network fit the register file
// at that occupancy without spilling (the default allocation gave 3).
template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_errors_learned(
    DevGrid a, LearnDev l, int par) {
    errors_learned_body<D>(a, l, blockIdx.x, gridDim.x, par);
}
template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_errors_learned_b(
    const DevGrid* grids, const LearnDev* ls, int par) {
    errors_learned_body<D>(batch_grid(grids), *in_constant(ls + blockIdx.y), blockIdx.x, gridDim.x, par);
}

hipError_t launch_errors_learned(Grid& g, int parity, hipStream_t st) {
    const dim3 grid(g.error_blocks()), block(256);
    switch (g.D) {
    case 3: hipLaunchKernelGGL(k_errors_learned<3>, grid, block, 0, st, g.dev, g.learn, parity); break;
    case 4: hipLaunchKernelGGL(k_errors_learned<4>, grid, block, 0, st, g.dev, g.learn, parity); break;
    case 5: hipLaunchKernelGGL(k_errors_learned<5>, grid, block, 0, st, g.dev, g.learn, parity); break;
    case 6: hipLaunchKernelGGL(k_errors_learned<6>, grid, block, 0, st, g.dev, g.learn, parity); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_errors_learned_b(int D, const DevGrid* grids, const LearnDev* ls, int n, int blocks,
                                   int parity, hipStream_t st) {
    const dim3 grid(blocks < 1024 ? blocks : 1024, n), block(256);
    switch (D) {
    case 3: hipLaunchKernelGGL(k_errors_learned_b<3>, grid, block, 0, st, grids, ls, parity); break;
    case 4: hipLaunchKernelGGL(k_errors_learned_b<4>, grid, block, 0, st, grids, ls, parity); break;
    case 5: hipLaunchKernelGGL(k_errors_learned_b<5>, grid, block, 0, st, grids, ls, parity); break;
    case 6: hipLaunchKernelGGL(k_errors_learned_b<6>, grid, block, 0, st, grids, ls, parity); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------ the network --
// bf16 forms of the weights from the FP32 blob.
__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ p, unsigned short* w1p,
                                                  unsigned short* w2p, float* w2r, float* w3r) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < 64 * 32) {
        const int n = t >> 5, k = t & 31;
        w1p[t] = k < kMlpIn ? f2bf(p[kOffW1 + n * kMlpIn + k]) : (unsigned short)0;
    }
    if (t < 64 * 64) {
        const unsigned short b = f2bf(p[kOffW2 + t]);
        w2p[t] = b;
        w2r[t] = bf2f(b);
    }
    if (t < 64) w3r[t] = bfround(p[kOffW3 + t]);
}

hipError_t launch_mlp_pack(float* p, unsigned short* w1p, unsigned short* w2p, float* w2r,
                           float* w3r, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_pack, dim3(16), dim3(256), 0, st, p, w1p, w2p, w2r, w3r);
    return hipGetLastError();
}

// Inference over n rows of raw features: one wave per 16-row tile.
__global__ __launch_bounds__(256) void k_mlp_forward(MlpDev M, const float* __restrict__ X,
                                                     long long n, float* __restrict__ Y) {
    __shared__ float xs[4][16 * kMlpIn];
    __shared__ float acts[4][16 * kMlpH];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long tiles = (n + 15) / 16;
    for (long long tile = (long long)blockIdx.x * 4 + w; tile < tiles; tile += (long long)gridDim.x * 4) {
        const long long r0 = tile * 16;
        if (lane < 16) {
            float f[kMlpIn];
            const long long r = r0 + lane;
#pragma unroll
            for (int k = 0; k < kMlpIn; ++k) f[k] = r < n ? X[r * kMlpIn + k] : 0.0f;
            mlp_stage_row(M, f, &xs[w][lane * kMlpIn]);
        }
        float y[4];
        mlp16(M, xs[w], acts[w], y);
        if ((lane & 15) == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const long long r = r0 + 4 * (lane >> 4) + i;
                if (r < n) Y[r] = y[i];
            }
        }
    }
}

hipError_t launch_mlp_forward(const MlpDev& M, const float* X, long long n, float* Y,
                              hipStream_t st) {
    long long blocks = ((n + 15) / 16 + 3) / 4;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)blocks), dim3(256), 0, st, M, X, n, Y);
    return hipGetLastError();
}

// Gradient of mean((y - t)^2) over a batch.  A wave takes 16 rows at a time:
// the bf16 MFMA forward, then the backward in FP32 on
// v_mfma_f32_16x16x4_f32.  All of a tile stays in registers in the layout the
// products leave (lane l: rows 4 (l/16) + i, column l%16): a K step that
// takes row 4 (l/16) + i from lane group l/16 is step i's register of both
// operands, so dW2 = dZ2^T A1 and dW1 = dZ1^T X need no data movement; only
// dA1 = dZ2 W2 turns dZ2 over through LDS (rows padded to 68 floats, X's to
// 20: conflict-free).  The sums of dW1, dW2 and a tile's activations leave
// 2 waves per SIMD, which is what bounds the kernel: a tile is one dependent
// chain from its rows to its sums.  The same sums on the vector units, one lane per hidden unit,
// read every dZ2 element through LDS broadcasts at 1 wave per SIMD: 116 us for
// 60013 rows, now 40 (18 of it a
// single tile's chain).  The four waves' sums are added in LDS, pairwise, and
// written as one partial per workgroup.
static const int kGradTr = 68, kGradX = 20;  // padded LDS rows of dZ2 / activations and X

// One wave's sums: row 16 t + 4 kg + i, column 16 u + col of dW2 and so on.
struct MlpSums {
    f32x4 w2[4][4], w1[4];
    float b1[4], b2[4], w3[4], b3, loss;
};

// f(parameter index, sum) over the sums this lane holds (those replicated
// over lane groups once); the loss goes last, at index kMlpParams.
template <typename F>
__device__ __forceinline__ void for_each_sum(MlpSums& g, int lane, F f) {
    const int col = lane & 15, kg = lane >> 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = 16 * t + 4 * kg + i;
            float v = g.w1[t][i];
            f(kOffW1 + n * kMlpIn + col, v);
            g.w1[t][i] = v;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v = g.w2[t][u][i];
                f(kOffW2 + n * kMlpH + 16 * u + col, v);
                g.w2[t][u][i] = v;
            }
        }
        if (kg == 0) {
            f(kOffB1 + 16 * t + col, g.b1[t]);
            f(kOffB2 + 16 * t + col, g.b2[t]);
            f(kOffW3 + 16 * t + col, g.w3[t]);
        }
    }
    if (lane == 0) {
        f(kOffB3, g.b3);
        f(kMlpParams, g.loss);
    }
}

__global__ __launch_bounds__(256, 2) void k_mlp_grad(MlpDev M, const float* __restrict__ X,
                                                     const float* __restrict__ T, long long n_rows,
                                                     long long start, int count,
                                                     unsigned long long pa, unsigned long long pc,
                                                     float* __restrict__ gpart,
                                                     float* __restrict__ lpart) {
    constexpr int kTile = 16 * (kGradTr + kGradX);         // a wave's scratch, floats
    constexpr int kWeights = (64 * 32 + 64 * 64) / 2;      // the bf16 weights, floats
    constexpr int kSumsPad = (kMlpParams + 1 + 3) & ~3;
    constexpr int kLds = 4 * kTile + kWeights + kMlpH * kGradTr;
    static_assert(kLds >= 2 * kSumsPad, "two waves' sums");
    __shared__ __align__(16) float lds[kLds];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int col = lane & 15, kg = lane >> 4;
    float* tr = lds + w * kTile;
    float* xs = tr + 16 * kGradTr;
    unsigned short* w1s = (unsigned short*)(lds + 4 * kTile);
    unsigned short* w2s = w1s + 64 * 32;
    for (int k = threadIdx.x; k < 64 * 32 / 8; k += 256) ((u16x8*)w1s)[k] = ((const u16x8*)M.w1p)[k];
    for (int k = threadIdx.x; k < 64 * 64 / 8; k += 256) ((u16x8*)w2s)[k] = ((const u16x8*)M.w2p)[k];
    // dA1's operand, W2 turned over: K step s takes unit n = 16 kg + s from
    // lane group kg
    float* w2t = lds + 4 * kTile + kWeights;
    for (int k = threadIdx.x; k < kMlpH * kMlpH; k += 256)
        w2t[(k % kMlpH) * kGradTr + k / kMlpH] = M.w2r[k];
    float b1[4], b2[4], w3[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        b1[t] = M.p[kOffB1 + 16 * t + col];
        b2[t] = M.p[kOffB2 + 16 * t + col];
        w3[t] = M.w3r[16 * t + col];
    }
    const float b3 = M.p[kOffB3];
    MlpSums g;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int u = 0; u < 4; ++u) g.w2[t][u] = zero;
        g.w1[t] = zero;
        g.b1[t] = g.b2[t] = g.w3[t] = 0.0f;
    }
    g.b3 = g.loss = 0.0f;
    const float scale = 2.0f / (float)count;
    const int tiles = (count + 15) / 16;
    __syncthreads();
    // lane l fetches quarter l%4 of the tile's row l/4 and that row's target,
    // one tile ahead
    const int fr = lane >> 2, fq = lane & 3;
    f32x4 xv = zero;
    float tv = 0.0f;
    auto fetch = [&](int tile) {
        const int q = tile * 16 + fr;
        if (tile < tiles && q < count) {
            const long long r = (long long)((pa * (unsigned long long)(start + q) + pc) %
                                            (unsigned long long)n_rows);
            xv = *(const f32x4u*)(X + r * kMlpIn + 4 * fq);
            tv = T[r];
        } else {
            xv = zero;
            tv = 0.0f;
        }
    };
    fetch(blockIdx.x * 4 + w);
    const float* mp = M.p + kOffMu + 4 * fq;
    const float* ip = M.p + kOffIsd + 4 * fq;
    const float4 mu = make_float4(mp[0], mp[1], mp[2], mp[3]), isd = make_float4(ip[0], ip[1], ip[2], ip[3]);
    for (int tile = blockIdx.x * 4 + w; tile < tiles; tile += gridDim.x * 4) {
        *(float4*)(xs + fr * kGradX + 4 * fq) =
            make_float4(bfround((xv.x - mu.x) * isd.x), bfround((xv.y - mu.y) * isd.y),
                        bfround((xv.z - mu.z) * isd.z), bfround((xv.w - mu.w) * isd.w));
        float tgt[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) tgt[i] = __shfl(tv, (4 * kg + i) * 4, 64);
        fetch(tile + gridDim.x * 4);
        wave_sync_lds();
        // forward, as mlp16
        float av[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) av[k] = kg < 2 ? xs[col * kGradX + 8 * kg + k] : 0.0f;
        const bf16x8 ax = pack_b8(av);
        float a1[4][4], g1[4][4], d2[4][4], a2[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                ax, load_b8(w1s + (16 * t + col) * 32 + 8 * kg), zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v;
                gelu_both(z[i] + b1[t], v, g1[t][i]);
                a1[t][i] = bfround(v);
                tr[(4 * kg + i) * kGradTr + 16 * t + col] = a1[t][i];
            }
        }
        wave_sync_lds();
        bf16x8 aa[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = tr[col * kGradTr + 32 * c + 8 * kg + k];
            aa[c] = pack_b8(v);
        }
        wave_sync_lds();  // tr is written again below
        float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 z = zero;
#pragma unroll
            for (int c = 0; c < 2; ++c)
                z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    aa[c], load_b8(w2s + (16 * t + col) * 64 + 32 * c + 8 * kg), z, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v;
                gelu_both(z[i] + b2[t], v, d2[t][i]);
                a2[t][i] = bfround(v);
                y[i] += a2[t][i] * w3[t];
            }
        }
        // output, loss, and layer 3
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float sum = y[i];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) sum += __shfl_xor(sum, o, 64);
            const float diff = sum + b3 - tgt[i];
            const bool in = tile * 16 + 4 * kg + i < count;
            const float dy = in ? scale * diff : 0.0f;
            g.loss += in ? diff * diff : 0.0f;
            g.b3 += dy;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                g.w3[t] += dy * a2[t][i];
                d2[t][i] = dy * w3[t] * d2[t][i];
                g.b2[t] += d2[t][i];
                tr[(4 * kg + i) * kGradTr + 16 * t + col] = d2[t][i];
            }
        }
        wave_sync_lds();
        // dA1 = dZ2 W2: row l%16 of dZ2, units 16 kg + s
        f32x4 da[4] = {zero, zero, zero, zero};
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const f32x4 v = *(const f32x4*)(tr + col * kGradTr + 16 * kg + 4 * q4);
            f32x4 wv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) wv[u] = *(const f32x4*)(w2t + (16 * u + col) * kGradTr + 16 * kg + 4 * q4);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    da[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[q], wv[u][q], da[u], 0, 0, 0);
        }
        // dW2 = dZ2^T A1
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    g.w2[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(d2[t][i], a1[u][i], g.w2[t][u], 0, 0, 0);
        // dZ1 and dW1 = dZ1^T X
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float xr = xs[(4 * kg + i) * kGradX + col];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float d1 = da[t][i] * g1[t][i];
                g.b1[t] += d1;
                g.w1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(d1, xr, g.w1[t], 0, 0, 0);
            }
        }
        wave_sync_lds();  // xs and tr are written by the next tile
    }
    // sums that every lane group holds a part of
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            g.b1[t] += __shfl_xor(g.b1[t], o, 64);
            g.b2[t] += __shfl_xor(g.b2[t], o, 64);
            g.w3[t] += __shfl_xor(g.w3[t], o, 64);
        }
        g.b3 += __shfl_xor(g.b3, o, 64);
        g.loss += __shfl_xor(g.loss, o, 64);
    }
    // the workgroup's partial: (wave 0 + wave 2) + (wave 1 + wave 3)
    __syncthreads();
    float* buf = lds + (w & 1) * kSumsPad;
    if (w >= 2) for_each_sum(g, lane, [&](int k, float& v) { buf[k] = v; });
    __syncthreads();
    if (w < 2) for_each_sum(g, lane, [&](int k, float& v) { v += buf[k]; });
    __syncthreads();
    if (w == 1) for_each_sum(g, lane, [&](int k, float& v) { lds[k] = v; });
    __syncthreads();
    if (w == 0) {
        float* o = gpart + (size_t)blockIdx.x * kMlpParams;
        float* lo = lpart + blockIdx.x;
        for_each_sum(g, lane, [&](int k, float& v) { *(k < kMlpParams ? o + k : lo) = v + lds[k]; });
    }
}

int launch_mlp_grad(const MlpDev& M, const float* X, const float* T, long long n_rows,
                    long long start, int count, unsigned long long pa, unsigned long long pc,
                    float* gpart, float* lpart, hipStream_t st, hipError_t* err) {
    int blocks = ((count + 15) / 16 + 3) / 4;
    if (blocks > kMlpGradBlocks) blocks = kMlpGradBlocks;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_mlp_grad, dim3(blocks), dim3(256), 0, st, M, X, T, n_rows, start, count,
                       pa, pc, gpart, lpart);
    *err = hipGetLastError();
    return blocks;
}

// Sum of the partials of the workgroup's 32 parameters, in a fixed order: 32
// slices of every 32nd partial, then the slices.  Returns parameter t's sum
// in the threads of slice 0.  One thread per parameter walking all the
// partials was a chain of 1024 dependent loads and adds (271 us a step, now 6.4
// with the update).
__device__ __forceinline__ float sum_partials(const float* __restrict__ part, int nparts, int stride,
                                              int t, int limit) {
    __shared__ float red[32][33];
    const int j = threadIdx.x & 31, slice = threadIdx.x >> 5;
    float s = 0.0f;
    if (t < limit)
#pragma unroll 8
        for (int q = slice; q < nparts; q += 32) s += part[(size_t)q * stride + t];
    __syncthreads();  // the previous sum's readers are done
    red[slice][j] = s;
    __syncthreads();
    s = 0.0f;
    if (slice == 0)
#pragma unroll
        for (int q = 0; q < 32; ++q) s += red[q][j];
    return s;
}

__global__ __launch_bounds__(1024) void k_mlp_sum(const float* __restrict__ gpart,
                                                  const float* __restrict__ lpart, int nparts,
                                                  float* gsum, float* loss) {
    const int t = blockIdx.x * 32 + (threadIdx.x & 31);
    const float s = sum_partials(gpart, nparts, kMlpParams, t, kMlpParams);
    if (threadIdx.x < 32 && t < kMlpParams) gsum[t] = s;
    if (blockIdx.x == 0) {
        const float l = sum_partials(lpart, nparts, 1, threadIdx.x & 31, 1);
        if (threadIdx.x == 0) *loss = l;
    }
}

hipError_t launch_mlp_sum(const float* gpart, const float* lpart, int nparts, float* gsum,
                          float* loss, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_sum, dim3((kMlpParams + 31) / 32), dim3(1024), 0, st, gpart, lpart,
                       nparts, gsum, loss);
    return hipGetLastError();
}

// Adam (beta1 0.9, beta2 0.999, eps 1e-8) on the summed gradient, FP32
// master weights, then the bf16 forms of the updated weight.  bc1 / bc2 are
// the bias corrections 1 - beta^t.  loss_acc (if non-null) accumulates the
// batch's squared-error sum.
__global__ __launch_bounds__(1024) void k_mlp_adam(float* p, float* m, float* v,
                                                   const float* __restrict__ gpart,
                                                   const float* __restrict__ lpart, int nparts,
                                                   float lr, float bc1, float bc2, float* loss_acc,
                                                   unsigned short* w1p, unsigned short* w2p,
                                                   float* w2r, float* w3r) {
    const int t = blockIdx.x * 32 + (threadIdx.x & 31);
    const float g = sum_partials(gpart, nparts, kMlpParams, t, kMlpParams);
    if (threadIdx.x < 32 && t < kMlpParams) {
        const float mt = 0.9f * m[t] + 0.1f * g;
        const float vt = 0.999f * v[t] + 0.001f * g * g;
        m[t] = mt;
        v[t] = vt;
        const float mh = mt / bc1, vh = vt / bc2;
        const float nw = p[t] - lr * mh / (sqrtf(vh) + 1.0e-8f);
        p[t] = nw;
        if (t < kOffB1) {
            const int n = t / kMlpIn, kk = t % kMlpIn;
            w1p[n * 32 + kk] = f2bf(nw);
        } else if (t >= kOffW2 && t < kOffB2) {
            const unsigned short b = f2bf(nw);
            w2p[t - kOffW2] = b;
            w2r[t - kOffW2] = bf2f(b);
        } else if (t >= kOffW3 && t < kOffB3) {
            w3r[t - kOffW3] = bfround(nw);
        }
    }
    if (blockIdx.x == 0 && loss_acc != nullptr) {
        const float l = sum_partials(lpart, nparts, 1, threadIdx.x & 31, 1);
        if (threadIdx.x == 0) *loss_acc += l;
    }
}

hipError_t launch_mlp_adam(float* p, float* m, float* v, const float* gpart, const float* lpart,
                           int nparts, float lr, float bc1, float bc2, float* loss_acc,
                           unsigned short* w1p, unsigned short* w2p, float* w2r, float* w3r,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + 31) / 32), dim3(1024), 0, st, p, m, v, gpart,
                       lpart, nparts, lr, bc1, bc2, loss_acc, w1p, w2p, w2r, w3r);
    return hipGetLastError();
}

// Per-workgroup sums and sums of squares (double) of the 16 features.
__global__ __launch_bounds__(256) void k_feat_stats(const float* __restrict__ X, long long n,
                                                    double* part) {
    __shared__ double red[2 * kMlpIn][4];
    const int j = threadIdx.x & 15;
    double s = 0.0, s2 = 0.0;
    for (long long r = (long long)blockIdx.x * 16 + (threadIdx.x >> 4); r < n;
         r += (long long)gridDim.x * 16) {
        const double x = X[r * kMlpIn + j];
        s += x;
        s2 += x * x;
    }
    // 16 rows per pass: lanes j, j+16, j+32, j+48 of a wave share feature j
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    s2 += __shfl_xor(s2, 16, 64);
    s2 += __shfl_xor(s2, 32, 64);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) < 16) {
        red[j][w] = s;
        red[kMlpIn + j][w] = s2;
    }
    __syncthreads();
    if (threadIdx.x < 2 * kMlpIn) {
        const double* r = red[threadIdx.x];
        part[(size_t)blockIdx.x * 2 * kMlpIn + threadIdx.x] = ((r[0] + r[1]) + r[2]) + r[3];
    }
}

hipError_t launch_feat_stats(const float* X, long long n, double* part, int nblocks,
                             hipStream_t st) {
    hipLaunchKernelGGL(k_feat_stats, dim3(nblocks), dim3(256), 0, st, X, n, part);
    return hipGetLastError();
}

}  // namespace mdas
