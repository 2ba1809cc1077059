// Analytic integrand launch: the replacement of optixLaunch over the new
// sample slice (optixMotionBlur.cpp:458-467 with sample_offset/sample_count,
// SDK/cuda/whitted.cu:164-293).  The scene's object table (<= 12 KB) is staged
// in LDS once per workgroup that has a sample; every thread then evaluates
// samples grid-stride.  A ray looks its spheres up by cell (scenes.hpp): what
// bounds the kernel is the serial chain of a ray's sphere tests and its lanes'
// divergence, so fewer tests per ray beat any arrangement of them.  Against
// group tests over all spheres: the 5D 1080p run's 41 launches 7.53 -> 2.79 ms,
// a launch for the ~500 samples of a thumbnail's pass 38 -> 10 us, the FP64
// ground truth at 240x135, 64 samples per pixel 2.28 -> 0.49 ms.
#include "mdas_leaf.hpp"
#include "scenes.hpp"

#pragma clang fp contract(off)

namespace mdas {

// The scene's object table into LDS (every thread of the workgroup takes
// part).
__device__ __forceinline__ void stage_scene(const mscene::SceneBlock* __restrict__ B, float* obj) {
    const int nobj = B->p.n_obj;
    for (int k = threadIdx.x; k < nobj * mscene::OBJ_STRIDE; k += blockDim.x) obj[k] = B->p.obj[k];
    __syncthreads();
}

// The cells' words follow the scene block.
__device__ __forceinline__ const uint64_t* cell_words(const mscene::SceneBlock* B) {
    return reinterpret_cast<const uint64_t*>(B + 1);
}

__device__ __forceinline__ void eval_body(const float* __restrict__ coords,
                                          float* __restrict__ values, int dim,
                                          const mscene::SceneBlock* __restrict__ B, int first,
                                          int count, const DevCounters* cnt, int dev_range, int blk,
                                          int nblk) {
    __shared__ float obj[mscene::MAX_OBJ * mscene::OBJ_STRIDE];
    int beg = first, end = first + count;
    if (dev_range) {
        if (cnt->done) return;
        const TreeCounts t = cnt->slot[cnt->cur];
        beg = t.N_old;
        end = t.N;
    }
    if (blk * 256 >= end - beg) return;  // uniform: no sample for this workgroup
    stage_scene(B, obj);
    const mscene::Params* P = &B->p;
    for (int i = beg + blk * 256 + threadIdx.x; i < end; i += nblk * 256) {
        float x[6];
        const float* c = coords + (size_t)i * dim;
        for (int d = 0; d < dim; ++d) x[d] = c[d];
        mscene::V3<float> v = mscene::eval<float>(*P, obj, x, &B->accel, &B->cells, cell_words(B));
        float* o = values + (size_t)i * 3;
        o[0] = v.x;
        o[1] = v.y;
        o[2] = v.z;
    }
}

__global__ __launch_bounds__(256) void k_eval(const float* __restrict__ coords,
                                              float* __restrict__ values, int dim,
                                              const mscene::SceneBlock* __restrict__ B,
                                              int first, int count, const DevCounters* cnt,
                                              int dev_range) {
    eval_body(coords, values, dim, B, first, count, cnt, dev_range, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(256) void k_eval_b(const DevGrid* __restrict__ grids,
                                                const void* const* __restrict__ params) {
    const DevGrid a = batch_grid(grids);
    eval_body(a.coords, a.values, a.D, in_constant((const mscene::SceneBlock*)params[blockIdx.y]), 0, 0,
              a.cnt, 1, blockIdx.x, gridDim.x);
}

// The words of a scene's cells (scenes.hpp), once per scene: a wave per word,
// a lane per sphere (a thread per word, its 64 spheres one after another, took
// 40 us on the 64-sphere scenes).
__global__ __launch_bounds__(256) void k_scene_cells(mscene::SceneBlock* B) {
    const mscene::Cells& C = B->cells;
    uint64_t* tab = reinterpret_cast<uint64_t*>(B + 1);
    const int n = C.n_cells * C.words, lane = threadIdx.x & 63;
    for (int i = blockIdx.x * 4 + (threadIdx.x >> 6); i < n; i += gridDim.x * 4) {
        const int c = i / C.words, k = 64 * (i % C.words) + lane;
        const uint64_t word = __ballot(k < B->p.n_obj && mscene::cell_holds(B->p, C, c, k));
        if (lane == 0) tab[i] = word;
    }
}

hipError_t launch_scene_cells(void* dparams, int words, hipStream_t st) {
    if (words <= 0) return hipSuccess;
    const int blocks = (words + 3) / 4;
    hipLaunchKernelGGL(k_scene_cells, dim3(blocks < 2048 ? blocks : 2048), dim3(256), 0, st,
                       (mscene::SceneBlock*)dparams);
    return hipGetLastError();
}

// ------------------------------------------------- QMC and ground truth --
// The reference's non-MDAS sampler (SDK/cuda/sampler.h:4-28, random.h:75-89,
// whitted.cu:59-83): per pixel a TEA-seeded set of 6 Cranley-Patterson
// offsets, sample s takes the Halton point s (bases 2, 3, 5, 7, 11, 13)
// shifted by the offsets and wrapped when above 1; dims 0 and 1 jitter inside
// the pixel.
// `real` = float gives the MC/QMC baseline images, double the FP64
// high-sample-count ground truth.
template <int BASE, typename real>
__device__ __forceinline__ real halton_r(int i) {
    real r = 0, f = (real)1 / (real)BASE;
    int j = i;
    while (j > 0) {
        r += f * (real)(j % BASE);
        j /= BASE;
        f = mscene::div_by<BASE>(f);
    }
    return r;
}
template <typename real>
__device__ __forceinline__ real halton_dim(int dim, int i) {
    switch (dim) {
    case 0: return halton_r<2, real>(i);
    case 1: return halton_r<3, real>(i);
    case 2: return halton_r<5, real>(i);
    case 3: return halton_r<7, real>(i);
    case 4: return halton_r<11, real>(i);
    default: return halton_r<13, real>(i);
    }
}

// 2^lsh lanes share a pixel: each evaluates every 2^lsh-th sample, and all of
// them add the samples' values in sample order (the sum of a single lane).
// The points of 64 samples at a time are computed once per workgroup.  One
// lane per pixel left half the CUs idle on images of 32 thousand pixels and
// every wave recomputed the points: 240x135 at 64 samples in FP64 took 485 us
// that way (before the lens map's cheaper divisions), 97 us now.
template <typename real>
__global__ __launch_bounds__(256) void k_qmc_image(const mscene::SceneBlock* __restrict__ B,
                                                   int W, int H, int spp, int first_sample,
                                                   unsigned frame, int lsh, real* out) {
    constexpr int CH = 64;  // samples whose points are staged together
    __shared__ float obj[mscene::MAX_OBJ * mscene::OBJ_STRIDE];
    __shared__ real pts[6][CH];
    stage_scene(B, obj);
    const mscene::Params* P = &B->p;
    const int dim = P->dim;
    const int S = 1 << lsh, part = threadIdx.x & (S - 1), npix = W * H;
    const int per = 256 >> lsh;  // pixels of a workgroup
    for (int base = blockIdx.x * per; base < npix; base += gridDim.x * per) {
        const int pix = base + (threadIdx.x >> lsh);
        const bool live = pix < npix;
        const int px = pix % W, py = pix / W;
        unsigned seed = tea4((unsigned)pix, frame);
        real off[6];
#pragma unroll
        for (int d = 0; d < 6; ++d) off[d] = (real)rnd(seed);
        real ax = 0, ay = 0, az = 0;
        for (int s0 = 0; s0 < spp; s0 += CH) {
            const int n = min(CH, spp - s0);
            __syncthreads();  // the chunk before is read
            for (int k = threadIdx.x; k < dim * CH; k += 256)
                if (k % CH < n) pts[k / CH][k % CH] = halton_dim<real>(k / CH, first_sample + s0 + k % CH);
            __syncthreads();
            for (int r = 0; r < n; r += S) {
                mscene::V3<real> v = mscene::v3((real)0, (real)0, (real)0);
                if (live && r + part < n) {
                    real x[6];
#pragma unroll
                    for (int d = 0; d < 6; ++d) {
                        if (d >= dim) break;
                        real h = pts[d][r + part] + off[d];
                        if (h > (real)1) h -= (real)1;
                        x[d] = h;
                    }
                    x[0] = ((real)px + x[0]) * (real)P->scale_x / (real)W;
                    x[1] = ((real)py + x[1]) * (real)P->scale_y / (real)H;
                    v = mscene::eval<real>(*P, obj, x, &B->accel, &B->cells, cell_words(B));
                }
                const int m = min(S, n - r);
                for (int j = 0; j < m; ++j) {
                    ax += __shfl(v.x, j, S);
                    ay += __shfl(v.y, j, S);
                    az += __shfl(v.z, j, S);
                }
            }
        }
        if (live && part == 0) {
            real* o = out + (size_t)pix * 4;
            const real inv = (real)1 / (real)spp;
            o[0] = ax * inv;
            o[1] = ay * inv;
            o[2] = az * inv;
            o[3] = 0;
        }
    }
}

hipError_t launch_qmc_image(const void* dparams, int W, int H, int spp, int first_sample,
                            unsigned frame, bool fp64, void* out, hipStream_t st) {
    // lanes per pixel: enough for 8 waves per SIMD (2^19 lanes), at most a
    // wave and one sample each
    int lsh = 0;
    while (lsh < 6 && ((long long)W * H << lsh) < (1ll << 19) && (2 << lsh) <= spp) ++lsh;
    long long blocks = (((long long)W * H << lsh) + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (fp64)
        hipLaunchKernelGGL(k_qmc_image<double>, dim3((unsigned)blocks), dim3(256), 0, st,
                           (const mscene::SceneBlock*)dparams, W, H, spp, first_sample, frame, lsh,
                           (double*)out);
    else
        hipLaunchKernelGGL(k_qmc_image<float>, dim3((unsigned)blocks), dim3(256), 0, st,
                           (const mscene::SceneBlock*)dparams, W, H, spp, first_sample, frame, lsh,
                           (float*)out);
    return hipGetLastError();
}

hipError_t launch_eval(Grid& g, const void* dparams, int first, int count, bool dev_range,
                       hipStream_t st) {
    long long n = dev_range ? (long long)g.cap_s : (long long)count;
    long long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_eval, dim3((unsigned)blocks), dim3(256), 0, st, g.dev.coords,
                       g.dev.values, g.D, (const mscene::SceneBlock*)dparams, first, count,
                       (const DevCounters*)g.dev.cnt, dev_range ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_eval_b(const DevGrid* grids, const void* const* params, int n, int blocks,
                         hipStream_t st) {
    hipLaunchKernelGGL(k_eval_b, dim3(blocks, n), dim3(256), 0, st, grids, params);
    return hipGetLastError();
}

}  // namespace mdas
