// Sampling kernels of the MDAS grid: initial Morton grid, per-leaf error with
// the global max, and the adaptive pass (selection, best-candidate placement,
// median split) with indices allocated in leaf order.
//
// Layout (HBM): sample coordinates AoS float[D] and values float3 (the
// integrand contract); one 128-byte line per leaf (slots, box and its first
// points) plus an overflow row for the other points (D >= 5), so a leaf
// touched at a random index costs one line; errors, LCG states and a one-byte
// flag word (the sample count) per leaf as separate streams for the per-pass
// sweep over all leaves.  Cross-workgroup totals go through 64 groups of
// atomics, a line each, and per-workgroup partials (no address takes more than
// a few dozen atomics).
#include "mdas_leaf.hpp"
#include "scenes.hpp"

#pragma clang fp contract(off)

namespace mdas {

#define MDAS_ERR_CAPACITY_DEV (-2)

// ----------------------------------------------------------------- initial --
// kdgrid.cu:121-202.  One thread per initial leaf; four samples per leaf are
// drawn from tea4(leaf, 0) in dimension order.  The 4*D coordinates of a
// workgroup's 256 leaves are one contiguous range, written through LDS so
// that every store instruction covers 256 contiguous bytes.
template <int D>
__device__ __forceinline__ void initial_body(const DevGrid& a, int L0, int blk, int nblk) {
    __shared__ float stage[256 * 4 * D];
    for (int base = blk * 256; base < L0; base += nblk * 256) {
        const int i = base + threadIdx.x;
        if (i < L0) {
            float off[D], ext[D];
            morton_cell<D>((unsigned)i, a.b, a.e, a.sX, a.sY, off, ext);
            unsigned s = tea4((unsigned)i, 0u);
            float pts[4][D];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float r[D];
#pragma unroll
                for (int d = 0; d < D; ++d) r[d] = rnd(s);
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    pts[j][d] = off[d] + r[d] * ext[d];
                    stage[threadIdx.x * 4 * D + j * D + d] = pts[j][d];
                }
            }
            float mx[D];
#pragma unroll
            for (int d = 0; d < D; ++d) mx[d] = off[d] + ext[d];
            // the leaf's line (slots, box, first points) and its overflow row
            store_line<D>(a, i, make_int4(4 * i, 4 * i + 1, 4 * i + 2, 4 * i + 3), off, mx, pts, 4);
            if constexpr (line_pts(D) < 4) {
                // the overflow row: the points past the line and the slots
                // kept beside them
                constexpr int P = line_pts(D), XS = xpts_stride(D);
                float x[XS];
#pragma unroll
                for (int k = 0; k < XS; ++k) x[k] = 0.0f;
#pragma unroll
                for (int q = P; q < 4; ++q)
#pragma unroll
                    for (int d = 0; d < D; ++d) x[xpt_at(D, q) + d] = pts[q][d];
#pragma unroll
                for (int q = 2; q < 4; ++q)
                    if (slot_at(D, q) < 0) x[-1 - slot_at(D, q)] = __int_as_float(4 * i + q);
                float4* xr = reinterpret_cast<float4*>(a.xpts + (size_t)i * XS);
#pragma unroll
                for (int k = 0; k < XS / 4; ++k) xr[k] = make_float4(x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]);
            }
            a.seed[i] = s;
            a.err[i] = -1.0f;
            a.flags[i] = 4;
        }
        __syncthreads();
        // leaf i's samples are 4i..4i+3: the workgroup's coordinates are one
        // contiguous range, stored from LDS in full lines
        const int nl = min(256, L0 - base);
        float* out = a.coords + (size_t)base * 4 * D;
        for (int k = threadIdx.x; k < nl * 4 * D; k += 256) out[k] = stage[k];
        __syncthreads();
    }
}

template <int D>
__global__ __launch_bounds__(256) void k_initial(DevGrid a, int L0) {
    initial_body<D>(a, L0, blockIdx.x, gridDim.x);
}

// Batched form: image blockIdx.y of the set, initial leaf count from its
// configuration.
template <int D>
__global__ __launch_bounds__(256) void k_initial_b(const DevGrid* __restrict__ grids) {
    const DevGrid a = batch_grid(grids);
    initial_body<D>(a, 1 << (a.b * D + 2 * a.e), blockIdx.x, gridDim.x);
}

// Counter set-up of InitialSampling (kdgrid.cu:639-642): g_error = 0, every
// total zero, the loop's limit (and the capacity as its guard when the limit
// is the capacity; below it a pass that would overflow is an error).
__device__ __forceinline__ void initial_counters_body(const DevGrid& a, int L0, int limit) {
    if (threadIdx.x < kSumSets * kSuper)
        a.ssum[threadIdx.x].sel = a.ssum[threadIdx.x].split = a.ssum[threadIdx.x].held = 0;
    a.smax[threadIdx.x].err = 0u;
    if (threadIdx.x != 0) return;
    DevCounters* c = a.cnt;
    c->cur = 0;
    // the first integrand launch covers all the samples
    c->slot[0] = c->slot[1] = TreeCounts{4 * L0, L0, 0, 0, 4 * L0, 0};
    c->done = 0;
    c->status = 0;
    c->passes = 0;
    c->limit = limit;
    c->guard_cap = limit >= a.cap_s ? a.cap_s : 0;
}
__global__ __launch_bounds__(kMaxSets* kSuper) void k_initial_counters(DevGrid a, int L0, int limit) {
    initial_counters_body(a, L0, limit);
}
// Batched form: one workgroup per image.
__global__ __launch_bounds__(kMaxSets* kSuper) void k_initial_counters_b(const DevGrid* grids, const int* limits) {
    const DevGrid& a = grids[blockIdx.x];
    initial_counters_body(a, 1 << (a.b * a.D + 2 * a.e), limits[blockIdx.x]);
}

// Before a single call: the pass kernels run again after a loop or a refused
// pass, without the loop's limit, from zero totals; before ComputeErrors
// (kdgrid.cu:684-685) g_error = 0.  The tree's counts move to the slot that the
// host launches the pass with, if they are in the other one (a graph of the
// caller's may have set the grid up since the host last saw it).
__global__ __launch_bounds__(kSuper) void k_arm(DevGrid a, int errors, int adaptive, int par) {
    DevCounters* c = a.cnt;
    SuperSum& t = a.ssum[par * kSuper + threadIdx.x];
    if (adaptive) t.sel = t.split = t.held = 0;
    if (errors) a.smax[kGError * kSuper + threadIdx.x].err = 0u;
    if (threadIdx.x != 0) return;
    c->done = 0;
    if (adaptive) {
        c->status = 0;
        if (c->cur != par) {
            c->slot[par] = c->slot[par ^ 1];
            c->cur = par;
        }
    }
    if (errors) {
        c->limit = 0x7fffffff;
        c->guard_cap = 0;
    }
}

// ------------------------------------------------------------------ errors --
// kdgrid.cu:204-288 as the reference runs it: every leaf with error < 0 is
// re-estimated and every leaf takes part in the global max.  The max of
// non-negative floats is the max of their bit patterns, so the reduction is
// exact in any order.
template <int D>
__global__ __launch_bounds__(256) void k_compute_errors(DevGrid a) {
    const int L = leaf_total(a);
    float m = 0.0f;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < L; i += gridDim.x * 256) {
        float e = a.err[i];
        if (e < 0.0f) {
            int n;
            e = leaf_error<D>(a, i, &n);
            a.err[i] = e;
        }
        m = fmaxf(m, e);
    }
    super_max(a.smax + kGError * kSuper, m, blockIdx.x);
}

// The same result inside the sampling loop without the sweep over all
// leaves: the only stale leaves are the two children of every leaf the last
// pass split (split_list[t] and L_old + t, whose sample indices and volumes
// the placement left in the split's entry; inside the loop it does not mark
// them -1, since they are re-estimated here); the max over the other leaves
// was carried into the pass's totals by the selection before.  The first pass
// after the initial grid re-estimates every leaf.
template <int D>
__device__ __forceinline__ void errors_body(const DevGrid& a, int blk, int nblk, int par) {
    const TreeCounts c = a.cnt->slot[par];
    if (a.cnt->done || loop_limit_reached(a.cnt, c.N, c.L)) return;
    float m = 0.0f;
    if (a.cnt->passes == 0) {
        for (int i = blk * 256 + threadIdx.x; i < c.L; i += nblk * 256) {
            int n;
            const float e = leaf_error<D>(a, i, &n);
            a.err[i] = e;
            m = fmaxf(m, e);
        }
    } else {
        // one thread per split: both children from the split's entry
        // (sample indices and volumes), not from their leaf records
        for (int t = blk * 256 + threadIdx.x; t < c.new_n; t += nblk * 256) {
            const int4 s0 = a.sdat[2 * t], s1 = a.sdat[2 * t + 1];
            const int il = a.split_list[t];
            LeafSamples lsl, lsr;
            const int idl[4] = {s0.x, s0.y, -1, -1};
            const int idr[4] = {s0.z, s0.w, s1.x, -1};
            load_values(a, idl, lsl);  // the five value loads together
            load_values(a, idr, lsr);
            const float el = error_of_values(idl, __int_as_float(s1.y), lsl);
            const float er = error_of_values(idr, __int_as_float(s1.z), lsr);
            a.err[il] = el;
            a.err[c.L_old + t] = er;
            m = fmaxf(m, el);
            m = fmaxf(m, er);
        }
    }
    super_max(a.smax + par * kSuper, m, blk);
}

template <int D>
__global__ __launch_bounds__(256) void k_errors(DevGrid a, int par) {
    errors_body<D>(a, blockIdx.x, gridDim.x, par);
}
template <int D>
__global__ __launch_bounds__(256) void k_errors_b(const DevGrid* __restrict__ grids, int par) {
    const DevGrid a = batch_grid(grids);
    errors_body<D>(a, blockIdx.x, gridDim.x, par);
}

// --------------------------------------------------------------- selection --
// Chunks a tree of L leaves is cut into, of the n launched (the others
// return): 256 leaves each until four workgroups per CU have one, then up to
// 512 before there are more of them, so that the 16 % or so that a pass selects
// fill their waves.  Runs without reconstruction, against 256 leaves up to 4096
// chunks: 333x517 884 -> 773 us, 3D 256x256 809 -> 740 us, 1080p the same; at
// least 1024 leaves (795 us) or 512 chunks (880 us) were slower at 333x517.
// One for a tree without leaves (an uploaded state): its pass adds nothing, and
// is reported like any other.
__device__ __forceinline__ int live_chunks(int L, int n) {
    return min(n, max(max(min((L + 255) / 256, 1024), L / 512), 1));
}

// kdgrid.cu:316-326.  Per leaf: the seed (tea4(i,0) when unset), one draw u,
// selected iff pow(err / g_error, alpha) >= u.  A selected full leaf splits.
// Writes the flags, and per chunk the (selected, split) counts and the
// samples held by the selected leaves, also added to the chunk's super group;
// the max error of the leaves that do not split goes on to the next pass
// (carried: null for single calls, whose next error pass sees every leaf).
// The LCG states are not written here: the compaction stores them once it has
// accepted the pass, so that a pass refused for capacity leaves every state
// as it was.
// Chunk blk of nblk (the compaction's partition of the leaves).
__device__ __forceinline__ void select_chunk(const DevGrid& a, int L, float gmax_part, int blk, int nblk,
                                             SuperSum* ssum, SuperMax* carried) {
    __shared__ int red[12];
    __shared__ float rmax[4];
    const float alpha = a.alpha;
    int beg, end;
    chunk_range(L, nblk, blk, beg, end);
    int ns = 0, nl = 0, nc = 0;
    float carry = 0.0f;
    // four leaves per thread and step, their loads issued together
    constexpr int U = 4;
    for (int t0 = beg; t0 < end; t0 += U * 256) {  // uniform: every lane takes part in wave_max
        const int i0 = t0 + (int)threadIdx.x;
        float ev[U];
        unsigned sv[U], fv[U];
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const int i = i0 + r * 256;
            if (i < end) {
                ev[r] = a.err[i];
                sv[r] = a.seed[i];
                fv[r] = a.flags[i];
            }
        }
        const float gmax = wave_max(gmax_part);  // each a maximum from 0, or all an uploaded g_error
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const int i = i0 + r * 256;
            if (i >= end) continue;
            const float e = ev[r];
            unsigned s = sv[r];
            if (s == 0u) s = tea4((unsigned)i, 0u);
            const float u = rnd(s);
            const bool sel = select_test(e / gmax, alpha, u);
            const unsigned cnt = fv[r] & 7u;
            const bool split = sel && cnt == 4u;
            a.flags[i] = (unsigned char)(cnt | (sel ? 8u : 0u) | (split ? 16u : 0u));
            ns += sel ? 1 : 0;
            nl += split ? 1 : 0;
            nc += sel ? (int)cnt : 0;
            if (!split) carry = fmaxf(carry, e);
        }
    }
    ns = wave_sum(ns);
    nl = wave_sum(nl);
    nc = wave_sum(nc);
    carry = wave_max(carry);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = ns;
        red[4 + (threadIdx.x >> 6)] = nl;
        red[8 + (threadIdx.x >> 6)] = nc;
        rmax[threadIdx.x >> 6] = carry;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const float cm = fmaxf(fmaxf(rmax[0], rmax[1]), fmaxf(rmax[2], rmax[3]));
        const int4 p = make_int4(red[0] + red[1] + red[2] + red[3], red[4] + red[5] + red[6] + red[7],
                                 red[8] + red[9] + red[10] + red[11], 0);
        a.part[blk] = p;
        const int g = blk / super_size(nblk);
        if (p.x != 0) atomicAdd(&ssum[g].sel, p.x);
        if (p.y != 0) atomicAdd(&ssum[g].split, p.y);
        if (p.z != 0) atomicAdd(&ssum[g].held, p.z);
        if (carried != nullptr && cm != 0.0f) atomicMax(&carried[g].err, __float_as_uint(cm));
    }
    __syncthreads();  // red / rmax are reused by the workgroup's next chunk
}
// Workgroup blk takes chunks [blk * cpw, (blk + 1) * cpw) of the compaction's
// n: the placement balances better over many small chunks, the selection's
// streaming sweep runs best with fewer, longer ones.  In the loop the stopping
// test and the largest error of the pass come first, from the pass's slot and
// totals (a single call selects against g_error as it stands).
__device__ __forceinline__ void select_body(const DevGrid& a, int blk, int n, int cpw, int par, int loop) {
    // the counts and the totals in one round of loads, the first leaves next,
    // their reduction after those are out (64x48 4.6 -> 4.1 us a pass, 4D 1080p
    // 18.6 -> 17.8)
    DevCounters* cn = a.cnt;
    const int done = cn->done, passes = cn->passes, lane = threadIdx.x & 63;
    const TreeCounts c = cn->slot[par];
    const unsigned e = a.smax[(loop ? par : kGError) * kSuper + lane].err;
    if (done) return;
    if (loop && loop_limit_reached(cn, c.N, c.L)) {  // every workgroup finds the same
        if (blk == 0 && threadIdx.x == 0) cn->done = 1;
        return;
    }
    n = live_chunks(c.L, n);
    if (blk * cpw >= n) return;
    for (int k = blk * cpw; k < min(n, (blk + 1) * cpw); ++k)
        select_chunk(a, c.L, __uint_as_float(e), k, n, a.ssum + par * kSuper,
                     loop ? a.smax + (par ^ 1) * kSuper : nullptr);
    if (loop && blk == 0 && threadIdx.x < kSuper) {
        a.smax[kGError * kSuper + lane].err = e;  // g_error of this pass, for the calls after the loop
        if (lane == 0 && a.lrows != nullptr && passes > 0) *a.lrows += c.new_n;  // collected by the error pass
    }
}
__global__ __launch_bounds__(256) void k_select(DevGrid a, int n, int cpw, int par, int loop) {
    select_body(a, blockIdx.x, n, cpw, par, loop);
}
__global__ __launch_bounds__(256) void k_select_b(const DevGrid* __restrict__ grids, int n, int cpw, int par) {
    const DevGrid a = batch_grid(grids);
    select_body(a, blockIdx.x, n, cpw, par, 1);
}

// Chunks per selection workgroup for `chunks` compaction chunks: as many as
// keep the selection at 4096 workgroups (chunks is then a multiple of it).
static int select_cpw(int chunks) { return chunks > 4096 && chunks % 4096 == 0 ? chunks / 4096 : 1; }

// ----------------------------------------------------- placement and split --
// kdgrid.cu:328-477 for one selected leaf: best candidate among
// candidatesNum uniform points of the box (max over candidates of the min
// Euclidean distance to the leaf's samples, earliest wins ties), appended at
// sample index k, the draws starting from LCG state s; a full leaf is split
// at the median of its 5 samples along the largest box axis, keeping the left
// half in place and the right half at leaf index m.
// With a scene B (MODE != PLACE_ONLY; its objects in LDS at obj) the new
// sample is evaluated here, and with PLACE_ERRORS a split's children get their
// errors here, from the leaf's values and the new one, in place of the next
// pass's error kernel; emax takes the larger.
template <int D, int MODE>
__device__ __forceinline__ void place_leaf(const DevGrid& a, int i, int k, int m, unsigned cnt,
                                           int L, unsigned s, const mscene::SceneBlock* B,
                                           const float* obj, float& emax) {
    constexpr int P = line_pts(D);
    // the leaf's line: slots, box and its first points, one 128-byte read
    float f[kLineFloats];
    load_line(a, i, f);
    // the overflow row (points past the line, the slots beside them) only
    // when the leaf holds those points
    constexpr int XS = xpts_stride(D) > 0 ? xpts_stride(D) : 4;
    float x[XS];
#pragma unroll
    for (int t = 0; t < XS; ++t) x[t] = 0.0f;
    if constexpr (P < 4) {
        if (cnt > (unsigned)P) {
            const float4* xr = reinterpret_cast<const float4*>(a.xpts + (size_t)i * xpts_stride(D));
#pragma unroll
            for (int t = 0; t < XS / 4; ++t) {
                const float4 v = xr[t];
                x[4 * t] = v.x;
                x[4 * t + 1] = v.y;
                x[4 * t + 2] = v.z;
                x[4 * t + 3] = v.w;
            }
        }
    }
    // slots past the leaf's count are stale: -1
    int ids[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int at = slot_at(D, q);
        const int v = at >= 0 ? __float_as_int(f[at]) : __float_as_int(x[-1 - at]);
        ids[q] = q < (int)cnt ? v : -1;
    }
    float mn[D], mx[D], diag[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        mn[d] = f[4 + d];
        mx[d] = f[4 + D + d];
        diag[d] = mx[d] - mn[d];
    }
    // the points by slot (the floats of empty slots are replaced, never used
    // in arithmetic); those past the line only when the leaf holds them
    float p[4][D];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int d = 0; d < D; ++d)
            p[q][d] = ids[q] < 0 ? 0.0f : (q < P ? f[line_pt(D, q) + d] : x[xpt_at(D, q) + d]);
    float maxDist = -1.0f;
    float best[D];
#pragma unroll
    for (int d = 0; d < D; ++d) best[d] = 0.0f;
    for (int j = 0; j < a.cand; ++j) {
        float c[D];
#pragma unroll
        for (int d = 0; d < D; ++d) c[d] = rnd(s);
#pragma unroll
        for (int d = 0; d < D; ++d) c[d] = mn[d] + c[d] * diag[d];
        // min over samples of sqrt(d2) = sqrt(min over samples of d2), since
        // sqrt is monotone and correctly rounded; one sqrt per candidate.
        float minD2 = __int_as_float(0x7f800000);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (ids[q] >= 0) {
                float acc = 0.0f;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    float t = c[d] - p[q][d];
                    acc += t * t;
                }
                if (minD2 > acc) minD2 = acc;
            }
        }
        const float minDist = minD2 < __int_as_float(0x7f800000) ? __builtin_sqrtf(minD2)
                                                                 : 3.402823466e+38f;
        if (maxDist < minDist) {
            maxDist = minDist;
#pragma unroll
            for (int d = 0; d < D; ++d) best[d] = c[d];
        }
    }
    float* out = a.coords + (size_t)k * D;
#pragma unroll
    for (int d = 0; d < D; ++d) __builtin_nontemporal_store(best[d], out + d);
    int kid[5] = {k, k, k, k, k};     // PLACE_ERRORS: a split's samples in sorted order,
    float vol_l = 0.0f, vol_r = 0.0f;  // its children's volumes
    if (cnt < 4u) {
        // kdgrid.cu:393-396: insert into the first free slot; the error is kept
        store_point_slot<D>(a, i, (int)cnt, best, k);
    } else {
        // kdgrid.cu:399-471: split.  LargestAxis scans from the last axis down
        // with a strict '<' (aabb.h:34-45).
        int axis = -1;
        float ext = -3.402823466e+38f;
#pragma unroll
        for (int d = D - 1; d >= 0; --d)
            if (ext < diag[d]) {
                ext = diag[d];
                axis = d;
            }
        float key[5];
        int v[5] = {ids[0], ids[1], ids[2], ids[3], k};
        int perm[5] = {0, 1, 2, 3, 4};  // which of p[0..3], best sits at each position
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float kv = p[q][0];
#pragma unroll
            for (int d = 1; d < D; ++d)
                if (d == axis) kv = p[q][d];
            key[q] = kv;
        }
        {
            float kv = best[0];
#pragma unroll
            for (int d = 1; d < D; ++d)
                if (d == axis) kv = best[d];
            key[4] = kv;
        }
        // stable bubble sort, strict '>' swaps (kdgrid.cu:409-417)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int q = 0; q < 4 - r; ++q) {
                if (key[q] > key[q + 1]) {
                    float tk = key[q];
                    key[q] = key[q + 1];
                    key[q + 1] = tk;
                    int tv = v[q];
                    v[q] = v[q + 1];
                    v[q + 1] = tv;
                    tv = perm[q];
                    perm[q] = perm[q + 1];
                    perm[q + 1] = tv;
                }
            }
        }
        const float pos = 0.5f * (key[1] + key[2]);
        const int E = ~D;
        float cmn[D], cmx[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            cmn[d] = d == axis ? pos : mn[d];
            cmx[d] = d == axis ? pos : mx[d];
        }
        // the points by sorted position: 0, 1 -> left child, 2..4 -> right
        float sp[5][D];
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
            for (int d = 0; d < D; ++d) {
                float x = best[d];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (perm[j] == q) x = p[q][d];
                sp[j][d] = x;
            }
        // the left child in the parent's line (slots, box, two points: whole
        // float4s, the rest stays, past the child's count of 2), the right child's
        // whole line, and its third point in its overflow row when the line
        // holds two (D = 6)
        store_line_head2<D>(a, i, make_int4(v[0], v[1], E, E), mn, cmx, sp[0], sp[1]);
        store_line<D>(a, m, make_int4(v[2], v[3], v[4], E), cmn, mx, &sp[2], 3);
        if constexpr (P < 3) store_point_slot<D>(a, m, 2, sp[4], v[4]);  // D = 6: overflow row
        if constexpr (MODE == PLACE_ERRORS) {
#pragma unroll
            for (int j = 0; j < 5; ++j) kid[j] = v[j];
            vol_l = box_volume<D>(mn, cmx);
            vol_r = box_volume<D>(cmn, mx);
        } else {
            // what the next error pass needs of both children, coalesced by
            // split rank: their sample indices and box volumes
            a.sdat[2 * (m - L)] = make_int4(v[0], v[1], v[2], v[3]);
            a.sdat[2 * (m - L) + 1] = make_int4(v[4], __float_as_int(box_volume<D>(mn, cmx)),
                                                __float_as_int(box_volume<D>(cmn, mx)), 0);
            if (a.sext) {  // learned mode: the children's extents for their features
                float ex[6];
#pragma unroll
                for (int d = 0; d < 6; ++d) ex[d] = d < D ? (d == axis ? cmx[d] - mn[d] : diag[d]) : 0.0f;
                a.sext[2 * (m - L)] = make_int4(__float_as_int(ex[0]), __float_as_int(ex[1]),
                                                __float_as_int(ex[2]), __float_as_int(ex[3]));
                float right = 0.0f;
#pragma unroll
                for (int d = 0; d < D; ++d)
                    if (d == axis) right = mx[d] - cmn[d];
                a.sext[2 * (m - L) + 1] = make_int4(__float_as_int(ex[4]), __float_as_int(ex[5]),
                                                    __float_as_int(right), axis);
            }
            if (!a.in_loop) {  // in the loop the next error pass overwrites both
                a.err[i] = -1.0f;
                a.err[m] = -1.0f;
            }
        }
        a.seed[m] = 0u;
        a.flags[m] = 3;
        a.split_list[m - L] = i;  // the split leaves in leaf order (right child m)
    }
    // the leaf's own state (already jumped) and count were written by the
    // selection and compaction kernels
    if constexpr (MODE != PLACE_ONLY) {
        // the line's stores are out and its registers free; a split's other
        // samples' values come after the new one (held meanwhile, their registers
        // cost a wave per SIMD)
        const bool split = MODE == PLACE_ERRORS && cnt == 4u;
        float xe[6];
#pragma unroll
        for (int d = 0; d < 6; ++d) xe[d] = d < D ? best[d] : 0.0f;
        const mscene::V3<float> val =
            mscene::eval<float>(B->p, obj, xe, &B->accel, &B->cells, reinterpret_cast<const uint64_t*>(B + 1));
        float* vo = a.values + (size_t)k * 3;
        vo[0] = val.x;
        vo[1] = val.y;
        vo[2] = val.z;
        LeafSamples ch[2];
        if (split) {
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                const float* o = a.values + (size_t)(kid[j] == k ? kid[j == 0 ? 1 : 0] : kid[j]) * 3;
                LeafSamples& c = ch[j < 2 ? 0 : 1];
                const int q = j < 2 ? j : j - 2;
                c.vx[q] = o[0];
                c.vy[q] = o[1];
                c.vz[q] = o[2];
            }
        }
        if (split) {
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                LeafSamples& c = ch[j < 2 ? 0 : 1];
                const int q = j < 2 ? j : j - 2;
                c.vx[q] = kid[j] == k ? val.x : c.vx[q];
                c.vy[q] = kid[j] == k ? val.y : c.vy[q];
                c.vz[q] = kid[j] == k ? val.z : c.vz[q];
            }
            const int two[4] = {0, 0, -1, -1}, three[4] = {0, 0, 0, -1};
            const float el = error_of_values(two, vol_l, ch[0]);
            const float er = error_of_values(three, vol_r, ch[1]);
            a.err[i] = el;
            a.err[m] = er;
            emax = fmaxf(emax, fmaxf(el, er));
        }
    }
}

// Where chunk blk's new samples and right children start (base: ranks among
// all selected and split leaves), from the super groups and the partials of
// its own group; every wave computes it for itself.  False if the pass would
// exceed the capacity.  One thread writes the next slot, a wave the totals' zeros
// for the pass after (no kernel of this pass reads those) and, into the host's
// memory, the pass's statistics in a loop, which knows before the placement
// itself whether another pass follows, or a single call's counters.
// s, P and t (the lane's super group) are loaded by the caller, together.  Only
// PLACE_ONLY runs outside a loop too.
template <int MODE>
__device__ __forceinline__ bool pass_offsets(const DevGrid& a, int blk, int nblk, int par, const TreeCounts& s,
                                             int P, const int3& t, int2& base) {
    DevCounters* cn = a.cnt;
    const int L = s.L, N = s.N;
    const int lane = threadIdx.x & 63;
    const int per = super_size(nblk), g = blk / per;
    int2 own = make_int2(0, 0);
    for (int c = g * per + lane; c < blk; c += 64) {
        const int4 p = a.part[c];
        own.x += p.x;
        own.y += p.y;
    }
    const int sel = wave_sum(t.x), split = wave_sum(t.y);
    const bool fits = (long long)N + sel <= a.cap_s && (long long)L + split <= a.cap_l;
    if (blk == 0 && threadIdx.x < kSuper) {
        const int held = wave_sum(t.z);
        // leaves whose errors were estimated since the last pass, and the
        // values that took: the initial leaves, then the children
        const int stale = P == 0 ? L : 2 * s.new_n, vals = P == 0 ? 4 * L : 5 * s.new_n;
        const bool in_loop = MODE != PLACE_ONLY || a.in_loop != 0;
        if (in_loop && lane < kPassWords) {
            const int w[kPassWords] = {L, N, sel, split, held, stale, vals, fits ? 0 : MDAS_ERR_CAPACITY_DEV};
            int v = 0;
#pragma unroll
            for (int q = 0; q < kPassWords; ++q) v = lane == q ? w[q] : v;
            __hip_atomic_store(&a.hrun->row[P & (kHostRows - 1)][lane],
                               ((unsigned long long)(a.htag + (unsigned)P) << 32) | (unsigned)v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (fits) {
            SuperSum& z = a.ssum[(par ^ 1) * kSuper + lane];
            z.sel = z.split = z.held = 0;
            a.smax[par * kSuper + lane].err = 0u;  // the selection has read them
        }
        if (lane == 0) {
            if (!fits) {
                cn->status = MDAS_ERR_CAPACITY_DEV;
                cn->done = 1;
            } else {
                cn->passes = P + 1;
                cn->slot[par ^ 1] = TreeCounts{N + sel, L + split, N, L, sel, split};
                cn->cur = par ^ 1;
            }
            if (!in_loop) a.hrun->cnt = *cn;
        }
    }
    if (!fits) return false;
    base.x = wave_sum(own.x + (lane < g ? t.x : 0));
    base.y = wave_sum(own.y + (lane < g ? t.y : 0));
    return true;
}

// Compaction and placement in one kernel.  Each workgroup ranks the selected
// leaves of its chunk (the selection's partition) in leaf order by wave
// ballots: a leaf of global rank r (r = the rank among all selected leaves)
// gets the new sample N_old + r, a split leaf of split rank q the right child
// L_old + q.  The entries (leaf | count << 30, right child or -1; leaf
// indices are below 2^30, a split leaf's count is 4) and the LCG states
// they start from queue up in LDS and are placed a round of 256 at a time,
// one per thread.  Every leaf's count and LCG state are rewritten in the
// same sweep, as they stand after the placement, in full coalesced lines.
// What bounds it at 1080p is the traffic of its scattered lines (5D, 39
// passes: 800 MB a pass of 238 us, 3/4 of a copy's rate) and, beside it, the vector units, half
// the time busy with some 3000 instructions per 64 new samples, a third of them
// the integrand's; a small tree's pass is the chain of its launches and of one
// leaf's work.  So the loads before the first leaf go out in two rounds, what
// the kernel does not write it reads through the scalar cache (the scene's
// 105 uniform loads in the integrand were vector loads, each waited for; a batch
// read its pointers as flat ones and spilled 20 registers), and registers are
// held to five waves: 4D 1080p 8.26 -> 7.50 ms a run, 5D 13.78 -> 13.65, batch of
// eight 12.48 -> 10.73, 333x517 840 -> 796 us (both timed in turn on one card,
// reconstruction included).  Taking the integrand and the
// children's errors along saves two launches of four and the split entries: 5D
// 1080p (1.5 M leaves a pass) 15.6 -> 14.6 ms a run, 64x48 (12 passes of 2000)
// 617 -> 457 us, 3D 256x256 1240 -> 861 us.  One chunk per wave in place of one
// per workgroup (fewer barriers, 4x the chunks) was slower at 1080p (12.0 ->
// 12.9 ms a run at its best count) and no faster below.  What streams through
// once, the flags and states of the sweep and the new coordinates, goes past
// the caches (5D 14.27 -> 13.86 ms, 333x517 829 -> 820 us); a line's float4s,
// several accesses each, must not (loads 17.6 ms, stores 15.2).
// MODE: see place_leaf.  The offsets come from the super groups' totals and
// the partials of the chunk's own group; every workgroup finds the same
// totals, so a pass beyond the capacity writes nothing.
template <int D, int MODE>
__device__ __forceinline__ void compact_place_body(const DevGrid& a, int blk, int nblk, int par,
                                                   const mscene::SceneBlock* B, float* obj) {
    constexpr int U = 4;                   // tiles whose flags and states are loaded together
    constexpr int QCAP = U * 256 + 256;    // one step's entries plus an unplaced remainder
    __shared__ int lds[8];
    __shared__ int2 qe[QCAP];
    __shared__ unsigned qs[QCAP];
    // two rounds of loads before the first leaf's line: the counts and totals,
    // then the partials, the scene's objects and the first flags and states
    const int done = a.cnt->done, P = a.cnt->passes;
    const TreeCounts s = a.cnt->slot[par];
    const int lane = threadIdx.x & 63;
    const SuperSum& ts_ = a.ssum[par * kSuper + lane];
    const int3 t = make_int3(ts_.sel, ts_.split, ts_.held);
    int n_obj = 0;
    if constexpr (MODE != PLACE_ONLY) n_obj = B->p.n_obj;
    if (done) return;
    nblk = live_chunks(s.L, nblk);
    if (blk >= nblk) return;
    const int L = s.L, N0 = s.N;
    int beg, end;
    chunk_range(L, nblk, blk, beg, end);
    unsigned fv[U], sv[U];
    auto load_tiles = [&](int t00) {
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const int i = t00 + r * 256 + threadIdx.x;
            fv[r] = i < end ? __builtin_nontemporal_load(a.flags + i) : 0u;
            sv[r] = i < end ? __builtin_nontemporal_load(a.seed + i) : 0u;
        }
    };
    load_tiles(beg);
    if constexpr (MODE != PLACE_ONLY) {
        for (int q = threadIdx.x; q < n_obj * mscene::OBJ_STRIDE; q += 256) obj[q] = B->p.obj[q];
    }
    int2 base;
    if (!pass_offsets<MODE>(a, blk, nblk, par, s, P, t, base)) return;
    float emax = 0.0f;
    int jq = base.x;  // global rank of the entry at the front of the queue
    int qn = 0;       // queued entries
    auto place_round = [&](int p0, int count) {
        const int p = p0 + (int)threadIdx.x;
        if ((int)threadIdx.x < count) {
            const int2 q = qe[p];
            const unsigned cnt = q.y >= 0 ? 4u : ((unsigned)q.x >> 30);
            place_leaf<D, MODE>(a, q.x & 0x3fffffff, N0 + jq + p, q.y, cnt, L, qs[p], B, obj, emax);
        }
    };
    for (int t00 = beg; t00 < end; t00 += U * 256) {
        if (t00 > beg) load_tiles(t00);
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const int t0 = t00 + r * 256;
            if (t0 >= end) break;  // uniform across the workgroup
            const int i = t0 + threadIdx.x;
            const unsigned f = fv[r];
            const bool sel = (f & 8u) != 0u, split = (f & 16u) != 0u;
            const unsigned cnt = f & 7u;
            int rs, rl, ts, tl;
            block_rank2(sel, split, lds, rs, rl, ts, tl);
            // the state after the selection's draw (kdgrid.cu:323-326): the
            // placement starts from it, and a selected leaf's stored state is
            // the one after the candidatesNum * D candidate draws (the LCG's
            // affine jump-ahead)
            unsigned s1 = sv[r];
            if (s1 == 0u) s1 = tea4((unsigned)i, 0u);
            s1 = 1664525u * s1 + 1013904223u;
            if (sel) {
                qe[qn + rs] = make_int2(i | (int)((cnt & 3u) << 30), split ? L + base.y + rl : -1);
                qs[qn + rs] = s1;
            }
            if (i < end) {
                __builtin_nontemporal_store((unsigned char)(split ? 2u : (sel ? cnt + 1u : cnt)), a.flags + i);
                __builtin_nontemporal_store(sel ? a.jmul * s1 + a.jadd : s1, a.seed + i);
            }
            qn += ts;
            base.y += tl;
        }
        __syncthreads();
        int placed = 0;
        for (; qn - placed >= 256; placed += 256) place_round(placed, 256);
        if (placed > 0) {  // the remainder (< 256) to the front of the queue
            const int rem = qn - placed;
            int2 e = make_int2(0, 0);
            unsigned st = 0u;
            if ((int)threadIdx.x < rem) {
                e = qe[placed + threadIdx.x];
                st = qs[placed + threadIdx.x];
            }
            __syncthreads();
            if ((int)threadIdx.x < rem) {
                qe[threadIdx.x] = e;
                qs[threadIdx.x] = st;
            }
            jq += placed;
            qn = rem;
        }
        __syncthreads();
    }
    place_round(0, qn);
    if constexpr (MODE == PLACE_ERRORS) {
        emax = wave_max(emax);
        if (lane == 0 && emax != 0.0f)
            atomicMax(&a.smax[(par ^ 1) * kSuper + blk / super_size(nblk)].err, __float_as_uint(emax));
    }
}

// The scene's objects in dynamic LDS (48 bytes each).  The registers are held to
// five waves per SIMD, which nothing spills for (4D 1080p, 57 passes: a run takes
// 6 % more with four, 8 % more with six, which spill); a 6D leaf needs the
// registers of four.
template <int D, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 6 ? 4 : 5))) void k_compact_place(
    DevGrid a, const mscene::SceneBlock* B, int par) {
    extern __shared__ float obj[];
    compact_place_body<D, MODE>(a, blockIdx.x, gridDim.x, par, in_constant(B), obj);
}
template <int D, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 6 ? 4 : 5))) void k_compact_place_b(
    const DevGrid* __restrict__ grids, const void* const* __restrict__ params, int par) {
    extern __shared__ float obj[];
    const DevGrid a = batch_grid(grids);
    compact_place_body<D, MODE>(a, blockIdx.x, gridDim.x, par,
                                in_constant((const mscene::SceneBlock*)params[blockIdx.y]), obj);
}

// The loop's state per image: finished once `done` or at the limit, so that the
// host need not launch another pass to learn it.
__global__ void k_loop_status_b(const DevGrid* grids, int n, int* out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const DevCounters* c = grids[t].cnt;
    const TreeCounts s = tree_counts(c);
    out[4 * t] = c->done || loop_limit_reached(c, s.N, s.L);
    out[4 * t + 1] = c->status;
    out[4 * t + 2] = s.N;
    out[4 * t + 3] = c->passes;
}

// After the device-side loop: when it stopped at its limit, no error pass
// followed the last placement, so its split children get the stale marker
// (error -1, kdgrid.cu:466-469) the placement left out.  Raises `done`, and
// leaves the counters to the host.
__device__ __forceinline__ void mark_last_children_body(const DevGrid& a, int blk, int nblk) {
    DevCounters* c = a.cnt;
    const TreeCounts s = tree_counts(c);
    const bool stopped = c->status == 0 && loop_limit_reached(c, s.N, s.L);
    if (blk == 0 && threadIdx.x == 0) {
        if (stopped) c->done = 1;
        a.hrun->cnt = *c;
    }
    if (!stopped) return;
    for (int t = blk * 256 + threadIdx.x; t < s.new_n; t += nblk * 256) {
        a.err[a.split_list[t]] = -1.0f;
        a.err[s.L_old + t] = -1.0f;
    }
}
__global__ __launch_bounds__(256) void k_mark_last_children(DevGrid a) {
    mark_last_children_body(a, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(256) void k_mark_last_children_b(const DevGrid* grids) {
    mark_last_children_body(batch_grid(grids), blockIdx.x, gridDim.x);
}

// One wave; the errors are not below 0, so their bits are ordered as they are
// (an uploaded g_error, which may be, is the same in every group).  A copy of
// the groups' 8 KB took 24 us, one of the counters alone, as before, 21, this 12.
__global__ __launch_bounds__(kSuper) void k_report(DevGrid a) {
    unsigned m = a.smax[kGError * kSuper + threadIdx.x].err;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    if (threadIdx.x != 0) return;
    a.hrun->g_error = m;
    a.hrun->cnt = *a.cnt;
}

// The leaves' points in their lines and overflow rows from the sample
// coordinates (after a state upload).
template <int D>
__global__ __launch_bounds__(256) void k_build_pts(DevGrid a, int L) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < L; i += gridDim.x * 256) {
        const int4 id = load_slots<D>(a, i, leaf_count(a, i));
        const int ids[4] = {id.x, id.y, id.z, id.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (ids[q] >= 0 && ids[q] < a.cap_s) {
                float* dst = point_addr<D>(a, i, q);
#pragma unroll
                for (int d = 0; d < D; ++d) dst[d] = a.coords[(size_t)ids[q] * D + d];
            }
        }
    }
}

// --------------------------------------------------------------- fills --
__global__ void k_fill_f32(float* p, float v, long long n) {
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (long long)gridDim.x * 256) p[i] = v;
}

// ------------------------------------------------------------ launchers --
static int grid_for(long long n, int cap_blocks = 8192) {
    long long b = (n + 255) / 256;
    if (b < 1) b = 1;
    if (b > cap_blocks) b = cap_blocks;
    return (int)b;
}

#define MDAS_DISPATCH_D(D_, STMT)                      \
    switch (D_) {                                      \
    case 3: { constexpr int DD = 3; STMT; } break;     \
    case 4: { constexpr int DD = 4; STMT; } break;     \
    case 5: { constexpr int DD = 5; STMT; } break;     \
    case 6: { constexpr int DD = 6; STMT; } break;     \
    default: return hipErrorInvalidValue;              \
    }

hipError_t launch_initial(Grid& g, int L0, int limit, hipStream_t st) {
    const int blocks = grid_for(L0, 4096);
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_initial<DD>, dim3(blocks), dim3(256), 0, st, g.dev, L0));
    hipLaunchKernelGGL(k_initial_counters, dim3(1), dim3(kMaxSets * kSuper), 0, st, g.dev, L0, limit);
    return hipGetLastError();
}

hipError_t launch_arm(Grid& g, bool errors, bool adaptive, hipStream_t st) {
    hipLaunchKernelGGL(k_arm, dim3(1), dim3(kSuper), 0, st, g.dev, errors ? 1 : 0, adaptive ? 1 : 0, g.host.cur);
    return hipGetLastError();
}

hipError_t launch_compute_errors(Grid& g, hipStream_t st) {
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_compute_errors<DD>, dim3(g.error_blocks()), dim3(256), 0, st, g.dev));
    return hipGetLastError();
}

hipError_t launch_errors(Grid& g, int parity, hipStream_t st) {
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_errors<DD>, dim3(g.error_blocks()), dim3(256), 0, st, g.dev, parity));
    return hipGetLastError();
}

static hipError_t select_chunks(Grid& g, int parity, int loop, hipStream_t st) {
    const int n = g.chunks(), cpw = select_cpw(n);
    hipLaunchKernelGGL(k_select, dim3(n / cpw), dim3(256), 0, st, g.dev, n, cpw, parity, loop);
    return hipGetLastError();
}
hipError_t launch_select(Grid& g, int parity, hipStream_t st) { return select_chunks(g, parity, 1, st); }

#define MDAS_DISPATCH_PLACE(D_, MODE_, KERNEL, ...)                                                    \
    switch (MODE_) {                                                                                   \
    case PLACE_ONLY: MDAS_DISPATCH_D(D_, hipLaunchKernelGGL((KERNEL<DD, PLACE_ONLY>), __VA_ARGS__)); break;     \
    case PLACE_EVAL: MDAS_DISPATCH_D(D_, hipLaunchKernelGGL((KERNEL<DD, PLACE_EVAL>), __VA_ARGS__)); break;     \
    default: MDAS_DISPATCH_D(D_, hipLaunchKernelGGL((KERNEL<DD, PLACE_ERRORS>), __VA_ARGS__)); break;           \
    }

hipError_t launch_place(Grid& g, int parity, int mode, const void* dparams, int n_obj, hipStream_t st) {
    const size_t lds = mode == PLACE_ONLY ? 0 : n_obj * mscene::OBJ_STRIDE * sizeof(float);
    MDAS_DISPATCH_PLACE(g.D, mode, k_compact_place, dim3(g.chunks()), dim3(256), lds, st, g.dev,
                        (const mscene::SceneBlock*)dparams, parity);
    return hipGetLastError();
}

hipError_t launch_adaptive(Grid& g, hipStream_t st) {
    const int parity = g.host.cur;  // where launch_arm has put the counts
    hipError_t e = select_chunks(g, parity, 0, st);
    if (e == hipSuccess) e = launch_place(g, parity, PLACE_ONLY, nullptr, 0, st);
    return e;
}

hipError_t launch_mark_last_children(Grid& g, hipStream_t st) {
    hipLaunchKernelGGL(k_mark_last_children, dim3(g.error_blocks()), dim3(256), 0, st, g.dev);
    return hipGetLastError();
}

hipError_t launch_mark_last_children_b(const DevGrid* grids, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_mark_last_children_b, dim3(256, n), dim3(256), 0, st, grids);
    return hipGetLastError();
}

hipError_t launch_report(Grid& g, hipStream_t st) {
    hipLaunchKernelGGL(k_report, dim3(1), dim3(kSuper), 0, st, g.dev);
    return hipGetLastError();
}

hipError_t launch_build_pts(Grid& g, int n_leaves, hipStream_t st) {
    if (n_leaves <= 0) return hipSuccess;
    const int blocks = grid_for(n_leaves, 4096);
    MDAS_DISPATCH_D(g.D, hipLaunchKernelGGL(k_build_pts<DD>, dim3(blocks), dim3(256), 0, st, g.dev, n_leaves));
    return hipGetLastError();
}

hipError_t launch_fill_f32(float* p, float v, long long n, hipStream_t st) {
    hipLaunchKernelGGL(k_fill_f32, dim3(grid_for(n)), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

// ------------------------------------------------------ batched launchers --
// `grids` is a device array of n DevGrid of one dimension D; every chunked
// kernel gives each image `blocks` workgroups (<= kChunkBlocks).
hipError_t launch_initial_b(int D, const DevGrid* grids, int n, int blocks, const int* limits,
                            hipStream_t st) {
    MDAS_DISPATCH_D(D, hipLaunchKernelGGL(k_initial_b<DD>, dim3(blocks, n), dim3(256), 0, st, grids));
    hipLaunchKernelGGL(k_initial_counters_b, dim3(n), dim3(kMaxSets * kSuper), 0, st, grids, limits);
    return hipGetLastError();
}

hipError_t launch_errors_b(int D, const DevGrid* grids, int n, int blocks, int parity, hipStream_t st) {
    MDAS_DISPATCH_D(D, hipLaunchKernelGGL(k_errors_b<DD>, dim3(blocks < 1024 ? blocks : 1024, n), dim3(256), 0, st,
                                          grids, parity));
    return hipGetLastError();
}

hipError_t launch_select_b(const DevGrid* grids, int n, int blocks, int parity, hipStream_t st) {
    const int cpw = select_cpw(blocks);
    hipLaunchKernelGGL(k_select_b, dim3(blocks / cpw, n), dim3(256), 0, st, grids, blocks, cpw, parity);
    return hipGetLastError();
}

hipError_t launch_place_b(int D, const DevGrid* grids, const void* const* params, int n_obj, int n,
                          int blocks, int parity, int mode, hipStream_t st) {
    const size_t lds = mode == PLACE_ONLY ? 0 : n_obj * mscene::OBJ_STRIDE * sizeof(float);
    MDAS_DISPATCH_PLACE(D, mode, k_compact_place_b, dim3(blocks, n), dim3(256), lds, st, grids, params, parity);
    return hipGetLastError();
}

hipError_t launch_loop_status_b(const DevGrid* grids, int n, int* out, hipStream_t st) {
    hipLaunchKernelGGL(k_loop_status_b, dim3((n + 63) / 64), dim3(64), 0, st, grids, n, out);
    return hipGetLastError();
}

}  // namespace mdas
