// MI355X (gfx950) cone-beam projector: forward ray march, volume VJP and
// 6-DoF pose VJP, FP32 and FP64 sampling, FP32/BF16/FP16 field storage.
//
// Semantics follow the reference kernels operation for operation:
//   FP32 sampling  kernels/projection_fp32.py:59-617
//   FP64 sampling  kernels/projection.py:79-296, 396-430, 802-1237
//   ray setup      kernels/projection.py:79-121 (FP64, once per ray)
//   pose algebra   kernels/geometry.py:13-74
// The translation unit is compiled with -ffp-contract=off; every FMA below is
// written explicitly (fmaf/fma).  Where the reference leaves a product-sum
// unmarked and its code generator (Warp, fuse_fp=True) fuses it, the fused form
// is written out, so the per-ray results are a fixed function of the inputs.
//
// Execution model (not the reference's): one launch covers all views.  A
// workgroup of 256 lanes owns one 16x16 detector tile of one view, or 8x8
// tiles of four consecutive views (one wave64 each); workgroup ids are
// remapped so each XCD walks a contiguous range of tiles.  Corners are
// gathered from the linear field (x-adjacent pairs) or from a copy (FP32: quads
// of 4 corners per plane, 16-bit: cells of 8; two or one 16-byte loads).  Pose cotangents are
// reduced per ray in FP64, across the wave with shuffles, then across tiles in
// a fixed-order FP64 pass.  Volume cotangents are a launch of their own: a lane
// steps from cell to cell along its ray, adds each cell's eight corner sums to
// an FP64 LDS brick of the slab of cells the workgroup is in, and the brick is
// drained into an FP64 accumulator with device atomics (vol_walk_kernel); rays
// whose factor f = seed * length * step lies outside [2^-102, 2^96] add the
// reference's per-increment RN(f * w), flushed to zero below 2^-126.  A final
// pass rounds the accumulator (plus the previous gradient when accumulating)
// once to FP32, or keeps FP64 for an FP64 destination.

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <cstdlib>
#include <algorithm>
#include <climits>
#include <mutex>
#include <type_traits>
#include <string>
#include <vector>

#include "../../include/dpt_amd.h"

#include "device_common.h"
#include "gather.h"

namespace dpt {

// ------------------------------------------------------- FP32 forward ------
// kernels/projection_fp32.py:334-374

template <typename T, bool COMPENSATED, int LAYOUT>
__global__ __launch_bounds__(kBlock) void forward32_kernel(Params P, const T *__restrict__ field,
                                                           float *__restrict__ out) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    if (!ray_in_range(P, view, row, col)) return;
    const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
    const double *pose = P.poses + 12 * (size_t)view;
    World w;
    ray_world(P, pose, view, row, col, w);
    Ray r;
    ray_grid(P, w, r);
    float o[3] = {(float)r.o[0], (float)r.o[1], (float)r.o[2]};
    float d[3] = {(float)r.d[0], (float)r.d[1], (float)r.d[2]};
    const float len = (float)r.len;
    if (!r.valid || !finite3f(o[0], o[1], o[2]) || !finite3f(d[0], d[1], d[2]) || !isfinite(len) ||
        len <= 0.0f) {
        flag(P, view, DPT_STATUS_RANGE);
        out[ray] = 0.0f;
        return;
    }
    const Interval32 iv = interval32(P, o, d);
    Acc<COMPENSATED> total;
    total.init();
    float result = 0.0f;
    if (iv.upper > iv.lower) {
        const float step = (iv.upper - iv.lower) / (float)P.samples;
        bool bad = false;
        // Lockstep sample walk with the current cell's corners cached in
        // registers: only lanes whose cell changed issue the (masked) loads.
        bad = !finite_span(o, d, iv.lower, step, 0, P.samples);
        float v[8];
        int cur = -1;
        auto walk = [&](auto interior, int k0, int k1, bool checked) {
            constexpr bool INTERIOR = decltype(interior)::value;
            for (int k = k0; k < k1; ++k) {
                if constexpr (COMPENSATED) {
                    if (k > 0 && (k % kFoldBlock) == 0) total.fold();
                }
                const float pos = fmaf(sample_centre(P, k), step, iv.lower);
                const float p0 = fmaf(pos, d[0], o[0]);
                const float p1 = fmaf(pos, d[1], o[1]);
                const float p2 = fmaf(pos, d[2], o[2]);
                Cell32 c;
                if constexpr (INTERIOR) {
                    cell32_interior(P, p0, p1, p2, c);
                } else {
                    if (checked && !inside32(P, p0, p1, p2)) continue;
                    cell32_inside(P, p0, p1, p2, c);
                }
                if (c.base != cur) {
                    load8<T, LAYOUT>(P, field, c.base, v);
                    cur = c.base;
                }
                float wt[8];
                weights32(c, wt);
                total.add(interpolate32(wt, v));
            }
        };
        // per-sample support tests only for waves with a ray whose end
        // samples leave the support; clamps only outside the samples that
        // are interior points for the whole wave
        const bool checked = __builtin_amdgcn_ballot_w64(!span_inside(P, o, d, iv.lower, step, 0, P.samples)) != 0;
        int ka, kb;
        interior_span(P, o, d, iv.lower, step, 0, P.samples, ka, kb);
        walk(std::false_type{}, 0, ka, checked);
        walk(std::true_type{}, ka, kb, false);
        walk(std::false_type{}, kb, P.samples, checked);
        if (bad) flag(P, view, DPT_STATUS_RANGE);
        result = total.value() * (len * step);
    }
    out[ray] = result;
    if (!isfinite(result)) flag(P, view, DPT_STATUS_RANGE);
}

// ----------------------------------------------------- pose reduction -----

// Sum C components over the 64 lanes of the wave (fixed shuffle tree); lane 0
// writes the wave tile's partials.
template <int C>
__device__ __forceinline__ void wave_store(const double *g, double *partial, bool valid) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const double s = wave_sum(g[c]);
        if (valid && (threadIdx.x & 63) == 0) partial[c] = s;
    }
}

// Store the epilogue's result: per ray for ray coordinates and per-ray
// tangents (6 values at partials + 6 * ray, non-finite flagged), else the
// wave tile's sum.
template <int C>
__device__ __forceinline__ void store_gradient(const Params &P, const double *g, double *partials, int wslot,
                                               bool wave_valid, int view, int row, int col) {
    if constexpr (C == kRayCoordinates || C == kRayTangent) {
        if (!ray_in_range(P, view, row, col)) return;
        const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
        bool bad = false;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            partials[6 * ray + c] = g[c];
            bad |= !isfinite(g[c]);
        }
        if (bad) flag(P, view, DPT_STATUS_RANGE);
    } else {
        wave_store<C>(g, partials + (size_t)wslot * C, wave_valid);
    }
}

// Brick = axis-aligned box of grid samples that one workgroup's rays touch in
// one slab, privatised in LDS.
struct Brick {
    int x0, y0, z0;      // first sample of the box
    int bx, by, bz;      // extents
    int lsx, lsy, lsz;   // local corner strides (0 on singleton grid axes)
    int volume;
    int origin;          // (z0 * by + y0) * bx + x0: local index = (z * by + y) * bx + x - origin
};

// First slabs per axis of the cell-Gauss volume adjoint, one per 55 voxels of
// the grid diagonal within [1, 64] (slabs then follow the brick's capacity).
inline int gauss_chunks(int nx, int ny, int nz) {
    const double diagonal = std::sqrt((double)nx * nx + (double)ny * ny + (double)nz * nz);
    return (int)std::lround(std::fmin(64.0, std::fmax(1.0, diagonal / 55.0)));
}

// Unit of the sample segments of small launches: 32 samples at 1024 over a
// 256^3 grid, scaled so that a chunk spans about the same distance in voxels --
// 32 * (S / 1024) * (443 / d), d = the grid diagonal in voxels -- within
// [8, 64].
inline int chunk_samples(int samples, int nx, int ny, int nz) {
    const double diagonal = std::sqrt((double)nx * nx + (double)ny * ny + (double)nz * nz);
    const double chunk = 32.0 * samples / 1024.0 * 443.4 / diagonal;
    return (int)std::lround(std::fmin(64.0, std::fmax(8.0, chunk)));
}

// Bound one slab's cells over the workgroup and, when the box fits the LDS
// brick of `cap` FP64 entries, describe it; e: the box's extents in grid samples.
// lo / nhi: this lane's lower cell corner minimum and negated maximum over its
// samples in the slab (INT_MAX when it has none).  Every lane gets the same
// answer (kept in SGPRs); one barrier.  gfx950 executes ds_add_f64 about ten
// times faster than ds_add_f32 (16.5 against 193 cycles per wave64 instruction at
// brick addresses, measured), so bricks accumulate in FP64.
__device__ __forceinline__ bool chunk_brick(const Params &P, int (*red)[6], int *lo, int *nhi, int cap, bool unit_x,
                                            Brick &B, int *e) {
    const int wv = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = wave_min(lo[a]);
        nhi[a] = wave_min(nhi[a]);
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            red[wv][a] = lo[a];
            red[wv][3 + a] = nhi[a];
        }
    }
    __syncthreads();
    int l[3], h[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        l[a] = min(min(red[0][a], red[1][a]), min(red[2][a], red[3][a]));
        h[a] = -min(min(red[0][3 + a], red[1][3 + a]), min(red[2][3 + a], red[3][3 + a]));
    }
    e[0] = e[1] = e[2] = 0;
    if (l[0] == INT_MAX) return false;
    const int n[3] = {P.nx, P.ny, P.nz};
#pragma unroll
    for (int a = 0; a < 3; ++a) e[a] = min(h[a] + 1, n[a] - 1) - l[a] + 1;
    if ((long long)e[0] * e[1] * e[2] > cap) return false;
    // every lane holds the same values: keep them in SGPRs
    B.x0 = __builtin_amdgcn_readfirstlane(l[0]);
    B.y0 = __builtin_amdgcn_readfirstlane(l[1]);
    B.z0 = __builtin_amdgcn_readfirstlane(l[2]);
    // odd row and plane strides when the padded box still fits (FP64 entries
    // whose indices differ by a multiple of 32 share an LDS bank, so even
    // strides line up the corners of neighbouring rays' cells); the padding
    // stays zero and the drain skips it
    int px = e[0], py = e[1];
    // Padded strides keep the walk's global-coordinate index of a corner below
    // 2^24 per operand and 2^31 overall when nz (ny + 1) and nz (ny + 1) (nx + 1) do.
    const long long plane = (long long)P.nz * (P.ny + 1);
    if ((long long)(px | 1) * (py | 1) * e[2] <= cap && plane <= (1 << 24) &&
        plane * (P.nx + 1) <= INT_MAX)
        px |= 1, py |= 1;
    B.bx = __builtin_amdgcn_readfirstlane(px);
    B.by = __builtin_amdgcn_readfirstlane(py);
    B.bz = __builtin_amdgcn_readfirstlane(e[2]);
    B.lsx = (unit_x || P.nx > 1) ? 1 : 0;
    B.lsy = P.ny > 1 ? B.bx : 0;
    B.lsz = P.nz > 1 ? B.bx * B.by : 0;
    B.volume = B.bx * B.by * B.bz;
    B.origin = (B.z0 * B.by + B.y0) * B.bx + B.x0;
    return true;
}

// The nine sums of a ray's pose adjoint, in sample order.
template <bool COMPENSATED>
struct PoseSums {
    Acc<COMPENSATED> mean, dor0, dor1, dor2, dd0, dd1, dd2, shl, shu;
    __device__ __forceinline__ void init() {
        mean.init();
        dor0.init();
        dor1.init();
        dor2.init();
        dd0.init();
        dd1.init();
        dd2.init();
        shl.init();
        shu.init();
    }
    __device__ __forceinline__ void fold() {
        mean.fold();
        dor0.fold();
        dor1.fold();
        dor2.fold();
        dd0.fold();
        dd1.fold();
        dd2.fold();
        shl.fold();
        shu.fold();
    }
    // sample k at position pos with value and slopes
    __device__ __forceinline__ void add(const Params &P, int k, float pos, float value, float g0, float g1, float g2,
                                        const float *d) {
        mean.add(value);
        dor0.add(g0);
        dor1.add(g1);
        dor2.add(g2);
        // contracted by the reference's code generator (fuse_fp)
        dd0.fma_add(pos, g0);
        dd1.fma_add(pos, g1);
        dd2.fma_add(pos, g2);
        const float along = fmaf(g2, d[2], fmaf(g1, d[1], g0 * d[0]));
        shl.fma_add(sample_beta(P, k), along);
        shu.fma_add(sample_alpha(P, k), along);
    }
};

// A ray's pose gradient from its sums (all zero for an inactive ray), stored
// or reduced over the wave.
template <int C, bool COMPENSATED>
__device__ __forceinline__ void pose_finish(const Params &P, const double *pose, bool active,
                                            const PoseSums<COMPENSATED> &q, const Interval32 &iv, float len, float seed,
                                            float span, float step, double *partials, int wslot, bool wave_valid,
                                            int view, int row, int col) {
    double gradient[kMaxComponents];
#pragma unroll
    for (int c = 0; c < kMaxComponents; ++c) gradient[c] = 0.0;
    if (active) {
        const float m = q.mean.value();
        const float lower_seed = fmaf(span, q.shl.value(), -m);
        const float upper_seed = fmaf(span, q.shu.value(), m);
        const float dor[3] = {q.dor0.value(), q.dor1.value(), q.dor2.value()};
        const float ddir[3] = {q.dd0.value(), q.dd1.value(), q.dd2.value()};
        double og[3], dg[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float lo_o = (iv.lo_axis == a) ? iv.lo_o : 0.0f;
            const float lo_d = (iv.lo_axis == a) ? iv.lo_d : 0.0f;
            const float up_o = (iv.up_axis == a) ? iv.up_o : 0.0f;
            const float up_d = (iv.up_axis == a) ? iv.up_d : 0.0f;
            og[a] = (double)fmaf(upper_seed, up_o, fmaf(lower_seed, lo_o, span * dor[a]));
            dg[a] = (double)fmaf(upper_seed, up_d, fmaf(lower_seed, lo_d, span * ddir[a]));
        }
        const float factor = (seed * len) / (float)P.samples;
        World w;  // recomputed: keeps 24 FP64 registers out of the sample loop
        ray_world(P, pose, view, row, col, w);
        pose_epilogue<C>(P, pose, w, (double)factor, og, dg, gradient, (double)seed, (double)(m * step));
    }
    store_gradient<C>(P, gradient, partials, wslot, wave_valid, view, row, col);
}

// ----------------------------------------------------- FP32 pose VJP ------
// kernels/projection_fp32.py:377-617, the pose half: each lane marches its ray
// once and sums the interpolated values, the slopes and the clip-face terms in
// sample order (the volume half is vol_walk_kernel).  Samples outside the
// support (only waves whose rays' end samples leave it test per sample) take
// the clamped cell with zero value and slopes: they add nothing, as the
// reference skips them.
template <typename T, int C, bool COMPENSATED, int LAYOUT>
__global__ __launch_bounds__(kBlock) void vjp32_kernel(Params P, const T *__restrict__ field,
                                                       const float *__restrict__ seeds,
                                                       double *__restrict__ partials) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    const double *pose = P.poses + 12 * (size_t)view;
    // ---- per-ray setup
    bool active = false, bad = false;
    float o[3] = {0, 0, 0}, d[3] = {0, 0, 0}, len = 0.0f, seed = 0.0f, span = 0.0f, step = 0.0f;
    Interval32 iv{};
    if (ray_in_range(P, view, row, col)) {
        const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
        World w;
        ray_world(P, pose, view, row, col, w);
        Ray r;
        ray_grid(P, w, r);
        o[0] = (float)r.o[0];
        o[1] = (float)r.o[1];
        o[2] = (float)r.o[2];
        d[0] = (float)r.d[0];
        d[1] = (float)r.d[1];
        d[2] = (float)r.d[2];
        len = (float)r.len;
        if (!r.valid || !finite3f(o[0], o[1], o[2]) || !finite3f(d[0], d[1], d[2]) || !isfinite(len) ||
            len <= 0.0f) {
            flag(P, view, DPT_STATUS_RANGE);
        } else {
            iv = interval32(P, o, d);
            span = iv.upper - iv.lower;
            seed = seeds[ray];
            if (!isfinite(seed)) flag(P, view, DPT_STATUS_RANGE);
            if (span > 0.0f && seed != 0.0f) {
                active = true;
                step = span / (float)P.samples;
                // sample points are monotone in the sample index: all are
                // finite iff the first and the last are
                bad = !finite_span(o, d, iv.lower, step, 0, P.samples);
            }
        }
    }

    PoseSums<COMPENSATED> q;
    q.init();
    if (active) {
        float v[8];
        int cur = -1;
        auto walk = [&](auto interior, int k0, int k1, bool checked) {
            constexpr bool INTERIOR = decltype(interior)::value;
            for (int k = k0; k < k1; ++k) {
                if constexpr (COMPENSATED) {
                    if (k > 0 && (k % kFoldBlock) == 0) q.fold();
                }
                const float pos = fmaf(sample_centre(P, k), step, iv.lower);
                const float p0 = fmaf(pos, d[0], o[0]);
                const float p1 = fmaf(pos, d[1], o[1]);
                const float p2 = fmaf(pos, d[2], o[2]);
                Cell32 c;
                float live = 1.0f;
                if constexpr (INTERIOR) {
                    cell32_interior(P, p0, p1, p2, c);
                } else {
                    cell32_inside(P, p0, p1, p2, c);
                    if (checked) {  // outside samples add nothing
                        const bool inside = inside32(P, p0, p1, p2);
                        c.fx = inside ? c.fx : 0.0f;
                        c.fy = inside ? c.fy : 0.0f;
                        c.fz = inside ? c.fz : 0.0f;
                        c.slx = inside ? c.slx : 0.0f;
                        c.sly = inside ? c.sly : 0.0f;
                        c.slz = inside ? c.slz : 0.0f;
                        live = inside ? 1.0f : 0.0f;
                    }
                }
                if (c.base != cur) {
                    load8<T, LAYOUT>(P, field, c.base, v);
                    cur = c.base;
                }
                float wt[8], g[3];
                weights32(c, wt);
                // an outside sample's slopes are zero (above); its value is zeroed here
                const float value = INTERIOR ? interpolate32(wt, v) : interpolate32(wt, v) * live;
                slopes32(c, v, g);
                q.add(P, k, pos, value, g[0], g[1], g[2], d);
            }
        };
        // per-sample support tests only for waves with a ray whose end
        // samples leave the support (uniform over the wave); clamps and
        // slope flags only outside the samples that are interior points
        // for the whole wave (full scan: 86.9 -> 75.9 ms)
        const bool checked = __builtin_amdgcn_ballot_w64(!span_inside(P, o, d, iv.lower, step, 0, P.samples)) != 0;
        int ka, kb;
        interior_span(P, o, d, iv.lower, step, 0, P.samples, ka, kb);
        walk(std::false_type{}, 0, ka, checked);
        walk(std::true_type{}, ka, kb, false);
        walk(std::false_type{}, kb, P.samples, checked);
    }
    pose_finish<C, COMPENSATED>(P, pose, active, q, iv, len, seed, span, step, partials, wslot, wave_valid, view, row,
                                col);
    if (bad) flag(P, view, DPT_STATUS_RANGE);
}

// ------------------------------------------------ FP32 small launches -----
// A launch of few rays (one 512^2 view is four waves per SIMD) leaves the
// march of a lane per ray exposed to the memory latency of every sample.
// Here a workgroup of eight waves holds 64 rays: seven waves sample, each
// kSplitRun consecutive samples a round with their loads in flight together,
// and leave values (and slopes) in LDS; the eighth adds the previous round's in
// sample order, so every sum is the sequential sum of the one-lane march, bit
// for bit.  Adding costs about 14 of the 85 instructions of a pose sample,
// hence the ratio.  MI355X, against a software pipeline of 8 samples in one
// lane: one 512^2 view of a 512 x 512 x 139 grid at S = 1024 (with rows of
// tiles dealt to the XCDs) forward 555 -> 268 us, pose VJP 1350 -> 346; 128^2
// over 128^3 at S = 256 69 -> 23 and 112 -> 30; 64^2 over 64^3 at S = 128
// forward 37 -> 12.
constexpr int kSplitWaves = 8, kSplitRun = 4, kSplitRound = (kSplitWaves - 1) * kSplitRun;

// Wave tile of this workgroup; P's walk is that of the wave tiles.
__device__ __forceinline__ bool split_tile(const Params &P, int &view, int &row, int &col, int &wslot) {
    wslot = tile_index(P);
    if (wslot >= P.total_tiles) return false;
    view = wslot / P.wt_per_view;
    const int r = wslot - view * P.wt_per_view, wy = r / P.wt_x, wx = r - wy * P.wt_x, lane = threadIdx.x & 63;
    row = P.bundle ? 0 : wy * 8 + (lane >> 3);
    col = P.bundle ? wx * 64 + lane : wx * 8 + (lane & 7);
    return true;
}

// One run of samples [k0, k0 + kSplitRun) of the lane's ray: emit(j, value,
// slopes).  An outside sample has zero slopes and the value `none`.
template <typename T, int LAYOUT, bool SLOPES, bool INTERIOR, typename F>
__device__ __forceinline__ void split_run(const Params &P, const T *field, const float *o, const float *d, float lower,
                                          float step, int k0, bool checked, float none, F emit) {
    float v[kSplitRun][8];
    Cell32 c[kSplitRun];
    bool in[kSplitRun], fresh[kSplitRun];
#pragma unroll
    for (int j = 0; j < kSplitRun; ++j) {
        const float pos = fmaf(sample_centre(P, min(k0 + j, P.samples - 1)), step, lower);
        const float p0 = fmaf(pos, d[0], o[0]);
        const float p1 = fmaf(pos, d[1], o[1]);
        const float p2 = fmaf(pos, d[2], o[2]);
        if constexpr (INTERIOR)
            cell32_interior(P, p0, p1, p2, c[j]);
        else
            cell32_inside(P, p0, p1, p2, c[j]);  // clamped: the load stays in the field
        in[j] = INTERIOR || !checked || inside32(P, p0, p1, p2);
        // only lanes whose cell changed load: requests to the L2 bound the march
        fresh[j] = j == 0 || c[j].base != c[j > 0 ? j - 1 : 0].base;
        if (fresh[j]) load8<T, LAYOUT>(P, field, c[j].base, v[j]);
    }
#pragma unroll
    for (int j = 0; j < kSplitRun; ++j) {
        if (j > 0) {
#pragma unroll
            for (int q = 0; q < 8; ++q) v[j][q] = fresh[j] ? v[j][q] : v[j > 0 ? j - 1 : 0][q];
        }
        float wt[8], g[3] = {0.0f, 0.0f, 0.0f};
        weights32(c[j], wt);
        const float value = interpolate32(wt, v[j]);
        if constexpr (SLOPES) {
            slopes32(c[j], v[j], g);
#pragma unroll
            for (int a = 0; a < 3; ++a) g[a] = in[j] ? g[a] : 0.0f;
        }
        emit(j, in[j] ? value : none, g);
    }
}

template <typename T, bool COMPENSATED, int LAYOUT>
__global__ __launch_bounds__(64 * kSplitWaves) void forward32_split_kernel(Params P, const T *__restrict__ field,
                                                                           float *__restrict__ out) {
    __shared__ float buffer[2][kSplitRound][64];
    int view, row, col, wslot;
    if (!split_tile(P, view, row, col, wslot)) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool adds = w == kSplitWaves - 1;
    const bool exists = ray_in_range(P, view, row, col);
    bool hit = false;
    float o[3] = {0, 0, 0}, d[3] = {0, 0, 0}, len = 0.0f, lower = 0.0f, step = 0.0f;
    if (exists) {
        World ww;
        ray_world(P, P.poses + 12 * (size_t)view, view, row, col, ww);
        Ray r;
        ray_grid(P, ww, r);
        const float ro[3] = {(float)r.o[0], (float)r.o[1], (float)r.o[2]};
        const float rd[3] = {(float)r.d[0], (float)r.d[1], (float)r.d[2]};
        len = (float)r.len;
        if (!r.valid || !finite3f(ro[0], ro[1], ro[2]) || !finite3f(rd[0], rd[1], rd[2]) || !isfinite(len) ||
            len <= 0.0f) {
            if (adds) flag(P, view, DPT_STATUS_RANGE);
        } else {
            const Interval32 iv = interval32(P, ro, rd);
            if (iv.upper > iv.lower) {
                lower = iv.lower;
                step = (iv.upper - iv.lower) / (float)P.samples;
                // a ray with non-finite sample points keeps the benign ray
                // (its image is flagged)
                hit = finite_span(ro, rd, lower, step, 0, P.samples);
                if (!hit && adds) flag(P, view, DPT_STATUS_RANGE);
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    o[a] = hit ? ro[a] : 0.0f;
                    d[a] = hit ? rd[a] : 0.0f;
                }
                if (!hit) lower = step = 0.0f;
            }
        }
    }
    float result = 0.0f;
    if (__builtin_amdgcn_ballot_w64(hit) != 0) {  // the same in every wave
        const bool checked = __builtin_amdgcn_ballot_w64(hit && !span_inside(P, o, d, lower, step, 0, P.samples)) != 0;
        int ka = P.samples, kb = P.samples;
        if (hit) interior_span(P, o, d, lower, step, 0, P.samples, ka, kb);
        // lanes without a hit sample the origin, an interior point on grids with cells on every axis
        const bool origin = interior32(P, 0.0f, 0.0f, 0.0f);
        const int first_hit = __ffsll((unsigned long long)__builtin_amdgcn_ballot_w64(hit)) - 1;
        ka = __builtin_amdgcn_readlane(ka, first_hit);
        kb = origin ? __builtin_amdgcn_readlane(kb, first_hit) : ka;
        Acc<COMPENSATED> total;
        total.init();
        const int rounds = (P.samples + kSplitRound - 1) / kSplitRound;
        for (int r = 0; r <= rounds; ++r) {
            if (!adds) {
                const int k0 = r * kSplitRound + w * kSplitRun;
                if (k0 < P.samples) {
                    float(*slot)[64] = &buffer[r & 1][w * kSplitRun];
                    auto emit = [&](int j, float value, const float *) { slot[j][lane] = value; };
                    // -0 is the identity of FP32 addition (the reference skips outside samples)
                    if (k0 >= ka && k0 + kSplitRun <= kb)
                        split_run<T, LAYOUT, false, true>(P, field, o, d, lower, step, k0, false, -0.0f, emit);
                    else
                        split_run<T, LAYOUT, false, false>(P, field, o, d, lower, step, k0, checked, -0.0f, emit);
                }
            } else if (r > 0) {
                const int base = (r - 1) * kSplitRound, count = min(kSplitRound, P.samples - base);
                const float(*slot)[64] = buffer[(r - 1) & 1];
                auto add = [&](int k, float value) {
                    if constexpr (COMPENSATED) {
                        if (k > 0 && (k % kFoldBlock) == 0) total.fold();
                    }
                    total.add(value);
                };
                if (count == kSplitRound) {  // every read in flight before the first addition
                    float e[kSplitRound];
#pragma unroll
                    for (int s = 0; s < kSplitRound; ++s) e[s] = slot[s][lane];
#pragma unroll
                    for (int s = 0; s < kSplitRound; ++s) add(base + s, e[s]);
                } else {
                    for (int s = 0; s < count; ++s) add(base + s, slot[s][lane]);
                }
            }
            __syncthreads();
        }
        if (hit) result = total.value() * (len * step);
    }
    if (adds && exists) {
        const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
        out[ray] = result;
        if (!isfinite(result)) flag(P, view, DPT_STATUS_RANGE);
    }
}

template <typename T, int C, bool COMPENSATED, int LAYOUT>
__global__ __launch_bounds__(64 * kSplitWaves) void vjp32_split_kernel(Params P, const T *__restrict__ field,
                                                                       const float *__restrict__ seeds,
                                                                       double *__restrict__ partials) {
    __shared__ float4 buffer[2][kSplitRound][64];
    int view, row, col, wslot;
    if (!split_tile(P, view, row, col, wslot)) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool adds = w == kSplitWaves - 1;
    const double *pose = P.poses + 12 * (size_t)view;
    bool active = false;
    float o[3] = {0, 0, 0}, d[3] = {0, 0, 0}, len = 0.0f, seed = 0.0f, span = 0.0f, lower = 0.0f, step = 0.0f;
    Interval32 iv{};
    if (ray_in_range(P, view, row, col)) {
        World ww;
        ray_world(P, pose, view, row, col, ww);
        Ray r;
        ray_grid(P, ww, r);
        const float ro[3] = {(float)r.o[0], (float)r.o[1], (float)r.o[2]};
        const float rd[3] = {(float)r.d[0], (float)r.d[1], (float)r.d[2]};
        len = (float)r.len;
        if (!r.valid || !finite3f(ro[0], ro[1], ro[2]) || !finite3f(rd[0], rd[1], rd[2]) || !isfinite(len) ||
            len <= 0.0f) {
            if (adds) flag(P, view, DPT_STATUS_RANGE);
        } else {
            iv = interval32(P, ro, rd);
            span = iv.upper - iv.lower;
            seed = seeds[((size_t)view * P.rows + row) * P.cols + col];
            if (!isfinite(seed) && adds) flag(P, view, DPT_STATUS_RANGE);
            if (span > 0.0f && seed != 0.0f) {
                lower = iv.lower;
                step = span / (float)P.samples;
                // a ray with non-finite sample points is flagged and adds nothing
                active = finite_span(ro, rd, lower, step, 0, P.samples);
                if (!active && adds) flag(P, view, DPT_STATUS_RANGE);
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    o[a] = active ? ro[a] : 0.0f;
                    d[a] = active ? rd[a] : 0.0f;
                }
                if (!active) lower = step = 0.0f;
            }
        }
    }
    PoseSums<COMPENSATED> q;
    q.init();
    if (__builtin_amdgcn_ballot_w64(active) != 0) {  // the same in every wave
        const bool checked = __builtin_amdgcn_ballot_w64(active && !span_inside(P, o, d, lower, step, 0, P.samples)) != 0;
        int ka = P.samples, kb = P.samples;
        if (active) interior_span(P, o, d, lower, step, 0, P.samples, ka, kb);
        const bool origin = interior32(P, 0.0f, 0.0f, 0.0f);  // as forward32_split_kernel
        const int first_hit = __ffsll((unsigned long long)__builtin_amdgcn_ballot_w64(active)) - 1;
        ka = __builtin_amdgcn_readlane(ka, first_hit);
        kb = origin ? __builtin_amdgcn_readlane(kb, first_hit) : ka;
        const int rounds = (P.samples + kSplitRound - 1) / kSplitRound;
        for (int r = 0; r <= rounds; ++r) {
            if (!adds) {
                const int k0 = r * kSplitRound + w * kSplitRun;
                if (k0 < P.samples) {
                    float4(*slot)[64] = &buffer[r & 1][w * kSplitRun];
                    auto emit = [&](int j, float value, const float *g) {
                        slot[j][lane] = make_float4(value, g[0], g[1], g[2]);
                    };
                    if (k0 >= ka && k0 + kSplitRun <= kb)
                        split_run<T, LAYOUT, true, true>(P, field, o, d, lower, step, k0, false, 0.0f, emit);
                    else
                        split_run<T, LAYOUT, true, false>(P, field, o, d, lower, step, k0, checked, 0.0f, emit);
                }
            } else if (r > 0) {
                const int base = (r - 1) * kSplitRound, count = min(kSplitRound, P.samples - base);
                const float4(*slot)[64] = buffer[(r - 1) & 1];
                auto add = [&](int k, const float4 &e) {
                    if constexpr (COMPENSATED) {
                        if (k > 0 && (k % kFoldBlock) == 0) q.fold();
                    }
                    q.add(P, k, fmaf(sample_centre(P, k), step, lower), e.x, e.y, e.z, e.w, d);
                };
                if (count == kSplitRound) {  // reads in flight, a wave's share at a time
                    constexpr int kPart = kSplitRound / 2;
#pragma unroll
                    for (int part = 0; part < 2; ++part) {
                        float4 e[kPart];
#pragma unroll
                        for (int s = 0; s < kPart; ++s) e[s] = slot[part * kPart + s][lane];
#pragma unroll
                        for (int s = 0; s < kPart; ++s) add(base + part * kPart + s, e[s]);
                    }
                } else {
                    for (int s = 0; s < count; ++s) add(base + s, slot[s][lane]);
                }
            }
            __syncthreads();
        }
    }
    if (adds)
        pose_finish<C, COMPENSATED>(P, pose, active, q, iv, len, seed, span, step, partials, wslot, true, view, row,
                                    col);
}

// --------------------------------------------------------- FP64 sampling --

struct Cell64 {
    int base;
    int lx, ly, lz;
    double fx, fy, fz;
    double slx, sly, slz;
};

// kernels/projection.py:124-134 + 199-214
__device__ __forceinline__ bool cell64(const Params &P, const double *p, Cell64 &c) {
    const double hx = (double)P.nx - 0.5, hy = (double)P.ny - 0.5, hz = (double)P.nz - 0.5;
    if (!(p[0] >= -0.5 && p[1] >= -0.5 && p[2] >= -0.5 && p[0] <= hx && p[1] <= hy && p[2] <= hz))
        return false;
    const double mx = (double)(P.nx - 1), my = (double)(P.ny - 1), mz = (double)(P.nz - 1);
    const double v0 = fmin(fmax(p[0], 0.0), mx);
    const double v1 = fmin(fmax(p[1], 0.0), my);
    const double v2 = fmin(fmax(p[2], 0.0), mz);
    const int lx = min((int)floor(v0), P.capx);
    const int ly = min((int)floor(v1), P.capy);
    const int lz = min((int)floor(v2), P.capz);
    c.lx = lx;
    c.ly = ly;
    c.lz = lz;
    c.fx = v0 - (double)lx;
    c.fy = v1 - (double)ly;
    c.fz = v2 - (double)lz;
    c.slx = (p[0] >= 0.0 && p[0] < mx) ? 1.0 : 0.0;
    c.sly = (p[1] >= 0.0 && p[1] < my) ? 1.0 : 0.0;
    c.slz = (p[2] >= 0.0 && p[2] < mz) ? 1.0 : 0.0;
    c.base = (lz * P.ny + ly) * P.nx + lx;
    return true;
}

// Clamped lower cell of an FP64 sample point (cell64's arithmetic without the
// support test: out-of-support samples only widen a chunk's box).
__device__ __forceinline__ void lower_cell64(const Params &P, const double *p, int *l) {
    l[0] = min((int)floor(fmin(fmax(p[0], 0.0), (double)(P.nx - 1))), P.capx);
    l[1] = min((int)floor(fmin(fmax(p[1], 0.0), (double)(P.ny - 1))), P.capy);
    l[2] = min((int)floor(fmin(fmax(p[2], 0.0), (double)(P.nz - 1))), P.capz);
}

// kernels/projection.py:236-274 (weighted lerps; differences before interpolation)
typedef const double __attribute__((address_space(4))) *constant_f64;

template <bool GRAD, bool INTERIOR = false>
__device__ __forceinline__ double sample_cell64(const Cell64 &c, const double *v, double *g) {
    const double v000 = v[0], v100 = v[1], v010 = v[2], v110 = v[3];
    const double v001 = v[4], v101 = v[5], v011 = v[6], v111 = v[7];
    const double fx = c.fx, fy = c.fy, fz = c.fz;
    const double ax = 1.0 - fx, ay = 1.0 - fy, az = 1.0 - fz;
    const double x00 = ax * v000 + fx * v100, x10 = ax * v010 + fx * v110;
    const double x01 = ax * v001 + fx * v101, x11 = ax * v011 + fx * v111;
    const double xy0 = ay * x00 + fy * x10, xy1 = ay * x01 + fy * x11;
    const double value = az * xy0 + fz * xy1;
    if constexpr (GRAD) {
        const double dx00 = v100 - v000, dx10 = v110 - v010, dx01 = v101 - v001, dx11 = v111 - v011;
        const double dx0 = ay * dx00 + fy * dx10, dx1 = ay * dx01 + fy * dx11;
        const double dy0 = ax * (v010 - v000) + fx * (v110 - v100);
        const double dy1 = ax * (v011 - v001) + fx * (v111 - v101);
        const double dz0 = ax * (v001 - v000) + fx * (v101 - v100);
        const double dz1 = ax * (v011 - v010) + fx * (v111 - v110);
        g[0] = az * dx0 + fz * dx1;
        g[1] = az * dy0 + fz * dy1;
        g[2] = ay * dz0 + fy * dz1;
        if constexpr (!INTERIOR) {
            g[0] = c.slx * g[0];
            g[1] = c.sly * g[1];
            g[2] = c.slz * g[2];
        }
    }
    return value;
}

// A point in [0, n - 1) on every axis: cell64's cell and fractions without its
// clamps, caps and support test (fract(p) = p - floor(p) is exact for p >= 0).
__device__ __forceinline__ void cell64_interior(const Params &P, const double *p, Cell64 &c) {
    c.lx = (int)p[0];
    c.ly = (int)p[1];
    c.lz = (int)p[2];
    c.fx = __builtin_amdgcn_fract(p[0]);
    c.fy = __builtin_amdgcn_fract(p[1]);
    c.fz = __builtin_amdgcn_fract(p[2]);
    c.slx = c.sly = c.slz = 1.0;
    c.base = (c.lz * P.ny + c.ly) * P.nx + c.lx;
}

// Sample k's position and point, in the reference's unfused arithmetic.
__device__ __forceinline__ double point64(const Ray &r, double lower, double step, int k, double *p) {
    const double pos = lower + ((double)k + 0.5) * step;
#pragma unroll
    for (int a = 0; a < 3; ++a) p[a] = r.o[a] + pos * r.d[a];
    return pos;
}

// interior_span (device_common.h) for FP64 sampling of all samples.  With the
// interior samples free of clamps, support tests and the division of the
// sample fraction (tabulated), 24 views of 256^2 over 128^3 at S = 512 run
// the forward in 1.02 ms (1.35 before) and the pose VJP in 2.21 (2.57); FP64
// instruction issue bounds both.  (Gathering from a quad copy, as FP32 does,
// changed neither.)
__device__ __forceinline__ void interior_span64(const Params &P, const Ray &r, double lower, double step, int &ka,
                                                int &kb) {
    const double top[3] = {(double)(P.nx - 1), (double)(P.ny - 1), (double)(P.nz - 1)};
    float enter = (float)lower, leave = 3e38f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float inverse = __builtin_amdgcn_rcpf((float)r.d[a]);
        const float u = (float)(0.0 - r.o[a]) * inverse, v = (float)(top[a] - r.o[a]) * inverse;
        enter = fmaxf(enter, fminf(u, v));
        leave = fminf(leave, fmaxf(u, v));
    }
    const float per = __builtin_amdgcn_rcpf((float)step), count = (float)P.samples;
    const int lo = (int)fminf(fmaxf(ceilf((enter - (float)lower) * per) + 2.0f, 0.0f), count);
    const int hi = (int)fminf(fmaxf(floorf((leave - (float)lower) * per) - 2.0f, 0.0f), count);
    uniform_span(lo, hi, 0, P.samples, ka, kb);
    if (kb > ka) {
        bool ok = true;
        for (int k : {ka, kb - 1}) {
            double p[3];
            point64(r, lower, step, k, p);
#pragma unroll
            for (int a = 0; a < 3; ++a) ok = ok && p[a] >= 0.0 && p[a] < top[a];
        }
        if (__builtin_amdgcn_ballot_w64(!ok) != 0) kb = ka;
    }
    if (kb <= ka) ka = kb = P.samples;
}

// The eight corners as FP64, fetched with the x-pair loads of the FP32 path
// on grids with nx > 1 (uniform branch).
template <typename T>
__device__ __forceinline__ void load8d(const Params &P, const T *field, int base, double *v) {
    float f[8];
    if (P.sx)
        load8<T, kLayoutPair>(P, field, base, f);
    else
        load8<T, kLayoutScalar>(P, field, base, f);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (double)f[k];
}

// kernels/projection.py:802-846 (midpoint, FP64 sampling)
template <typename T>
__global__ __launch_bounds__(kBlock) void forward64_kernel(Params P, const T *__restrict__ field,
                                                           double *__restrict__ out) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    if (!ray_in_range(P, view, row, col)) return;
    const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
    const double *pose = P.poses + 12 * (size_t)view;
    World w;
    ray_world(P, pose, view, row, col, w);
    Ray r;
    ray_grid(P, w, r);
    if (!r.valid) {
        flag(P, view, DPT_STATUS_RANGE);
        out[ray] = 0.0;
        return;
    }
    const Interval64 iv = interval64(P, r.o, r.d);
    double integral = 0.0;
    if (iv.upper > iv.lower) {
        const double step = (iv.upper - iv.lower) / (double)P.samples;
        // sample points are monotone in the sample index: all are finite iff
        // the first and the last are
        double ends[6];
        point64(r, iv.lower, step, 0, ends);
        point64(r, iv.lower, step, P.samples - 1, ends + 3);
        if (!finite3d(ends) || !finite3d(ends + 3)) flag(P, view, DPT_STATUS_RANGE);
        double v[8];
        int cur = -1;  // corners cached while consecutive samples share a cell
        auto walk = [&](auto interior, int k0, int k1) {
            for (int k = k0; k < k1; ++k) {
                double p[3];
                point64(r, iv.lower, step, k, p);
                Cell64 c;
                if constexpr (decltype(interior)::value) {
                    cell64_interior(P, p, c);
                } else {
                    if (!cell64(P, p, c)) continue;
                }
                if (c.base != cur) {
                    load8d<T>(P, field, c.base, v);
                    cur = c.base;
                }
                integral += sample_cell64<false>(c, v, nullptr);
            }
        };
        int ka, kb;
        interior_span64(P, r, iv.lower, step, ka, kb);
        walk(std::false_type{}, 0, ka);
        walk(std::true_type{}, ka, kb);
        walk(std::false_type{}, kb, P.samples);
        integral *= r.len * step;
    }
    out[ray] = integral;
    if (!isfinite(integral)) flag(P, view, DPT_STATUS_RANGE);
}

// kernels/projection.py:873-1237 (midpoint, FP64 sampling), the pose half
template <typename T, int C>
__global__ __launch_bounds__(kBlock) void vjp64_kernel(Params P, const T *__restrict__ field,
                                                       const double *__restrict__ seeds,
                                                       double *__restrict__ partials) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    double gradient[kMaxComponents];
#pragma unroll
    for (int c = 0; c < kMaxComponents; ++c) gradient[c] = 0.0;
    const double *pose = P.poses + 12 * (size_t)view;

    // ---- per-ray setup
    bool active = false;
    Ray r{};
    Interval64 iv{};
    double span = 0.0, seed = 0.0, factor = 0.0, step = 0.0;
    const double S = (double)P.samples;
    if (ray_in_range(P, view, row, col)) {
        const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
        World w;
        ray_world(P, pose, view, row, col, w);
        ray_grid(P, w, r);
        if (!r.valid) {
            flag(P, view, DPT_STATUS_RANGE);
        } else {
            iv = interval64(P, r.o, r.d);
            span = iv.upper - iv.lower;
            seed = seeds[ray];
            if (seed == 0.0) span = 0.0;
            if (span > 0.0) {
                active = true;
                factor = seed * r.len;
                step = span / S;
            }
        }
    }
    double mean = 0.0, dor[3] = {0, 0, 0}, ddir[3] = {0, 0, 0};
    double shift_lower = 0.0, shift_upper = 0.0;
    if (active) {
        double ends[6];  // as forward64_kernel
        point64(r, iv.lower, step, 0, ends);
        point64(r, iv.lower, step, P.samples - 1, ends + 3);
        if (!finite3d(ends) || !finite3d(ends + 3)) flag(P, view, DPT_STATUS_RANGE);
        double v[8];
        int cur = -1;  // corners cached while consecutive samples share a cell
        auto walk = [&](auto interior, int k0, int k1) {
            constexpr bool INTERIOR = decltype(interior)::value;
            for (int k = k0; k < k1; ++k) {
                double p[3], g[3];
                const double pos = point64(r, iv.lower, step, k, p);
                Cell64 c;
                if constexpr (INTERIOR) {
                    cell64_interior(P, p, c);
                } else {
                    if (!cell64(P, p, c)) continue;
                }
                if (c.base != cur) {
                    load8d<T>(P, field, c.base, v);
                    cur = c.base;
                }
                mean += sample_cell64<true, INTERIOR>(c, v, g);
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    dor[a] += g[a];
                    ddir[a] += pos * g[a];
                }
                const double along = g[0] * r.d[0] + g[1] * r.d[1] + g[2] * r.d[2];
                // uniform: scalar loads
                shift_lower += ((constant_f64)P.alpha64)[P.samples + k] * along;
                shift_upper += ((constant_f64)P.alpha64)[k] * along;
            }
        };
        int ka, kb;
        interior_span64(P, r, iv.lower, step, ka, kb);
        walk(std::false_type{}, 0, ka);
        walk(std::true_type{}, ka, kb);
        walk(std::false_type{}, kb, P.samples);
    }
    if (active) {
        const double lower_seed = -mean + span * shift_lower;
        const double upper_seed = mean + span * shift_upper;
        double og[3], dg[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double lo_o = (iv.lo_axis == a) ? iv.lo_o : 0.0;
            const double lo_d = (iv.lo_axis == a) ? iv.lo_d : 0.0;
            const double up_o = (iv.up_axis == a) ? iv.up_o : 0.0;
            const double up_d = (iv.up_axis == a) ? iv.up_d : 0.0;
            og[a] = span * dor[a] + lower_seed * lo_o + upper_seed * up_o;
            dg[a] = span * ddir[a] + lower_seed * lo_d + upper_seed * up_d;
        }
        World w;  // recomputed: keeps its FP64 registers out of the sample loop
        ray_world(P, pose, view, row, col, w);
        const double f = factor / S;
        if (isfinite(f)) {
            pose_epilogue<C>(P, pose, w, f, og, dg, gradient, seed, mean * step, true);
        } else {
            // kernels/projection.py:1163-1183 range-safe products
            double sa[3], da[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double s = P.g[i] * og[0] + P.g[3 + i] * og[1] + P.g[6 + i] * og[2];
                const double t = P.g[i] * dg[0] + P.g[3 + i] * dg[1] + P.g[6 + i] * dg[2];
                sa[i] = product4(seed, r.len, 1.0 / S, s);
                da[i] = product4(seed, r.len, 1.0 / S, t);
            }
            Params unit = P;
            for (int i = 0; i < 9; ++i) unit.g[i] = (i % 4 == 0) ? 1.0 : 0.0;
            pose_epilogue<C>(unit, pose, w, 1.0, sa, da, gradient, seed, mean * step, true);
        }
    }
    store_gradient<C>(P, gradient, partials, wslot, wave_valid, view, row, col);
}

// ------------------------------------------------ exact cell-Gauss (FP64) --
// kernels/projection.py:522-746: the clipped ray is cut at every
// interpolation plane it crosses and each piece gets two Gauss nodes, exact
// for the cubic a trilinear field is along a line inside one cell.  Same
// operation order as the oracle, so images agree bit for bit.

struct CellWalk {
    int plane[3], step[3];
    double next[3], inv[3];
};

struct CellPiece {
    double end, radius, first_position, second_position;
    double first[3], second[3];
    int lower[3];
    bool shared;
};

// kernels/projection.py:629-640: cached reciprocal with one FMA residual
// correction; range extremes keep the division
__device__ __forceinline__ double crossing_quotient(double delta, double direction, double inverse) {
    if (inverse == 0.0) return delta / direction;
    const double q = delta * inverse;
    if (!isfinite(q) || fabs(q) < 2.2250738585072014e-308) return delta / direction;
    return fma(fma(-q, direction, delta), inverse, q);
}

// kernels/projection.py:643-655
__device__ __forceinline__ double cell_crossing(const Ray &r, int a, int plane, int n, double upper, double inv) {
    if (r.d[a] == 0.0 || plane < 0 || plane >= n) return upper;
    const double c = crossing_quotient((double)plane - r.o[a], r.d[a], inv);
    return c < upper ? c : upper;
}

// kernels/projection.py:659-695 (begin_cells)
__device__ __forceinline__ void begin_cells(const Params &P, const Ray &r, const Interval64 &iv, CellWalk &w) {
    const int n[3] = {P.nx, P.ny, P.nz};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double entry = r.o[a] + iv.lower * r.d[a];
        const double v = r.d[a];
        w.inv[a] = 0.0;
        w.step[a] = 0;
        w.plane[a] = 0;
        if (v != 0.0) {
            const double inverse = 1.0 / v;
            if (isfinite(inverse) && fabs(inverse) >= 2.2250738585072014e-308 && fabs(v) >= 2.2250738585072014e-308)
                w.inv[a] = inverse;
        }
        if (v > 0.0) {
            w.step[a] = 1;
            w.plane[a] = max((int)ceil(entry), 0);
        } else if (v < 0.0) {
            w.step[a] = -1;
            w.plane[a] = min((int)floor(entry), n[a] - 1);
        }
        double crossing = cell_crossing(r, a, w.plane[a], n[a], iv.upper, w.inv[a]);
        if (crossing <= iv.lower) {
            w.plane[a] += w.step[a];
            crossing = cell_crossing(r, a, w.plane[a], n[a], iv.upper, w.inv[a]);
        }
        w.next[a] = crossing;
    }
}

// kernels/projection.py:710-742 (cell_segment)
__device__ __forceinline__ void cell_piece(const Params &P, const Ray &r, const CellWalk &w, double start,
                                           CellPiece &s) {
    const double m = w.next[1] < w.next[2] ? w.next[1] : w.next[2];
    s.end = w.next[0] < m ? w.next[0] : m;
    s.radius = (s.end - start) * 0.5;
    const double centre = start + s.radius;
    const double offset = s.radius / sqrt(3.0);
    s.first_position = centre - offset;
    s.second_position = centre + offset;
    double mid[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s.first[a] = r.o[a] + s.first_position * r.d[a];
        s.second[a] = r.o[a] + s.second_position * r.d[a];
        mid[a] = r.o[a] + centre * r.d[a];
    }
    lower_cell64(P, mid, s.lower);
    const int n[3] = {P.nx, P.ny, P.nz};
    s.shared = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double lo = (double)s.lower[a], up = lo + 1.0, top = (double)(n[a] - 1);
        const double c1 = fmin(fmax(s.first[a], 0.0), top), c2 = fmin(fmax(s.second[a], 0.0), top);
        if (c1 < lo || c2 < lo) s.shared = false;
        if (s.lower[a] < n[a] - 2 && (c1 >= up || c2 >= up)) s.shared = false;
    }
}

// kernels/projection.py:745-755 (advance_cells): every tied plane advances
__device__ __forceinline__ void advance_cells(const Params &P, const Ray &r, CellWalk &w, double end, double upper) {
    const int n[3] = {P.nx, P.ny, P.nz};
#pragma unroll
    for (int a = 0; a < 3; ++a)
        if (w.next[a] <= end) {
            w.plane[a] += w.step[a];
            w.next[a] = cell_crossing(r, a, w.plane[a], n[a], upper, w.inv[a]);
        }
}

__device__ __forceinline__ bool inside_support64(const Params &P, const double *p) {
    return p[0] >= -0.5 && p[1] >= -0.5 && p[2] >= -0.5 && p[0] <= (double)P.nx - 0.5 &&
           p[1] <= (double)P.ny - 0.5 && p[2] <= (double)P.nz - 0.5;
}

// Value (and slope) of one node: sample_cell in the piece's cell when it is
// shared (kernels/projection.py:278-284), else sample_field (:288-295); zero
// outside the support.
template <typename T, bool GRAD>
__device__ __forceinline__ double node_value(const Params &P, const T *field, const double *pt, const int *lower,
                                             double *g) {
    if (GRAD) g[0] = g[1] = g[2] = 0.0;
    Cell64 c;
    if (!cell64(P, pt, c)) return 0.0;
    if (lower != nullptr) {
        c.lx = lower[0];
        c.ly = lower[1];
        c.lz = lower[2];
        c.fx = fmin(fmax(pt[0], 0.0), (double)(P.nx - 1)) - (double)c.lx;
        c.fy = fmin(fmax(pt[1], 0.0), (double)(P.ny - 1)) - (double)c.ly;
        c.fz = fmin(fmax(pt[2], 0.0), (double)(P.nz - 1)) - (double)c.lz;
        c.base = (c.lz * P.ny + c.ly) * P.nx + c.lx;
    }
    double v[8];
    load8d<T>(P, field, c.base, v);
    return sample_cell64<GRAD>(c, v, g);
}

// Value (and slope) of a node in a shared piece whose 8 corner values v of
// the cell at lower are already loaded (sample_cell, kernels/projection.py:
// 278-284); zero outside the support.
template <bool GRAD>
__device__ __forceinline__ double node_in_cell(const Params &P, const double *pt, const int *lower, const double *v,
                                               double *g) {
    if (GRAD) g[0] = g[1] = g[2] = 0.0;
    Cell64 c;
    if (!cell64(P, pt, c)) return 0.0;
    c.lx = lower[0];
    c.ly = lower[1];
    c.lz = lower[2];
    c.fx = fmin(fmax(pt[0], 0.0), (double)(P.nx - 1)) - (double)c.lx;
    c.fy = fmin(fmax(pt[1], 0.0), (double)(P.ny - 1)) - (double)c.ly;
    c.fz = fmin(fmax(pt[2], 0.0), (double)(P.nz - 1)) - (double)c.lz;
    return sample_cell64<GRAD>(c, v, g);
}

// Grid index of corner k of the cell at lower (kernels/projection.py:217-222)
__device__ __forceinline__ int corner_of(const Params &P, const int *lower, int k) {
    const int x = min(lower[0] + (k & 1), P.nx - 1);
    const int y = min(lower[1] + ((k >> 1) & 1), P.ny - 1);
    const int z = min(lower[2] + ((k >> 2) & 1), P.nz - 1);
    return (z * P.ny + y) * P.nx + x;
}

// kernels/projection.py:802-846 with cell_gauss: integral * length
template <typename T>
__global__ __launch_bounds__(kBlock) void forward_gauss_kernel(Params P, const T *__restrict__ field,
                                                               double *__restrict__ out) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    if (!ray_in_range(P, view, row, col)) return;
    const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
    const double *pose = P.poses + 12 * (size_t)view;
    World w;
    ray_world(P, pose, view, row, col, w);
    Ray r;
    ray_grid(P, w, r);
    if (!r.valid) {
        flag(P, view, DPT_STATUS_RANGE);
        out[ray] = 0.0;
        return;
    }
    const Interval64 iv = interval64(P, r.o, r.d);
    double integral = 0.0;
    if (iv.upper > iv.lower) {
        CellWalk walk;
        begin_cells(P, r, iv, walk);
        double start = iv.lower;
        const long long limit = (long long)P.nx + P.ny + P.nz + 1;
        bool bad = false;
        for (long long segments = 0; start < iv.upper && segments < limit; ++segments) {
            CellPiece s;
            cell_piece(P, r, walk, start, s);
            if (s.end <= start) {
                bad = true;
                break;
            }
            bad |= !finite3d(s.first) || !finite3d(s.second);
            if (s.shared) {  // one load of the cell for both nodes
                double v[8];
                load8d<T>(P, field, (s.lower[2] * P.ny + s.lower[1]) * P.nx + s.lower[0], v);
                integral += s.radius * node_in_cell<false>(P, s.first, s.lower, v, nullptr);
                integral += s.radius * node_in_cell<false>(P, s.second, s.lower, v, nullptr);
            } else {
                integral += s.radius * node_value<T, false>(P, field, s.first, nullptr, nullptr);
                integral += s.radius * node_value<T, false>(P, field, s.second, nullptr, nullptr);
            }
            start = s.end;
            advance_cells(P, r, walk, s.end, iv.upper);
        }
        bad |= start < iv.upper;
        if (bad) flag(P, view, DPT_STATUS_RANGE);
        integral *= r.len;
    }
    out[ray] = integral;
    if (!isfinite(integral)) flag(P, view, DPT_STATUS_RANGE);
}

// Increment of one corner into the FP64 accumulator, rounded as the
// destination requires (zeros add nothing and are skipped)
__device__ __forceinline__ bool add_increment(const Params &P, double *acc, int index, double contribution) {
    const double rounded = destination_increment(P, contribution);
    if (rounded != 0.0) unsafeAtomicAdd(acc + index, rounded);
    return isfinite(rounded);
}

// Factors whose FP64 increments neither vanish nor overflow in the destination.
__device__ __forceinline__ bool walk_factor64(const Params &P, double m) {
    return m >= (P.volume_f64 ? 0x1p-900 : 0x1p-102) && m <= (P.volume_f64 ? 0x1p900 : 0x1p96);
}

// Whether vol_walk_kernel takes a ray of the cell-Gauss rule: a factor in range
// and a clip interval that stays inside the support.
__device__ __forceinline__ bool gauss_summed(const Params &P, const Ray &r, const Interval64 &iv, double factor) {
    const double span = iv.upper - iv.lower;
    const double pa = iv.lower + 1e-6 * span, pb = iv.upper - 1e-6 * span;
    const double qa[3] = {r.o[0] + pa * r.d[0], r.o[1] + pa * r.d[1], r.o[2] + pa * r.d[2]};
    const double qb[3] = {r.o[0] + pb * r.d[0], r.o[1] + pb * r.d[1], r.o[2] + pb * r.d[2]};
    return walk_factor64(P, fabs(factor * span)) && inside_support64(P, qa) && inside_support64(P, qb);
}

// The rays it does not take: the reference's products piece by piece, by device
// atomics.
__global__ __launch_bounds__(kBlock) void gauss_scatter_kernel(Params P, const double *__restrict__ seeds,
                                                               double *__restrict__ acc) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    if (!ray_in_range(P, view, row, col)) return;
    World w;
    ray_world(P, P.poses + 12 * (size_t)view, view, row, col, w);
    Ray r;
    ray_grid(P, w, r);
    if (!r.valid) return;  // flagged by vol_walk_kernel
    const Interval64 iv = interval64(P, r.o, r.d);
    const double seed = seeds[((size_t)view * P.rows + row) * P.cols + col], factor = seed * r.len;
    if (seed == 0.0 || !(iv.upper > iv.lower) || gauss_summed(P, r, iv, factor)) return;
    CellWalk walk{};
    begin_cells(P, r, iv, walk);
    double start = iv.lower;
    bool good = true;
    const long long limit = (long long)P.nx + P.ny + P.nz + 1;
    for (long long segments = 0; start < iv.upper && segments < limit; ++segments) {
        CellPiece s;
        cell_piece(P, r, walk, start, s);
        if (s.end <= start) {
            good = false;
            break;
        }
        good = good && finite3d(s.first) && finite3d(s.second);
        double vf = factor * s.radius;
        if (!isfinite(factor)) vf = product3(seed, r.len, s.radius);
        if (s.shared) {
            // kernels/projection.py:405-430 (scatter_cell)
            double f1[3], f2[3];
            const int n[3] = {P.nx, P.ny, P.nz};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double top = (double)(n[a] - 1);
                f1[a] = fmin(fmax(s.first[a], 0.0), top) - (double)s.lower[a];
                f2[a] = fmin(fmax(s.second[a], 0.0), top) - (double)s.lower[a];
            }
            const double w1 = inside_support64(P, s.first) ? vf : 0.0;
            const double w2 = inside_support64(P, s.second) ? vf : 0.0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                double first = w1, second = w2;
#pragma unroll
                for (int a = 0; a < 3; ++a) first *= ((k >> a) & 1) ? f1[a] : 1.0 - f1[a];
#pragma unroll
                for (int a = 0; a < 3; ++a) second *= ((k >> a) & 1) ? f2[a] : 1.0 - f2[a];
                good = add_increment(P, acc, corner_of(P, s.lower, k), first + second) && good;
            }
        } else {
            // kernels/projection.py:437-470 (scatter per node)
#pragma unroll
            for (int node = 0; node < 2; ++node) {
                const double *pt = node == 0 ? s.first : s.second;
                Cell64 c;
                if (!cell64(P, pt, c)) continue;
                const int lower[3] = {c.lx, c.ly, c.lz};
                const double f[3] = {c.fx, c.fy, c.fz};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    double contribution = vf;
#pragma unroll
                    for (int a = 0; a < 3; ++a) contribution *= ((k >> a) & 1) ? f[a] : 1.0 - f[a];
                    good = add_increment(P, acc, corner_of(P, lower, k), contribution) && good;
                }
            }
        }
        start = s.end;
        advance_cells(P, r, walk, s.end, iv.upper);
    }
    if (!good || start < iv.upper) flag(P, view, DPT_STATUS_RANGE);
}

// kernels/projection.py:873-1237 with cell_gauss, the pose half (the volume
// half is vol_walk_kernel).  Held to three waves per SIMD (168 VGPRs, 16 bytes
// of spills): left free it takes 172 and two (24 views of 256^2 over 128^3,
// whole call: 4.42 -> 4.05 ms).
template <typename T, int C>
__global__ __launch_bounds__(kBlock, 3) void vjp_gauss_kernel(Params P, const T *__restrict__ field,
                                                           const double *__restrict__ seeds,
                                                           double *__restrict__ partials) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    double gradient[kMaxComponents];
#pragma unroll
    for (int c = 0; c < kMaxComponents; ++c) gradient[c] = 0.0;
    const double *pose = P.poses + 12 * (size_t)view;

    // ---- per-ray setup
    bool active = false, bad = false;
    World w{};
    Ray r{};
    Interval64 iv{};
    double seed = 0.0, span = 0.0;
    if (ray_in_range(P, view, row, col)) {
        const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
        ray_world(P, pose, view, row, col, w);
        ray_grid(P, w, r);
        if (!r.valid) {
            flag(P, view, DPT_STATUS_RANGE);
        } else {
            iv = interval64(P, r.o, r.d);
            span = iv.upper - iv.lower;
            seed = seeds[ray];
            active = seed != 0.0 && span > 0.0;
        }
    }
    const double factor = seed * r.len;
    double og[3] = {0.0, 0.0, 0.0}, dg[3] = {0.0, 0.0, 0.0};
    double integral = 0.0;  // sum of radius x node value (ray coordinates)
    CellWalk walk{};
    double start = iv.lower;
    if (active) begin_cells(P, r, iv, walk);
    const long long limit = (long long)P.nx + P.ny + P.nz + 1;
    long long segments = 0;

    if (active) {
        for (; start < iv.upper && segments < limit; ++segments) {
            CellPiece s;
            cell_piece(P, r, walk, start, s);
            if (s.end <= start) {
                bad = true;
                break;
            }
            bad |= !finite3d(s.first) || !finite3d(s.second);
            double g1[3], g2[3], v1, v2;
            if (s.shared) {  // one load of the cell for both nodes
                double v[8];
                load8d<T>(P, field, (s.lower[2] * P.ny + s.lower[1]) * P.nx + s.lower[0], v);
                v1 = node_in_cell<true>(P, s.first, s.lower, v, g1);
                v2 = node_in_cell<true>(P, s.second, s.lower, v, g2);
            } else {
                v1 = node_value<T, true>(P, field, s.first, nullptr, g1);
                v2 = node_value<T, true>(P, field, s.second, nullptr, g2);
            }
            if constexpr (C == kRayCoordinates) {
                integral += s.radius * v1;
                integral += s.radius * v2;
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                og[a] += s.radius * g1[a];
                og[a] += s.radius * g2[a];
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                dg[a] += s.radius * s.first_position * g1[a];
                dg[a] += s.radius * s.second_position * g2[a];
            }
            start = s.end;
            advance_cells(P, r, walk, s.end, iv.upper);
        }
    }
    if (active) {
        bad |= start < iv.upper;
        // kernels/projection.py:1031-1046: endpoint terms of the
        // zero-extended support at the clamped clip points
        double lo_pt[3], up_pt[3];
        const int n[3] = {P.nx, P.ny, P.nz};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double hi = (double)n[a] - 0.5;
            lo_pt[a] = fmin(fmax(r.o[a] + iv.lower * r.d[a], -0.5), hi);
            up_pt[a] = fmin(fmax(r.o[a] + iv.upper * r.d[a], -0.5), hi);
        }
        const double lower_value = node_value<T, false>(P, field, lo_pt, nullptr, nullptr);
        const double upper_value = node_value<T, false>(P, field, up_pt, nullptr, nullptr);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double lo_o = (iv.lo_axis == a) ? iv.lo_o : 0.0, lo_d = (iv.lo_axis == a) ? iv.lo_d : 0.0;
            const double up_o = (iv.up_axis == a) ? iv.up_o : 0.0, up_d = (iv.up_axis == a) ? iv.up_d : 0.0;
            og[a] += upper_value * up_o - lower_value * lo_o;
            dg[a] += upper_value * up_d - lower_value * lo_d;
        }
        if (isfinite(factor)) {
            pose_epilogue<C>(P, pose, w, factor, og, dg, gradient, seed, integral, true);
        } else {
            double sa[3], da[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double sg = P.g[i] * og[0] + P.g[3 + i] * og[1] + P.g[6 + i] * og[2];
                const double rg = P.g[i] * dg[0] + P.g[3 + i] * dg[1] + P.g[6 + i] * dg[2];
                sa[i] = product4(seed, r.len, 1.0, sg);
                da[i] = product4(seed, r.len, 1.0, rg);
            }
            Params unit = P;
            for (int i = 0; i < 9; ++i) unit.g[i] = (i % 4 == 0) ? 1.0 : 0.0;
            pose_epilogue<C>(unit, pose, w, 1.0, sa, da, gradient, seed, integral, true);
        }
    }
    if (bad) flag(P, view, DPT_STATUS_RANGE);
    store_gradient<C>(P, gradient, partials, wslot, wave_valid, view, row, col);
}

// --------------------------------------------------- volume adjoint walk ---
// Volume cotangents of the FP32 and FP64 midpoint rules
// (kernels/projection_fp32.py:437-548, kernels/projection.py:396-430), one
// step per (ray, cell) instead of one per sample.  Inside a cell the fractions
// are linear in the sample index, so the corner sums of the cell's n samples
// follow from the fractions m at their mean and the variance v = (n^2 - 1) / 12
// of the index: sum fx fy = n (mx my + v bx by), b the advance per sample, and
// likewise the triple product (the odd moments vanish).  About 80 VALU
// instructions a cell, against 110 a sample (2.5 samples a cell on the full
// scan) when every sample formed its weights; the sums leave out the FP32
// rounding of each sample's position (volume gradient of a 4-view full scan
// against FP64: 2.0e-6, sample by sample 8.3e-6).  Which of two cells takes a
// sample on their common face does not matter: the weights are continuous.
//
// A workgroup walks its rays through slabs of grid samples along the axis most
// of them advance fastest along, every lane its samples inside the slab, and
// privatises the box of cells they visit in an LDS brick.  Lanes take about
// the same number of steps per slab whatever their sample spacing, so a slab
// costs no lockstep waste; a slab whose box overflows the brick is halved, and
// the next one doubled while it fits.
//
// Where rays lie more than three to four voxels apart (kWalkSparse) a brick holds
// mostly zeros: its box fills the LDS with a slab of a few samples, and the
// bounds, barriers and drain of every slab cost more than the few sums they
// merge.  Such a workgroup adds its corner sums by device atomics at once, two
// x-adjacent entries a request from a pair of lanes; it is found when a slab of
// eight samples overflows (asked at sixteen, 30 views of 128^2 over 128^3 ran 6
// % slower; asked at four, 24 views of 128^2 over 256^3 at S = 64 took 4.3
// instead of 2.1 ms).  Bricks pay longer for rays along y and z: their slabs are
// thin across x no more than the rays allow, and a drain request adds a run of
// a row, where the entries of rays along x follow one another in pairs anyway.
// MI355X, bricks and atomics: 24 views over 256^3 at S = 512, panels of 96^2 /
// 128^2 / 160^2 (0.06 / 0.11 / 0.17 rays a voxel) 8.6 and 4.3 / 9.2 and 7.5 /
// 12.4 and 11.6 ms, of 192^2 (0.25) 8.5 and 16.4; 60 views of 24^2 over 128^3
// 3.9 and 0.45 ms; 2^18 random rays in 256^3 5.8 and 2.2; 2^16 by the exact rule
// in 128^3 1.51 and 0.49.  Over 101 scenes of 20 to 30 views (128 x 40 x 128 to
// 512^3, 0.06 to 0.2 rays a voxel, S 48 to 1024) the walk takes 0.56 of the time of
// bricks alone, worst 1.29 (1.7 -> 2.2 ms, 300 x 74 x 225 at S = 1000), with 0.12
// for every axis 0.60 and 1.54.
//
// Bound by the device atomics of the drain (one request per 64-byte block,
// 23.6 G/s), the LDS atomics and VALU issue, in turn.  MI355X, before (per
// sample, joint with the pose) and after (walk + pose launch): 360-view 512^2
// scan of 256^3 at S = 1024 262 -> 62 + 74 ms; 24 views of 256^2 over 256^3 in
// bfloat16 24.5 -> 5.7 + 2.2 ms; 60 views of 256^2 over 128^3 (volume only)
// 7.8 -> 2.0 ms; FP64 24 views of 256^2 over 128^3 18.5 -> 0.9 + 2.2 ms.
// A ray in sample-index units: coordinate a of sample k is A[a] + k B[a].
struct WalkRay {
    double A[3], B[3];
};

constexpr double kWalkBias = 0x1.8p20;         // 1.5 * 2^20: a sum's low word is the fraction in 2^-32 units
constexpr int kWalkBiasHigh = 0x41380000;      // high word of the bias: the difference is floor(coordinate)
constexpr int kWalkWidth = 16;                  // grid samples of the first slab
constexpr int kWalkMaxAxis = 1 << 18;          // largest axis of the biased form
// Least rays per grid sample of a slab's cross-section worth a brick: rays that
// advance fastest along x, and others.
constexpr float kWalkSparseX = 0.12f, kWalkSparse = 0.06f;

// Floor and fraction of coordinate a of sample k (R float: through the bias,
// 2^-32 resolution; R double: exact).
template <typename R>
__device__ __forceinline__ void walk_split(double A, double B, double k, int &l, R &f) {
    if constexpr (std::is_same<R, float>::value) {
        const double q = fma(k, B, A);  // A carries the bias
        l = __double2hiint(q) - kWalkBiasHigh;
        f = (float)(unsigned)__double2loint(q) * 0x1p-32f;
    } else {
        const double p = fma(k, B, A);
        const double lo = floor(p);
        l = (int)lo;
        f = p - lo;
    }
}

template <typename R>
__device__ __forceinline__ int walk_lower(double A, double B, double k, int cap) {
    int l;
    if constexpr (std::is_same<R, float>::value) {
        l = __double2hiint(fma(k, B, A)) - kWalkBiasHigh;
    } else {
        l = (int)floor(fma(k, B, A));
    }
    return min(max(l, 0), cap);
}

__device__ __forceinline__ float walk_min(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double walk_min(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ float walk_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double walk_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float walk_floor(float a) { return floorf(a); }
__device__ __forceinline__ double walk_floor(double a) { return floor(a); }
__device__ __forceinline__ float walk_unit(float a) { return __builtin_amdgcn_fmed3f(a, 0.0f, 1.0f); }
__device__ __forceinline__ double walk_unit(double a) { return fmin(fmax(a, 0.0), 1.0); }

// The value of the other lane of a pair of lanes (quad_perm [1, 0, 3, 2]); both
// must be active.
__device__ __forceinline__ int pair_lane(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true); }
__device__ __forceinline__ float pair_lane(float v) { return __int_as_float(pair_lane(__float_as_int(v))); }
__device__ __forceinline__ double pair_lane(double v) {
    return __hiloint2double(pair_lane(__double2hiint(v)), pair_lane(__double2loint(v)));
}

// Add the brick's non-zero entries to the FP64 accumulator and clear them,
// 16 lanes to a row of x-adjacent entries: device atomics cost per 64-byte
// block (23.6 G blocks/s measured, whether 1 or 8 entries of it are added).
__device__ __forceinline__ void walk_drain(const Params &P, const Brick &B, double *brick, double *acc) {
    const float inv_by = 1.0f / (float)B.by;
    const int rows = B.by * B.bz;
    for (int q = threadIdx.x >> 4; q < rows; q += kBlock / 16) {
        int z = (int)((float)q * inv_by);
        z -= (z * B.by > q) ? 1 : 0;
        z += ((z + 1) * B.by <= q) ? 1 : 0;
        const int y = q - z * B.by;
        const int row = ((B.z0 + z) * P.ny + (B.y0 + y)) * P.nx + B.x0;
        for (int x = (int)(threadIdx.x & 15) - (row & 7); x < B.bx; x += 16) {
            const double v = x >= 0 ? brick[q * B.bx + x] : 0.0;
            if (v != 0.0) {
                brick[q * B.bx + x] = 0.0;
                unsafeAtomicAdd(&acc[row + x], v);
            }
        }
    }
}

// S: sampling arithmetic (float / double), R: arithmetic of the fractions and
// corner sums (float, or double for FP64 sampling and for FP32 sampling of
// grids with an axis beyond kWalkMaxAxis).
// GAUSS: the exact cell-Gauss rule; the walk runs in the ray parameter, a step is
// a piece between crossings, and its two nodes at centre +- radius / sqrt(3)
// are a run of two samples with index variance radius^2 / 3 (24 views of 256^2
// over 128^3: joint adjoint 4.15 -> 1.09 + 1.45 ms; two products a corner and
// node and 6.1e7 device atomics before).
// FP32 sums keep six waves per SIMD (80 VGPRs, 32 bytes of spills; 90 and five
// without the bound: full scan 61.9 and 62.9 ms), FP64 ones take four (121; five
// spill 92 bytes: 24 views of 256^2 over 128^3 by the exact rule 1.25 and 1.40
// ms).
template <typename S, typename R, bool GAUSS = false>
__global__ __launch_bounds__(kBlock, (std::is_same<R, float>::value ? 6 : 4)) void vol_walk_kernel(Params P, const S *__restrict__ seeds,
                                                          double *__restrict__ acc) {
    extern __shared__ double brick[];
    __shared__ int bound_red[kBlock / 64][6], ray_red[kBlock / 64];
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    const double *pose = P.poses + 12 * (size_t)view;
    int first = 0, last = P.samples;
    if (P.segments > 1) {
        const int seg = tile_index(P) / P.base_tiles;
        first = seg * P.segment_samples;
        last = min(first + P.segment_samples, P.samples);
    }
    // the range of the walk: sample indices, or ray parameters (GAUSS)
    double walk_first = (double)first, walk_last = (double)last;
    bool summed = false, scattered = false, bad = false;
    WalkRay W{};
    S o[3] = {0, 0, 0}, d[3] = {0, 0, 0}, lower = 0, step = 0, volume_factor = 0;
    if (ray_in_range(P, view, row, col)) {
        const size_t ray = ((size_t)view * P.rows + row) * P.cols + col;
        World w;
        ray_world(P, pose, view, row, col, w);
        Ray r;
        ray_grid(P, w, r);
        if constexpr (std::is_same<S, float>::value) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                o[a] = (float)r.o[a];
                d[a] = (float)r.d[a];
            }
            const float len = (float)r.len;
            if (!r.valid || !finite3f(o[0], o[1], o[2]) || !finite3f(d[0], d[1], d[2]) || !isfinite(len) ||
                len <= 0.0f) {
                flag(P, view, DPT_STATUS_RANGE);
            } else {
                const Interval32 iv = interval32(P, o, d);
                const float span = iv.upper - iv.lower;
                const float seed = seeds[ray];
                if (!isfinite(seed)) flag(P, view, DPT_STATUS_RANGE);
                if (span > 0.0f && seed != 0.0f) {
                    lower = iv.lower;
                    step = span / (float)P.samples;
                    volume_factor = seed * (len * step);
                    const bool finite = finite_span(o, d, lower, step, 0, P.samples);
                    bad = !finite;
                    const float m = fabsf(volume_factor);
                    summed = finite && m >= 0x1p-102f && m <= 0x1p96f;
                    scattered = !summed;
                    if (summed && !span_inside(P, o, d, lower, step, 0, P.samples)) {
                        // rounding put end samples outside (chords of a tenth
                        // of a voxel and less): the samples inside are a run
                        const auto inside = [&](int k) {
                            const float pos = fmaf((float)k + 0.5f, step, lower);
                            return inside32(P, fmaf(pos, d[0], o[0]), fmaf(pos, d[1], o[1]), fmaf(pos, d[2], o[2]));
                        };
                        const int middle = P.samples / 2;
                        if (inside(middle)) {
                            int below = 0, above = middle;  // first sample inside
                            while (below < above) {
                                const int k = (below + above) >> 1;
                                if (inside(k))
                                    above = k;
                                else
                                    below = k + 1;
                            }
                            walk_first = fmax(walk_first, (double)below);
                            below = middle;
                            above = P.samples - 1;  // last sample inside
                            while (below < above) {
                                const int k = (below + above + 1) >> 1;
                                if (inside(k))
                                    below = k;
                                else
                                    above = k - 1;
                            }
                            walk_last = fmin(walk_last, (double)(below + 1));
                            summed = walk_last > walk_first;
                        } else {
                            summed = false;
                            scattered = true;
                        }
                    }
                }
            }
        } else {
            if (!r.valid) {
                flag(P, view, DPT_STATUS_RANGE);
            } else {
                const Interval64 iv = interval64(P, r.o, r.d);
                double span = iv.upper - iv.lower;
                const double seed = seeds[ray];
                if (seed == 0.0) span = 0.0;
                if (span > 0.0) {
                    const double count = (double)P.samples;
                    const double factor = seed * r.len;
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        o[a] = r.o[a];
                        d[a] = r.d[a];
                    }
                    lower = iv.lower;
                    if constexpr (GAUSS) {
                        walk_first = iv.lower;
                        walk_last = iv.upper;
                        volume_factor = factor;
                        summed = gauss_summed(P, r, iv, factor);
                    } else {
                        step = span / count;
                        volume_factor = factor * span / count;
                        if (!isfinite(factor)) volume_factor = product4(seed, r.len, span, 1.0 / count);
                        const double pa = lower + 0.5 * step, pb = lower + (count - 0.5) * step;
                        const double qa[3] = {o[0] + pa * d[0], o[1] + pa * d[1], o[2] + pa * d[2]};
                        const double qb[3] = {o[0] + pb * d[0], o[1] + pb * d[1], o[2] + pb * d[2]};
                        const double m = fabs(volume_factor);
                        summed = walk_factor64(P, m) && inside_support64(P, qa) && inside_support64(P, qb);
                        scattered = !summed;
                    }
                }
            }
        }
    }
    for (int i = threadIdx.x; i < P.walk_cap; i += kBlock) brick[i] = 0.0;
    if (summed) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            W.B[a] = GAUSS ? (double)d[a] : (double)step * (double)d[a];
            W.A[a] = GAUSS ? (double)o[a] : fma((double)lower + 0.5 * (double)step, (double)d[a], (double)o[a]);
        }
    }

    // ---- slabs along the axis most rays advance fastest along
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double ad[3] = {fabs(W.B[0]), fabs(W.B[1]), fabs(W.B[2])};
    const int mine = ad[0] >= ad[1] && ad[0] >= ad[2] ? 0 : (ad[1] >= ad[2] ? 1 : 2);
    int my_votes[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) my_votes[a] = __popcll(__builtin_amdgcn_ballot_w64(summed && mine == a));
    if (lane == 0)
        for (int a = 0; a < 3; ++a) bound_red[wv][a] = my_votes[a];
    __syncthreads();
    int votes[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) votes[a] = bound_red[0][a] + bound_red[1][a] + bound_red[2][a] + bound_red[3][a];
    const int axis = votes[0] >= votes[1] && votes[0] >= votes[2] ? 0 : (votes[1] >= votes[2] ? 1 : 2);
    const double slab_A = axis == 0 ? W.A[0] : (axis == 1 ? W.A[1] : W.A[2]);
    const double slab_B = axis == 0 ? W.B[0] : (axis == 1 ? W.B[1] : W.B[2]);
    int lo = INT_MAX, nhi = INT_MAX;
    if (summed) {
        const double q0 = fma(walk_first, slab_B, slab_A);
        const double q1 = fma(GAUSS ? walk_last : walk_last - 1.0, slab_B, slab_A);
        lo = (int)floor(fmin(q0, q1));
        nhi = -((int)floor(fmax(q0, q1)) + 1);
    }
    lo = wave_min(lo);
    nhi = wave_min(nhi);
    __syncthreads();  // every wave has read the votes
    if (lane == 0) {
        bound_red[wv][3] = lo;
        bound_red[wv][4] = nhi;
    }
    __syncthreads();
    const int slab_lo = min(min(bound_red[0][3], bound_red[1][3]), min(bound_red[2][3], bound_red[3][3]));
    const int slab_hi = -min(min(bound_red[0][4], bound_red[1][4]), min(bound_red[2][4], bound_red[3][4]));
    __syncthreads();  // bound_red is reused by the slab bounds
    if (slab_lo != INT_MAX) {
        // the sample index at which the slab coordinate reaches b: (b - A) / B
        const bool up = slab_B >= 0.0;
        const double slab_inv = fabs(slab_B) > 1e-30 ? 1.0 / slab_B : 1e30;
        double done = up ? walk_first : walk_last;  // samples on the low side of the slab are walked
        R inv[3], lead[3], adv[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const bool moves = fabs(W.B[a]) > 1e-18;
            inv[a] = moves ? (R)(1.0 / W.B[a]) : (R)0;
            lead[a] = moves ? (W.B[a] > 0.0 ? inv[a] : (R)0) : (R)1e30;
            adv[a] = (R)W.B[a];
            if constexpr (std::is_same<R, float>::value) W.A[a] += kWalkBias;
        }
        const int cap[3] = {P.capx, P.capy, P.capz};
        int width = GAUSS ? max(1, (slab_hi - slab_lo) / P.gauss_chunks) : kWalkWidth;
        // where the walk crosses slab coordinate b; `whole`: the first sample beyond it
        auto crossing = [&](int b, bool whole) {
            double t = ((double)b - slab_A) * slab_inv;
            if (whole) t = up ? ceil(t) : floor(t) + 1.0;
            return fmin(fmax(t, walk_first), walk_last);
        };
        auto cell_bounds = [&](double k0, double k1, bool inclusive, int *blo, int *bnhi) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                blo[a] = bnhi[a] = INT_MAX;
                if (k1 > k0) {
                    const int la = walk_lower<R>(W.A[a], W.B[a], k0, cap[a]);
                    const int lb = walk_lower<R>(W.A[a], W.B[a], inclusive ? k1 : k1 - 1.0, cap[a]);
                    blo[a] = min(la, lb);
                    bnhi[a] = -max(la, lb);
                }
            }
        };
        // the rays through a thin slab in the middle against the cross-section
        // of its box (one barrier before, one after the bound's own)
        auto too_sparse = [&]() {
            const int m0 = (slab_lo + slab_hi) / 2 - 2;
            const double t0 = crossing(m0, false), t1 = crossing(m0 + 4, false);
            const double k0 = fmin(t0, t1), k1 = summed ? fmax(t0, t1) : k0;
            const int rays = __popcll(__builtin_amdgcn_ballot_w64(k1 > k0));
            int blo[3], bnhi[3], e[3];
            cell_bounds(k0, k1, true, blo, bnhi);
            __syncthreads();  // the bound rewrites bound_red
            if (lane == 0) ray_red[wv] = rays;
            Brick B{};
            (void)chunk_brick(P, bound_red, blo, bnhi, P.walk_cap, P.nx > 1, B, e);
            const float across = axis == 0 ? (float)e[1] * e[2] : (axis == 1 ? (float)e[0] * e[2] : (float)e[0] * e[1]);
            const bool sparse = (float)(ray_red[0] + ray_red[1] + ray_red[2] + ray_red[3]) <
                                (axis == 0 ? kWalkSparseX : kWalkSparse) * across;
            return (bool)__builtin_amdgcn_readfirstlane(sparse);
        };
        bool weighed = false, sparse = false;  // asked once, when a thin slab's box overflows the brick
        for (int s0 = slab_lo; s0 < slab_hi;) {
            // ---- this slab's samples [k0, k1) of the lane and its brick
            double k0, k1, next;
            int s1;
            long long box;
            Brick B{};
            bool use_lds;
            for (;;) {
                s1 = sparse ? slab_hi : min(s0 + width, slab_hi);  // sparse: all that is left
                const double t = s1 == slab_hi ? (up ? walk_last : walk_first) : crossing(s1, !GAUSS);
                next = up ? fmax(t, done) : fmin(t, done);
                k0 = fmin(next, done);
                k1 = summed ? fmax(next, done) : k0;
                use_lds = false;
                box = 0;
                if (sparse) break;
                int blo[3], bnhi[3], e[3];
                cell_bounds(k0, k1, GAUSS, blo, bnhi);
                use_lds = chunk_brick(P, bound_red, blo, bnhi, P.walk_cap, P.nx > 1, B, e);
                box = (long long)e[0] * e[1] * e[2];
                if (box <= P.walk_cap || s1 - s0 <= 1) break;
                width = max(1, (s1 - s0) >> 1);
                if (!weighed && s1 - s0 <= kWalkWidth / 2) {
                    weighed = true;
                    sparse = too_sparse();
                }
                __syncthreads();  // the next bound rewrites bound_red
            }
            done = next;
            // as wide as the brick holds
            width = 2 * (use_lds ? (long long)B.volume : box) <= P.walk_cap ? 2 * (s1 - s0) : s1 - s0;
            s0 = s1;
            // Mean corner weights of a run at mean fractions f, index variance
            // var and advances b, times g.  Each is a product of its own
            // fractions plus the covariances, not a difference of the others,
            // so a small corner keeps its relative accuracy, and is clamped to
            // [0, 1] (the mean of weights; an output modifier of the multiply-
            // add) where the covariances cancel it: sums of a non-negative
            // image stay non-negative.  Four instructions more than corners
            // by subtraction.
            auto realised = [&](R x) { return GAUSS ? destination_increment(P, (double)x) : (double)x; };
            // IN_BRICK: into the brick.  Otherwise by device atomics, and the
            // whole wave calls: the two lanes of a pair add the x-adjacent
            // entries of the even lane's rows, then of the odd lane's, one
            // request for both entries (a lane without a run adds nothing).
            auto deposit = [&](auto in_brick, bool live, const int *l, const R *f, const R *b, R var, R g) {
                const R fx = f[0], fy = f[1], fz = f[2];
                const R gx = (R)1 - fx, gy = (R)1 - fy, gz = (R)1 - fz;
                const R vx = var * b[0], vy = var * b[1];
                const R exy = vx * b[1], exz = vx * b[2], eyz = vy * b[2];
                const R m[4] = {walk_fma(gx, gy, exy), walk_fma(fx, gy, -exy), walk_fma(gx, fy, -exy),
                                walk_fma(fx, fy, exy)};
                const R xf = exz * fy, xg = exz * gy, yf = eyz * fx, yg = eyz * gx;
                const R u[4] = {-(xg + yg), xg - yf, yg - xf, xf + yf};
                R c[8];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    c[k] = walk_unit(walk_fma(m[k], gz, -u[k]));
                    c[k + 4] = walk_unit(walk_fma(m[k], fz, u[k]));
                }
                if constexpr (decltype(in_brick)::value) {
                    const int at = (int)(__umul24(__umul24((unsigned)l[2], (unsigned)B.by) + (unsigned)l[1],
                                                  (unsigned)B.bx) + (unsigned)l[0]) - B.origin;
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        atomicAdd(&brick[at + ((k & 1) ? B.lsx : 0) + ((k & 2) ? B.lsy : 0) + ((k & 4) ? B.lsz : 0)],
                                  realised(g * c[k]));
                } else {
                    const bool odd = lane & 1;
                    const int at = (l[2] * P.ny + l[1]) * P.nx + l[0], pair = pair_lane(at);
                    const int even_at = odd ? pair + P.sx : at, odd_at = odd ? at + P.sx : pair;
#pragma unroll
                    for (int k = 0; k < 8; k += 2) {
                        const R low = live ? g * c[k] : (R)0, high = live ? g * c[k + 1] : (R)0;
                        const R from = pair_lane(odd ? low : high);
                        const double even_sum = realised(odd ? from : low), odd_sum = realised(odd ? high : from);
                        const int row = corner_offset(P, k);
                        if (even_sum != 0.0) unsafeAtomicAdd(&acc[even_at + row], even_sum);
                        if (odd_sum != 0.0) unsafeAtomicAdd(&acc[odd_at + row], odd_sum);
                    }
                }
            };
            // the half cell beyond a face, and a singleton axis: the clamped
            // coordinate is constant
            const unsigned top[3] = {(unsigned)P.nx - 1u, (unsigned)P.ny - 1u, (unsigned)P.nz - 1u};
            auto clamp_cell = [&](int *l, R *f, R *b) {
                if ((unsigned)l[0] >= top[0] || (unsigned)l[1] >= top[1] ||
                    (unsigned)l[2] >= top[2]) {
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const bool outside = (unsigned)l[a] >= top[a];
                        const bool below = l[a] < 0;
                        b[a] = outside ? (R)0 : b[a];
                        f[a] = outside ? (below ? (R)0 : (R)1) : f[a];
                        l[a] = min(max(l[a], 0), cap[a]);
                    }
                }
            };
            auto march = [&](auto in_brick) {
                constexpr bool IN_BRICK = decltype(in_brick)::value;
                // lanes step alone, or (IN_BRICK false) the wave as one
                const auto more = [](bool left) { return IN_BRICK ? left : __builtin_amdgcn_ballot_w64(left) != 0; };
                if constexpr (GAUSS) {
                    // ---- one step per piece
                    double t0 = k0, plane[3], next_t[3];
                    const auto unit = [&](int a) { return W.B[a] >= 0.0 ? 1.0 : -1.0; };
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const double q = fma(t0, W.B[a], W.A[a]);
                        const bool moves = inv[a] != 0.0;
                        plane[a] = W.B[a] >= 0.0 ? floor(q) + 1.0 : ceil(q) - 1.0;
                        next_t[a] = moves ? (plane[a] - W.A[a]) * inv[a] : 1e300;
                        if (next_t[a] <= t0) {
                            plane[a] += unit(a);
                            next_t[a] = (plane[a] - W.A[a]) * inv[a];
                        }
                    }
                    // every step passes a plane or ends the slab; one that does not
                    // advance (planes closer than the rounding of the ray
                    // parameter) flags the view, as in the other kernels of the rule
                    for (int left = P.nx + P.ny + P.nz + 8; left > 0 && more(t0 < k1); --left) {
                        const double t1 = fmin(fmin(next_t[0], next_t[1]), fmin(next_t[2], k1));
                        const bool live = t0 < k1, ahead = t1 > t0;
                        bad |= live && !ahead;
                        if (!IN_BRICK || ahead) {
                            const double radius = 0.5 * (t1 - t0), centre = t0 + radius;
                            int l[3];
                            R f[3], b[3];
#pragma unroll
                            for (int a = 0; a < 3; ++a) {
                                walk_split<R>(W.A[a], W.B[a], centre, l[a], f[a]);
                                b[a] = adv[a];
                            }
                            clamp_cell(l, f, b);
                            deposit(in_brick, live && ahead, l, f, b, radius * radius * (1.0 / 3.0),
                                    2.0 * (radius * volume_factor));
                        }
#pragma unroll
                        for (int a = 0; a < 3; ++a)
                            if (next_t[a] <= t1) {
                                plane[a] += unit(a);
                                next_t[a] = (plane[a] - W.A[a]) * inv[a];
                            }
                        t0 = fmax(t0, t1);
                    }
                    bad |= t0 < k1;
                } else {
                    // ---- one step per cell
                    R kf = (R)k0;
                    const R kend = (R)k1;
                    while (more(kf < kend)) {
                        const bool live = kf < kend;
                        int l[3];
                        R f[3], b[3];
                        R run = (R)1e30;
#pragma unroll
                        for (int a = 0; a < 3; ++a) {
                            walk_split<R>(W.A[a], W.B[a], (double)kf, l[a], f[a]);
                            // samples until the coordinate leaves [l, l + 1]
                            run = walk_min(run, walk_fma(-f[a], inv[a], lead[a]));
                            b[a] = adv[a];
                        }
                        R n = walk_min(walk_floor(run) + (R)1, kend - kf);
                        if (!IN_BRICK) n = live ? n : (R)0;
                        kf += n;
                        clamp_cell(l, f, b);
                        const R half = (R)0.5 * (n - (R)1);
                        const R var = walk_fma(n * (R)(1.0 / 12.0), n, (R)(-1.0 / 12.0));
#pragma unroll
                        for (int a = 0; a < 3; ++a) f[a] = walk_fma(b[a], half, f[a]);
                        deposit(in_brick, live, l, f, b, var, n * (R)volume_factor);
                    }
                }
            };
            if (use_lds) {
                march(std::true_type{});
                __syncthreads();
                walk_drain(P, B, brick, acc);
            } else {
                march(std::false_type{});
            }
            __syncthreads();
        }
    }
    // Rays outside the factor range, or whose middle sample (FP64: whose first or
    // last one) falls outside the support: the reference's increments, per sample
    // and corner, by device atomics.
    if (scattered) {
        if constexpr (std::is_same<S, float>::value) {
            for (int k = first; k < last; ++k) {
                const float pos = fmaf((float)k + 0.5f, step, lower);
                const float p0 = fmaf(pos, d[0], o[0]);
                const float p1 = fmaf(pos, d[1], o[1]);
                const float p2 = fmaf(pos, d[2], o[2]);
                if (!inside32(P, p0, p1, p2)) continue;
                Cell32 c;
                cell32_inside(P, p0, p1, p2, c);
                float wt[8];
                weights32(c, wt);
                const int voxel = (c.lz * P.ny + c.ly) * P.nx + c.lx;
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    const float inc = P.volume_f64 ? volume_factor * wt[kk] : scatter_increment(volume_factor, wt[kk]);
                    bad |= !isfinite(inc);
                    if (inc != 0.0f) unsafeAtomicAdd(&acc[voxel + corner_offset(P, kk)], (double)inc);
                }
            }
        } else if constexpr (!GAUSS) {
            for (int k = first; k < last; ++k) {
                const double pos = lower + ((double)k + 0.5) * step;
                const double p[3] = {o[0] + pos * d[0], o[1] + pos * d[1], o[2] + pos * d[2]};
                bad |= !finite3d(p);
                Cell64 c;
                if (!cell64(P, p, c)) continue;
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    double contribution = volume_factor;
                    contribution *= (kk & 1) ? c.fx : 1.0 - c.fx;
                    contribution *= (kk & 2) ? c.fy : 1.0 - c.fy;
                    contribution *= (kk & 4) ? c.fz : 1.0 - c.fz;
                    const double rounded = destination_increment(P, contribution);
                    bad |= !isfinite(rounded);
                    if (rounded != 0.0) unsafeAtomicAdd(&acc[c.base + corner_offset(P, kk)], rounded);
                }
            }
        }
    }
    if (bad) flag(P, view, DPT_STATUS_RANGE);
}

// ------------------------------------------------------- small kernels ----

// Fixed-order FP64 sum of the tile partials of one view (kernels/reductions.py
// role), then write or accumulate and flag non-finite results.
template <int C>
__global__ __launch_bounds__(kBlock) void pose_reduce_kernel(const double *__restrict__ partials,
                                                             int tiles_per_view, double *grad_pose,
                                                             int accumulate, int *status) {
    const int view = blockIdx.x;
    // every component at once: per-thread strided sums, then one pairwise
    // tree per component (the order of a component-by-component pass)
    __shared__ double s[C][kBlock];
    const double *base = partials + (size_t)view * tiles_per_view * C;
    double v[C];
#pragma unroll
    for (int c = 0; c < C; ++c) v[c] = 0.0;
    for (int t = threadIdx.x; t < tiles_per_view; t += kBlock) {
#pragma unroll
        for (int c = 0; c < C; ++c) v[c] += base[(size_t)t * C + c];
    }
#pragma unroll
    for (int c = 0; c < C; ++c) s[c][threadIdx.x] = v[c];
    __syncthreads();
    for (int stride = kBlock / 2; stride > 0; stride >>= 1) {
        if (threadIdx.x < stride) {
#pragma unroll
            for (int c = 0; c < C; ++c) s[c][threadIdx.x] += s[c][threadIdx.x + stride];
        }
        __syncthreads();
    }
    if (threadIdx.x < C) {
        const int c = threadIdx.x;
        double result = s[c][0];
        if (accumulate) result += grad_pose[(size_t)view * C + c];
        grad_pose[(size_t)view * C + c] = result;
        if (!isfinite(result)) atomicOr(&status[view], DPT_STATUS_RANGE);
    }
}

// kernels/projection_checks.py:20-24 / :36-46 (physical field: finite, >= 0)
template <typename T>
__global__ __launch_bounds__(kBlock) void check_field_kernel(const T *__restrict__ field, int64_t n,
                                                             int *status) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const float v = load_value<T>(field, (int)i);
        bad |= !(isfinite(v) && v >= 0.0f);
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(&status[0], DPT_STATUS_DOMAIN);
}

// kernels/projection_checks.py:49-58
template <typename T>
__global__ __launch_bounds__(kBlock) void check_finite_kernel(const T *__restrict__ x, int64_t n,
                                                              int *status) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        bad |= !isfinite(x[i]);
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(&status[0], DPT_STATUS_RANGE);
}

// kernels/batched_geometry.py:71-88 + kernels/geometry.py:55-74
__global__ void check_poses_kernel(const double *__restrict__ poses, int views, int *status) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= views) return;
    const bool valid = pose_is_rigid(poses + 12 * (size_t)v);
    if (!valid) atomicOr(&status[v], DPT_STATUS_POSE);
}

__global__ __launch_bounds__(kBlock) void fill_f64_kernel(double *__restrict__ x, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        x[i] = 0.0;
}

__global__ void fill_i32_kernel(int *__restrict__ x, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0;
}

// FP64 accumulator -> FP32 or FP64 gradient (write or accumulate) + finite
// check (kernels/projection_checks.py:49-58 applied to the final gradient).
template <typename G>
__global__ __launch_bounds__(kBlock) void finish_volume_kernel(const double *__restrict__ acc,
                                                               G *__restrict__ grad, int64_t n,
                                                               int accumulate, int *status) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        // the previous value joins the FP64 sum: one rounding to G, and no
        // FP32 overflow of a sum that the previous value brings back in range
        double sum = acc[i];
        if (accumulate) sum += (double)grad[i];
        const G v = (G)sum;
        grad[i] = v;
        bad |= !isfinite(v);
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(&status[0], DPT_STATUS_RANGE);
}

// FP32 -> bf16/f16 with round-to-nearest-even, plus the physical-field check.
template <typename T>
__global__ __launch_bounds__(kBlock) void convert_kernel(const float *__restrict__ src, T *__restrict__ dst,
                                                         int64_t n, int *status) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const float v = src[i];
        bad |= !(isfinite(v) && v >= 0.0f);
        if constexpr (std::is_same<T, __half>::value) {
            dst[i] = __float2half_rn(v);
        } else {
            dst[i] = __float2bfloat16(v);
        }
    }
    if (status != nullptr && __any(bad) && (threadIdx.x & 63) == 0) atomicOr(&status[0], DPT_STATUS_DOMAIN);
}

// Linear (nz, ny, nx) field -> cell layout (DPT_STORE_CELLS), one lane per
// cell: the 8 corners of cell (i, j, k) in corner order (bit 0 x, bit 1 y,
// bit 2 z), +1 neighbours clamped to the grid as the gather's zero strides
// do on singleton axes.  E is the element's bit pattern (uint32_t for FP32,
// uint16_t for BF16/FP16); a cell is written with 16-byte stores.
template <typename E>
__global__ __launch_bounds__(kBlock) void cells_kernel(const E *__restrict__ src, E *__restrict__ dst, int nx,
                                                       int ny, int nz, int mx, int my, int cells) {
    for (int c = blockIdx.x * kBlock + threadIdx.x; c < cells; c += gridDim.x * kBlock) {
        const int i = c % mx, r = c / mx;
        const int j = r % my, k = r / my;
        const int i1 = min(i + 1, nx - 1), j1 = min(j + 1, ny - 1), k1 = min(k + 1, nz - 1);
        const int64_t slab = (int64_t)nx * ny;
        const int64_t a = k * slab + (int64_t)j * nx, b = k * slab + (int64_t)j1 * nx;
        const int64_t e = k1 * slab + (int64_t)j * nx, f = k1 * slab + (int64_t)j1 * nx;
        const uint32_t v[8] = {src[a + i], src[a + i1], src[b + i], src[b + i1],
                               src[e + i], src[e + i1], src[f + i], src[f + i1]};
        if constexpr (sizeof(E) == 4) {
            Quad *q = reinterpret_cast<Quad *>(dst) + 2 * (size_t)c;
            q[0] = Quad{v[0], v[1], v[2], v[3]};
            q[1] = Quad{v[4], v[5], v[6], v[7]};
        } else {
            Quad *q = reinterpret_cast<Quad *>(dst) + (size_t)c;
            *q = Quad{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
        }
    }
}

// Linear FP32 field -> quad layout, one lane per (i, j, plane): corners (i, j),
// (i+1, j), (i, j+1), (i+1, j+1) of the plane, +1 neighbours clamped as in the
// cell layout.
__global__ __launch_bounds__(kBlock) void quads_kernel(const uint32_t *__restrict__ src, Quad *__restrict__ dst, int nx,
                                                       int ny, int mx, int my, int64_t quads) {
    for (int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x; c < quads; c += (int64_t)gridDim.x * kBlock) {
        const int i = (int)(c % mx);
        const int64_t r = c / mx;
        const int j = (int)(r % my);
        const int64_t k = r / my;
        const int i1 = min(i + 1, nx - 1), j1 = min(j + 1, ny - 1);
        const int64_t a = (k * ny + j) * nx, b = (k * ny + j1) * nx;
        dst[c] = Quad{src[a + i], src[a + i1], src[b + i], src[b + i1]};
    }
}

// Count rays whose FP32 clipped interval is non-empty (effective samples =
// count * samples); same setup arithmetic as the forward kernel.
__global__ __launch_bounds__(kBlock) void count_hits_kernel(Params P, unsigned long long *count) {
    int view, row, col, wslot;
    bool wave_valid;
    if (!lane_ray(P, view, row, col, wslot, wave_valid)) return;
    bool hit = false;
    if (ray_in_range(P, view, row, col)) {
        const double *pose = P.poses + 12 * (size_t)view;
        World w;
        ray_world(P, pose, view, row, col, w);
        Ray r;
        ray_grid(P, w, r);
        float o[3] = {(float)r.o[0], (float)r.o[1], (float)r.o[2]};
        float d[3] = {(float)r.d[0], (float)r.d[1], (float)r.d[2]};
        if (r.valid) {
            const Interval32 iv = interval32(P, o, d);
            hit = iv.upper > iv.lower;
        }
    }
    const unsigned long long lanes = __popcll(__ballot(hit));
    if ((threadIdx.x & 63) == 0 && lanes) atomicAdd(count, lanes);
}

// Expand per-view panel records into world segments, one per pixel
// (kernels/batched_geometry.py:9-39): record = source (the beam direction
// for parallel panels), pixel (0,0), u, v, column and row pitch, length
// (parallel source distance, or the cylinder radius), radial vector; mode 0
// flat cone, 1 parallel, 2 cylindrical.
__global__ __launch_bounds__(kBlock) void panel_rays_kernel(const double *__restrict__ meta,
                                                            const int *__restrict__ modes, int64_t per_view,
                                                            int cols, int64_t total, double *__restrict__ src,
                                                            double *__restrict__ end) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (int64_t)gridDim.x * kBlock) {
        const int view = (int)(i / per_view);
        const int pixel = (int)(i - (int64_t)view * per_view);
        const int row = pixel / cols, col = pixel - row * cols;
        const double *m = meta + 18 * (size_t)view;
        const double du = m[12], dv = m[13], length = m[14];
        double a[3], b[3];
        for (int k = 0; k < 3; ++k) {
            a[k] = m[k];
            b[k] = m[3 + k] + (double)col * du * m[6 + k] + (double)row * dv * m[9 + k];
        }
        if (modes[view] == 1) {
            for (int k = 0; k < 3; ++k) a[k] = b[k] - length * a[k];
        } else if (modes[view] == 2) {
            const double angle = (double)col * du / length;
            const double c = cos(angle) - 1.0, sn = sin(angle);
            for (int k = 0; k < 3; ++k)
                b[k] = m[3 + k] + c * m[15 + k] + sn * length * m[6 + k] + (double)row * dv * m[9 + k];
        }
        for (int k = 0; k < 3; ++k) {
            src[3 * i + k] = a[k];
            end[3 * i + k] = b[k];
        }
    }
}

}  // namespace dpt

// ================================================================ C ABI ====

using namespace dpt;

struct dpt_plan {
    int device = 0;
    Params base{};
    int arithmetic = 0, storage = 0;
    unsigned needs = 0;
    int64_t voxels = 0, pixels = 0;
    double *d_panels = nullptr, *d_ray_src = nullptr, *d_ray_end = nullptr;
    int *d_status = nullptr;
    int32_t *h_status = nullptr;
    double *d_partials = nullptr;
    double *d_acc = nullptr;
    float *d_alpha = nullptr;
    double *d_alpha64 = nullptr;
    unsigned long long *d_count = nullptr;
    bool cell_gauss = false;  // FP64 exact cell-Gauss integration instead of midpoints
    bool cells = false;       // FP32 sampling gathers from the plan's copy: quads (FP32) or cells (16-bit)
    int mx = 1, my = 1;       // cells along x and y
    void *d_copy = nullptr;   // the gather copy
    int vjp_vb = 1;          // views per workgroup of the VJP launches
    int forward_vb = 1;      // views per workgroup of the forward launch
    double view_gap = 0.0;   // voxels between neighbouring views of a workgroup at the grid's rim
    bool timing = false;
    double *ray_out = nullptr;             // destination of a ray-coordinate VJP (caller's buffer)
    GatherRay *d_gather_rays = nullptr;    // adjoint gather workspace, allocated at its first call
    GatherView *d_gather_views = nullptr;
    int *d_guard = nullptr;
    double *d_panel_meta = nullptr;  // panel records of a plan made from them (the gather's parallel-panel windows)
    int *d_panel_modes = nullptr;
    int image_cols = 0;              // detector columns of such a plan
    hipEvent_t ev[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    bool timed[3] = {false, false, false};
};

namespace {

thread_local std::string g_error;

int fail(int code, const std::string &msg) {
    g_error = msg;
    return code;
}

#define HIP_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return fail(DPT_E_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));    \
    } while (0)

struct DeviceGuard {
    int previous = -1;
    explicit DeviceGuard(int device) {
        if (hipGetDevice(&previous) != hipSuccess) previous = -1;
        if (previous != device) (void)hipSetDevice(device);
    }
    ~DeviceGuard() {
        int now = -1;
        if (previous >= 0 && hipGetDevice(&now) == hipSuccess && now != previous) (void)hipSetDevice(previous);
    }
};

unsigned grid_blocks(int64_t n) {
    int64_t b = (n + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    if (b > 8192) b = 8192;
    return (unsigned)b;
}

// XCD walk of a launch (tile_index): rows of tiles in turn for few views with
// rows for every XCD, else contiguous runs.  MI355X, rows against runs,
// geometric mean (worst) over 128^3, 139 x 512 x 512, 97 x 181 x 203 (FP64:
// 300^3) and panels of 128^2 to 512^2, at 1 / 3 / 5 / 7 / 10 / 15 views: split
// forward 0.72 (1.00) / 0.63 (0.89) / 0.82 (1.00) / 0.94 (1.10) / 0.87 (0.95) /
// 0.92 (0.95); FP32 forward of a lane per ray from 3 views 0.52 (0.70) / 0.73
// (0.87) / 0.92 (1.25) / 0.87 (1.14) / 0.94 (1.15), volume walk 0.96 (1.08) /
// 0.94 (1.06) / 0.97 (1.06) / 0.99 (1.07) / 0.95 (1.18) / 1.00 (1.10); FP64
// forward 1.00 (1.20) / 0.78 (1.00) / 0.78 (1.07) / 0.92 (1.26) / 0.87 (1.02) /
// 0.94 (1.08), exact pose adjoint 0.92 / 0.78 / 0.80 / 0.90 / 0.90 / 1.02 (1.31).
// Eight FP32 views keep runs, one view to an XCD: on average as fast (0.99),
// and 8 views of 257 x 301 over 139 x 512 x 512 take 0.89 ms, by rows 1.32.
// From 24 views on each run's L2 holds a part of the volume (FP64 24 x 256^2
// over 128^3: 4.7 ms, by rows 5.8).
// Row pitch 5 (mod 8) spreads a few views over the XCDs; for more views of a
// lane per ray an odd pitch, most often no blank row, keeps an XCD on
// neighbouring rows of consecutive views (7 views of 257 x 301 over 97 x 181 x
// 203: pose adjoint 0.43 ms, with pitch 5 0.62).
void set_walk(Params &P, bool wave_tiles = false) {
    const int rows = P.total_tiles / P.tiles_x;
    P.row_pitch = 0;
    P.chunk = (P.total_tiles + kXcds - 1) / kXcds;
    if (P.bundle || rows < 2 * kXcds || P.views >= 2 * kXcds) return;
    if (P.views == kXcds && !P.fp64 && !wave_tiles) return;
    const bool spread = wave_tiles || P.views < kXcds - 1;
    P.row_pitch = P.tiles_y;
    while (spread ? P.row_pitch % kXcds != 5 : P.row_pitch % 2 == 0) ++P.row_pitch;
    P.chunk = (rows / P.tiles_y * P.row_pitch + kXcds - 1) / kXcds * P.tiles_x;
}

// Tile geometry for `vb` views per workgroup (see lane_ray).
void configure_tiles(Params &P, int vb) {
    P.vb = P.bundle ? 1 : vb;
    if (P.bundle) {
        P.tile_w = kBlock;
        P.tile_h = 1;
        P.wt_x = (P.cols + 63) / 64;
        P.wt_y = 1;
    } else {
        P.tile_w = P.vb == 4 ? 8 : 16;
        P.tile_h = P.vb == 1 ? 16 : 8;
        P.wt_x = (P.cols + 7) / 8;
        P.wt_y = (P.rows + 7) / 8;
    }
    P.wt_per_view = P.wt_x * P.wt_y;
    P.tiles_x = (P.cols + P.tile_w - 1) / P.tile_w;
    P.tiles_y = (P.rows + P.tile_h - 1) / P.tile_h;
    P.tiles_per_group = P.tiles_x * P.tiles_y;
    P.total_tiles = P.tiles_per_group * ((P.views + P.vb - 1) / P.vb);
    set_walk(P);
    P.segments = 1;
    P.base_tiles = P.total_tiles;
    P.segment_samples = P.samples;
}

// Whether the FP32 forward or pose launch runs as a workgroup per wave tile
// (split kernels).  Never above 8192 waves of a lane per ray (8 per SIMD), always
// up to 512.  Between, its eightfold ray set-up and its adding wave have to be
// won back: enough samples a ray, few waves for them (6 a sample) or rays so
// far apart that every lane misses its own cells (`dense` rays per face of a
// voxel; denser lanes share the L1's lines and issue bounds the march, the pose
// march first).  Four views in a workgroup within two voxels of each other share
// cells at any density, and a workgroup per wave tile fetches them again: only
// many samples outweigh that, down to half as many on panels above 24^2 pixels
// as on smaller ones.  MI355X, a lane per ray against split: one 512^2
// view over 128^3 at S = 1: forward 14 and 36 us, pose adjoint 33 and 81;
// S = 256: 137 and 103, 157 and 177; over 139 x 512 x 512, S = 64: 109 and 79,
// 124 and 108; 2000 views of 16^2 over 32^3, S = 128: 131 and 179, 181 and 329;
// 24 views of 80^2 at one angle over 128^3, S = 64: 42 and 51, 59 and 85; S =
// 1000: 267 and 195, 454 and 328.
// Over 1458 points of views a degree or more apart on a circle, or 2000 of
// them (1 to 2000 views, S 1 to 1024, 32^3 to 256^3) the rule is 2 % off the
// better of both, split wherever it fits 9 % (forward) and 19 % (pose), a lane
// per ray 34 % and 31 %; over 540 of 4 to 32 views at one angle or within 8
// degrees it is 5 % off (forward) and 2 % (pose), split 7 % and 15 %, a lane per
// ray 19 % and 20 %.
bool split_launch(const dpt_plan *p, const Params &P, bool pose) {
    const long long waves = (long long)P.total_tiles * (kBlock / 64);
    if (waves > 8192) return false;
    if (waves <= 512) return true;
    if (P.samples < (pose ? 48 : 32)) return false;
    const bool near = P.vb == 4 && p->view_gap < 2.0;
    if (waves <= (near && P.rows * P.cols >= 24 * 24 ? 12LL : 6LL) * P.samples) return true;
    if (near) return false;
    const double side = std::cbrt((double)P.nx * P.ny * P.nz);
    const double rays_per_face = (double)P.vb * P.rows * P.cols / (side * side), dense = pose ? 4.5 : 32.0;
    return rays_per_face <= dense;
}

// Sample-range segments of the volume adjoint: a launch of few tiles (one view
// of 512^2 is 1024 workgroups, one wave per SIMD) runs each tile as `segments`
// workgroups over consecutive ranges of whole chunks (at least two chunks and
// 256 samples each), aiming at 16384 waves.  DPT_AMD_VJP_SEGMENTS overrides
// the count (1..8; not the two-chunk floor).
void configure_segments(Params &P) {
    const long long waves = (long long)P.total_tiles * (kBlock / 64);
    int g = 1;
    while (g < 8 && waves * (2 * g) <= 16384 && P.samples >= 256 * (2 * g)) g *= 2;
    if (const char *forced = std::getenv("DPT_AMD_VJP_SEGMENTS")) {
        const int v = std::atoi(forced);
        if (v >= 1 && v <= 8) g = v;
    }
    const int chunks = (P.samples + P.chunk_samples - 1) / P.chunk_samples;
    g = std::max(1, std::min(g, chunks / 2));
    if (g <= 1) return;
    const int per = (chunks + g - 1) / g;  // whole chunks per segment
    g = (chunks + per - 1) / per;
    if (g <= 1) return;
    P.segments = g;
    P.segment_samples = per * P.chunk_samples;
    P.base_tiles = P.total_tiles;
    P.total_tiles = P.base_tiles * g;
    set_walk(P);
}

// Least cosine between the central rays of two views of one group of `vb`
// consecutive views.
double least_cosine(const double *panels, int views, int rows, int cols, int vb) {
    std::vector<double> dir(3 * (size_t)views);
    for (int v = 0; v < views; ++v) {
        const double *pn = panels + 12 * (size_t)v;
        double len = 0.0;
        for (int i = 0; i < 3; ++i) {
            const double centre = pn[3 + i] + 0.5 * (cols - 1) * pn[6 + i] + 0.5 * (rows - 1) * pn[9 + i];
            dir[3 * v + i] = centre - pn[i];
            len += dir[3 * v + i] * dir[3 * v + i];
        }
        len = std::sqrt(len);
        for (int i = 0; i < 3; ++i) dir[3 * v + i] /= len;
    }
    double least = 1.0;
    for (int g = 0; g + 1 < views; g += vb)
        for (int a = g; a < g + vb && a < views; ++a)
            for (int b = a + 1; b < g + vb && b < views; ++b)
                least = std::fmin(least, dir[3 * a] * dir[3 * b] + dir[3 * a + 1] * dir[3 * b + 1] +
                                             dir[3 * a + 2] * dir[3 * b + 2]);
    return least;
}

// Views share a workgroup (and its LDS brick) only when their central rays
// differ by at most ~4 degrees: then their samples of one chunk overlap.
int choose_views_per_block(const double *panels, int views, int rows, int cols) {
    if (views < 2) return 1;
    const double cos_limit = std::cos(4.0 * 3.14159265358979323846 / 180.0);
    for (int vb : {4, 2})
        if (least_cosine(panels, views, rows, cols, vb) >= cos_limit) return vb;
    return 1;
}

// FP64 LDS brick entries per workgroup of the volume adjoint (vol_walk_kernel):
// the least multiple of 512 that holds a slab of kWalkWidth grid samples for
// half of the sampled tiles at the identity pose.  Smaller bricks leave more
// workgroups on a CU, larger ones fewer and wider slabs: the volume adjoint takes
// 62 / 68 / 78 ms at 2048 / 4096 / 8192 entries on the full scan (rule: 2048),
// 2.3 / 2.1 / 2.7 for 60 views of 256^2 over 128^3 (3072: 2.0), 17.6 / 10.2 / 5.7
// for 24 views over 256^3 (8192).  Explicit rays and panel records take 8192
// (kWalkCapMost): 24 parallel views of 256^2 over 128^3 1.76 / 1.37 / 1.31 ms, 24
// cylindrical ones 3.9 / 2.2 / 1.7; an ordered bundle of 512^2 rays over 256^3
// would do better with less, 0.74 / 0.73 / 0.90.
constexpr int kWalkCapLeast = 2048, kWalkCapMost = 8192;
int choose_walk_cap(const Params &base, const double *panels, int vb) {
    Params P = base;
    configure_tiles(P, vb);
    const int n[3] = {P.nx, P.ny, P.nz};
    const int groups = (P.views + P.vb - 1) / P.vb;
    std::vector<long long> boxes;
    for (int sg = 0; sg < std::min(groups, 4); ++sg) {
        const int first = (int)((long long)sg * groups / std::min(groups, 4)) * P.vb;
        for (int ty = 0; ty < P.tiles_y; ty += std::max(1, P.tiles_y / 8))
            for (int tx = 0; tx < P.tiles_x; tx += std::max(1, P.tiles_x / 8)) {
                // the tile's corner rays in grid coordinates
                std::vector<double> o, d;
                double mean[3] = {0.0, 0.0, 0.0};
                for (int v = first; v < std::min(first + P.vb, P.views); ++v)
                    for (int corner = 0; corner < 4; ++corner) {
                        const double *pv = panels + 12 * (size_t)v;
                        const double c = std::min(tx * P.tile_w + (corner & 1 ? P.tile_w - 1 : 0), P.cols - 1);
                        const double r = std::min(ty * P.tile_h + (corner & 2 ? P.tile_h - 1 : 0), P.rows - 1);
                        for (int a = 0; a < 3; ++a) {
                            double oa = 0.0, da = 0.0;
                            for (int b = 0; b < 3; ++b) {
                                oa += P.g[3 * a + b] * (pv[b] - P.go[b]);
                                da += P.g[3 * a + b] * (pv[3 + b] + c * pv[6 + b] + r * pv[9 + b] - pv[b]);
                            }
                            o.push_back(oa);
                            d.push_back(da);
                            mean[a] += da;
                        }
                    }
                int A = 0;
                for (int a = 1; a < 3; ++a)
                    if (std::fabs(mean[a]) > std::fabs(mean[A])) A = a;
                for (int quarter = 1; quarter < 4; ++quarter) {
                    const double s0 = std::floor(quarter * (n[A] - 1) / 4.0), s1 = std::min(s0 + kWalkWidth, n[A] - 1.0);
                    long long volume = (long long)(s1 - s0) + 1;
                    bool meets = true;
                    for (int a = 0; a < 3; ++a) {
                        if (a == A) continue;
                        double lo = 1e300, hi = -1e300;
                        for (size_t q = 0; q < o.size(); q += 3)
                            for (double s : {s0, s1}) {
                                const double x = o[q + a] + (s - o[q + A]) / d[q + A] * d[q + a];
                                lo = std::min(lo, x);
                                hi = std::max(hi, x);
                            }
                        if (!(hi >= -0.5 && lo <= n[a] - 0.5)) {  // false for NaN
                            meets = false;
                            break;
                        }
                        volume *= (long long)(std::min(hi, n[a] - 1.0) - std::max(lo, 0.0)) + 2;
                    }
                    if (meets) boxes.push_back(volume);
                }
            }
    }
    if (boxes.empty()) return kWalkCapLeast;
    std::sort(boxes.begin(), boxes.end());
    const long long box = std::min<long long>(boxes[boxes.size() / 2], kWalkCapMost);
    return std::min(std::max((int)((box + 511) / 512 * 512), kWalkCapLeast), kWalkCapMost);
}

Params launch_params(const dpt_plan *p, const double *poses) {
    Params P = p->base;
    P.poses = poses;
    P.status = p->d_status;
    return P;
}

unsigned tile_grid(const Params &P) { return (unsigned)(P.chunk * kXcds); }
// One workgroup per wave tile (split_tile).
Params split_params(Params P) {
    P.tiles_x = P.wt_x;
    P.tiles_y = P.wt_y;
    P.total_tiles = P.views * P.wt_per_view;
    set_walk(P, true);
    return P;
}

// Launch parameters of a gather from the plan's copy (quads or cells).
Params copy_params(const dpt_plan *p, Params P) {
    P.ix = p->mx;
    P.iy = p->my;
    P.qz = P.nz > 1 ? p->mx * p->my : 0;
    return P;
}

template <typename T>
int launch_forward(dpt_plan *p, const Params &P, const void *field, void *out, bool cells, hipStream_t s) {
    const T *f = static_cast<const T *>(field);
    const dim3 grid(tile_grid(P)), block(kBlock);
    if (p->arithmetic == DPT_ARITH_FP32) {
        float *o = static_cast<float *>(out);
        constexpr bool HALF = !std::is_same<T, float>::value;
        if (split_launch(p, P, false)) {
            const Params Q = split_params(P);
            const dim3 tiles(tile_grid(Q)), lanes(64 * kSplitWaves);
            if (cells)
                hipLaunchKernelGGL((forward32_split_kernel<T, HALF, kGatherCopy<T>>), tiles, lanes, 0, s,
                                   copy_params(p, Q), static_cast<const T *>(p->d_copy), o);
            else if (P.nx > 1)
                hipLaunchKernelGGL((forward32_split_kernel<T, HALF, kLayoutPair>), tiles, lanes, 0, s, Q, f, o);
            else
                hipLaunchKernelGGL((forward32_split_kernel<T, HALF, kLayoutScalar>), tiles, lanes, 0, s, Q, f, o);
            HIP_TRY(hipGetLastError());
            return DPT_OK;
        }
        if (cells)
            hipLaunchKernelGGL((forward32_kernel<T, HALF, kGatherCopy<T>>), grid, block, 0, s, copy_params(p, P),
                               static_cast<const T *>(p->d_copy), o);
        else if (P.nx > 1)
            hipLaunchKernelGGL((forward32_kernel<T, HALF, kLayoutPair>), grid, block, 0, s, P, f, o);
        else
            hipLaunchKernelGGL((forward32_kernel<T, HALF, kLayoutScalar>), grid, block, 0, s, P, f, o);
    } else if (p->cell_gauss) {
        hipLaunchKernelGGL((forward_gauss_kernel<T>), grid, block, 0, s, P, f, static_cast<double *>(out));
    } else {
        hipLaunchKernelGGL((forward64_kernel<T>), grid, block, 0, s, P, f, static_cast<double *>(out));
    }
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

// Pose partials, or the caller's per-ray buffer for ray coordinates and
// per-ray tangents
template <int C>
double *pose_destination(dpt_plan *p) {
    return (C == kRayCoordinates || C == kRayTangent) ? p->ray_out : p->d_partials;
}

template <typename T, int C, int LAYOUT>
void launch_vjp32(dpt_plan *p, const Params &P, const T *f, const float *sd, hipStream_t s) {
    constexpr bool HALF = !std::is_same<T, float>::value;
    double *partials = pose_destination<C>(p);
    if (split_launch(p, P, true)) {
        const Params Q = split_params(P);
        hipLaunchKernelGGL((vjp32_split_kernel<T, C, HALF, LAYOUT>), dim3(tile_grid(Q)), dim3(64 * kSplitWaves), 0, s,
                           Q, f, sd, partials);
    } else {
        hipLaunchKernelGGL((vjp32_kernel<T, C, HALF, LAYOUT>), dim3(tile_grid(P)), dim3(kBlock), 0, s, P, f, sd,
                           partials);
    }
}

template <typename T, int C>
int launch_vjp_c(dpt_plan *p, const Params &P, const void *field, const void *seeds, bool cells,
                 hipStream_t s) {
    const T *f = static_cast<const T *>(field);
    const dim3 grid(tile_grid(P)), block(kBlock);
    double *partials = pose_destination<C>(p);
    if (p->arithmetic == DPT_ARITH_FP32) {
        const float *sd = static_cast<const float *>(seeds);
        if (cells && P.nx > 1)
            launch_vjp32<T, C, kGatherCopy<T>>(p, copy_params(p, P), static_cast<const T *>(p->d_copy), sd, s);
        else if (P.nx > 1)
            launch_vjp32<T, C, kLayoutPair>(p, P, f, sd, s);
        else
            launch_vjp32<T, C, kLayoutScalar>(p, P, f, sd, s);
    } else if (p->cell_gauss) {
        hipLaunchKernelGGL((vjp_gauss_kernel<T, C>), grid, block, 0, s, P, f, static_cast<const double *>(seeds),
                           partials);
    } else {
        hipLaunchKernelGGL((vjp64_kernel<T, C>), grid, block, 0, s, P, f, static_cast<const double *>(seeds),
                           partials);
    }
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

template <typename T>
int launch_vjp(dpt_plan *p, const Params &P, const void *field, const void *seeds, int components, bool cells,
               hipStream_t s) {
    if (components == kRayCoordinates) return launch_vjp_c<T, kRayCoordinates>(p, P, field, seeds, cells, s);
    if (components == kRayTangent) return launch_vjp_c<T, kRayTangent>(p, P, field, seeds, cells, s);
    if (components == 6) return launch_vjp_c<T, 6>(p, P, field, seeds, cells, s);
    return launch_vjp_c<T, 12>(p, P, field, seeds, cells, s);
}

int launch_walk(dpt_plan *p, const Params &P, const void *seeds, hipStream_t s) {
    const dim3 grid(tile_grid(P)), block(kBlock);
    const size_t lds = (size_t)P.walk_cap * sizeof(double);
    const bool biased = std::max(P.nx, std::max(P.ny, P.nz)) <= kWalkMaxAxis && P.samples <= (1 << 22);
    if (p->cell_gauss) {
        hipLaunchKernelGGL((vol_walk_kernel<double, double, true>), grid, block, lds, s, P,
                           static_cast<const double *>(seeds), p->d_acc);
        hipLaunchKernelGGL(gauss_scatter_kernel, grid, block, 0, s, P, static_cast<const double *>(seeds), p->d_acc);
    } else if (p->arithmetic == DPT_ARITH_FP64)
        hipLaunchKernelGGL((vol_walk_kernel<double, double>), grid, block, lds, s, P,
                           static_cast<const double *>(seeds), p->d_acc);
    else if (biased)
        hipLaunchKernelGGL((vol_walk_kernel<float, float>), grid, block, lds, s, P,
                           static_cast<const float *>(seeds), p->d_acc);
    else
        hipLaunchKernelGGL((vol_walk_kernel<float, double>), grid, block, lds, s, P,
                           static_cast<const float *>(seeds), p->d_acc);
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

int launch_cells(const void *src, void *dst, int nx, int ny, int nz, int storage, hipStream_t s) {
    const int mx = nx > 1 ? nx - 1 : 1, my = ny > 1 ? ny - 1 : 1, mz = nz > 1 ? nz - 1 : 1;
    const int64_t cells = (int64_t)mx * my * mz;
    if (cells == 0) return DPT_OK;
    if (storage == DPT_STORE_F32)
        hipLaunchKernelGGL(cells_kernel<uint32_t>, dim3(grid_blocks(cells)), dim3(kBlock), 0, s,
                           static_cast<const uint32_t *>(src), static_cast<uint32_t *>(dst), nx, ny, nz, mx, my,
                           (int)cells);
    else
        hipLaunchKernelGGL(cells_kernel<uint16_t>, dim3(grid_blocks(cells)), dim3(kBlock), 0, s,
                           static_cast<const uint16_t *>(src), static_cast<uint16_t *>(dst), nx, ny, nz, mx, my,
                           (int)cells);
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

// Rebuild the plan's gather copy of the field.
int refresh_copy(dpt_plan *p, const void *field, hipStream_t s) {
    const Params &P = p->base;
    if (p->storage != DPT_STORE_F32) return launch_cells(field, p->d_copy, P.nx, P.ny, P.nz, p->storage, s);
    const int64_t quads = (int64_t)p->mx * p->my * P.nz;
    hipLaunchKernelGGL(quads_kernel, dim3(grid_blocks(quads)), dim3(kBlock), 0, s, static_cast<const uint32_t *>(field),
                       static_cast<Quad *>(p->d_copy), P.nx, P.ny, p->mx, p->my, quads);
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

void timer_begin(dpt_plan *p, int kind, hipStream_t s) {
    if (p->timing) (void)hipEventRecord(p->ev[2 * kind], s);
}
void timer_end(dpt_plan *p, int kind, hipStream_t s) {
    if (p->timing) {
        (void)hipEventRecord(p->ev[2 * kind + 1], s);
        p->timed[kind] = true;
    }
}

}  // namespace

extern "C" {

int32_t dpt_abi_version(void) { return DPT_ABI_VERSION; }

const char *dpt_last_error(void) { return g_error.c_str(); }

int dpt_plan_destroy(dpt_plan *p) {
    if (p == nullptr) return DPT_OK;
    DeviceGuard guard(p->device);
    (void)hipFree(p->d_panels);
    (void)hipFree(p->d_ray_src);
    (void)hipFree(p->d_ray_end);
    (void)hipFree(p->d_status);
    (void)hipFree(p->d_partials);
    (void)hipFree(p->d_acc);
    (void)hipFree(p->d_alpha);
    (void)hipFree(p->d_alpha64);
    (void)hipFree(p->d_copy);
    (void)hipFree(p->d_count);
    (void)hipFree(p->d_gather_rays);
    (void)hipFree(p->d_gather_views);
    (void)hipFree(p->d_guard);
    (void)hipFree(p->d_panel_meta);
    (void)hipFree(p->d_panel_modes);
    if (p->h_status) (void)hipHostFree(p->h_status);
    for (auto &e : p->ev)
        if (e) (void)hipEventDestroy(e);
    delete p;
    return DPT_OK;
}

}  // extern "C"

namespace {

// Shared body of dpt_plan_create (panels or host rays) and
// dpt_plan_create_panels (panel records expanded into rays on the device;
// the plan is then a bundle of rows*cols rays per view).
int plan_create(const dpt_grid_desc *grid, int32_t views, int32_t rows, int32_t cols, const double *panels,
                const double *ray_sources, const double *ray_endpoints, const double *panel_meta,
                const int32_t *panel_modes, int32_t samples, int32_t arithmetic, int32_t storage, uint32_t needs,
                int32_t device, dpt_plan **out) {
    if (out == nullptr || grid == nullptr) return fail(DPT_E_INVALID, "grid and out are required");
    const bool generated = panel_meta != nullptr;
    int image_cols = cols;  // columns of one detector row (the bundle below is rows*cols rays per view)
    if (generated) {
        if (panel_modes == nullptr || panels != nullptr || ray_sources != nullptr || ray_endpoints != nullptr)
            return fail(DPT_E_INVALID, "panel records take modes and no panels or rays");
        if (views < 1 || rows < 1 || cols < 1) return fail(DPT_E_INVALID, "views, rows and cols must be positive");
        if ((int64_t)rows * cols > INT32_MAX) return fail(DPT_E_INVALID, "image exceeds signed 32-bit indexing");
        for (int v = 0; v < views; ++v) {
            if (panel_modes[v] < 0 || panel_modes[v] > 2) return fail(DPT_E_INVALID, "panel mode must be 0, 1 or 2");
            for (int k = 0; k < 18; ++k)
                if (!std::isfinite(panel_meta[18 * (size_t)v + k]))
                    return fail(DPT_E_INVALID, "panel records must be finite");
            if (panel_modes[v] != 0 && !(panel_meta[18 * (size_t)v + 14] > 0.0))
                return fail(DPT_E_INVALID, "parallel length / cylinder radius must be positive");
        }
        image_cols = cols;
        cols = rows * cols;
        rows = 1;
    }
    *out = nullptr;
    if (grid->nx < 1 || grid->ny < 1 || grid->nz < 1)
        return fail(DPT_E_INVALID, "grid counts must be positive");
    const int64_t voxels = (int64_t)grid->nx * grid->ny * grid->nz;
    if (voxels > INT32_MAX) return fail(DPT_E_INVALID, "grid exceeds signed 32-bit indexing");
    if ((long long)grid->ny * grid->nz > kMaxSliceProduct)
        return fail(DPT_E_INVALID, "grid ny * nz exceeds 2^24 (24-bit cell index arithmetic)");
    if (views < 1 || rows < 1 || cols < 1) return fail(DPT_E_INVALID, "views, rows and cols must be positive");
    const int64_t pixels = (int64_t)views * rows * cols;
    if (pixels > INT32_MAX) return fail(DPT_E_INVALID, "image exceeds signed 32-bit indexing");
    if (samples < 1) return fail(DPT_E_INVALID, "samples must be positive");
    if (arithmetic != DPT_ARITH_FP32 && arithmetic != DPT_ARITH_FP64)
        return fail(DPT_E_INVALID, "arithmetic must be DPT_ARITH_FP32 or DPT_ARITH_FP64");
    if (storage != DPT_STORE_F32 && storage != DPT_STORE_BF16 && storage != DPT_STORE_F16)
        return fail(DPT_E_INVALID, "storage must be DPT_STORE_F32, DPT_STORE_BF16 or DPT_STORE_F16");
    if (arithmetic == DPT_ARITH_FP32 && (grid->nx > (1 << 24) || grid->ny > (1 << 24) || grid->nz > (1 << 24)))
        return fail(DPT_E_INVALID, "FP32 sampling requires grid axis counts at most 2**24");
    if (!generated && panels == nullptr && (ray_sources == nullptr || ray_endpoints == nullptr))
        return fail(DPT_E_INVALID, "supply panels or explicit ray sources and endpoints");
    if (panels == nullptr && rows != 1) return fail(DPT_E_INVALID, "explicit rays require rows == 1");
    if ((needs & DPT_CELL_GAUSS) && arithmetic != DPT_ARITH_FP64)
        return fail(DPT_E_INVALID, "cell-Gauss integration requires DPT_ARITH_FP64");
    for (int i = 0; i < 9; ++i)
        if (!std::isfinite(grid->object_to_grid[i])) return fail(DPT_E_INVALID, "object_to_grid must be finite");

    DeviceGuard guard(device);
    dpt_plan *p = new dpt_plan();
    p->device = device;
    p->arithmetic = arithmetic;
    p->storage = storage;
    p->needs = needs;
    p->cell_gauss = (needs & DPT_CELL_GAUSS) != 0;
    p->voxels = voxels;
    p->pixels = pixels;
    Params &P = p->base;
    P.nx = grid->nx;
    P.ny = grid->ny;
    P.nz = grid->nz;
    P.ix = grid->nx;
    P.iy = grid->ny;
    P.sx = grid->nx > 1 ? 1 : 0;
    P.sy = grid->ny > 1 ? grid->nx : 0;
    P.sz = grid->nz > 1 ? grid->nx * grid->ny : 0;
    P.hx = (float)grid->nx - 0.5f;
    P.hy = (float)grid->ny - 0.5f;
    P.hz = (float)grid->nz - 0.5f;
    P.cx = (float)(grid->nx - 1);
    P.cy = (float)(grid->ny - 1);
    P.cz = (float)(grid->nz - 1);
    P.capx = grid->nx - 2 > 0 ? grid->nx - 2 : 0;
    P.capy = grid->ny - 2 > 0 ? grid->ny - 2 : 0;
    P.capz = grid->nz - 2 > 0 ? grid->nz - 2 : 0;
    std::memcpy(P.g, grid->object_to_grid, sizeof P.g);
    std::memcpy(P.go, grid->grid_origin, sizeof P.go);
    P.views = views;
    P.rows = rows;
    P.cols = cols;
    P.samples = samples;
    P.bundle = panels == nullptr ? 1 : 0;
    P.fp64 = arithmetic == DPT_ARITH_FP64;
    configure_tiles(P, 1);
    P.chunk_samples = chunk_samples(samples, grid->nx, grid->ny, grid->nz);
    if (const char *chunk = std::getenv("DPT_AMD_CHUNK")) {
        const int forced = std::atoi(chunk);
        if (forced >= 1 && forced <= 1024) P.chunk_samples = forced;
    }
    P.gauss_chunks = gauss_chunks(grid->nx, grid->ny, grid->nz);
    if (const char *chunks = std::getenv("DPT_AMD_GAUSS_CHUNKS")) {
        const int forced = std::atoi(chunks);
        if (forced >= 1 && forced <= 256) P.gauss_chunks = forced;
    }
    P.walk_cap = P.bundle ? kWalkCapMost : choose_walk_cap(P, panels, choose_views_per_block(panels, views, rows, cols));
    if (const char *cap = std::getenv("DPT_AMD_BRICK_CAP")) {
        const int forced = std::atoi(cap);
        if (forced >= 512 && forced <= 8192) P.walk_cap = forced;
    }
    p->vjp_vb = P.bundle ? 1 : choose_views_per_block(panels, views, rows, cols);
    if (const char *vb = std::getenv("DPT_AMD_VIEWS_PER_BLOCK")) {
        const int forced = std::atoi(vb);
        if (!P.bundle && (forced == 1 || forced == 2 || forced == 4)) p->vjp_vb = forced;
    }
    p->forward_vb = p->vjp_vb;
    if (!P.bundle && views > 1) {
        const double n[3] = {(double)grid->nx, (double)grid->ny, (double)grid->nz};
        const double angle = std::acos(std::fmin(1.0, least_cosine(panels, views, rows, cols, 2)));
        p->view_gap = 0.5 * angle * std::sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    }
    if (const char *vb = std::getenv("DPT_AMD_FORWARD_VIEWS_PER_BLOCK")) {
        const int forced = std::atoi(vb);
        if (!P.bundle && (forced == 1 || forced == 2 || forced == 4)) p->forward_vb = forced;
    }
    p->cells = (needs & DPT_GATHER_CELLS) != 0;
    if (const char *gather = std::getenv("DPT_AMD_GATHER")) {
        if (std::strcmp(gather, "cells") == 0) p->cells = true;
        if (std::strcmp(gather, "linear") == 0) p->cells = false;
    }
    p->cells = p->cells && arithmetic == DPT_ARITH_FP32;
    p->mx = grid->nx > 1 ? grid->nx - 1 : 1;
    p->my = grid->ny > 1 ? grid->ny - 1 : 1;
    const int64_t planes = (int64_t)p->mx * p->my;

    auto cleanup = [&](int code, const std::string &msg) {
        dpt_plan_destroy(p);
        return fail(code, msg);
    };
#define ALLOC(ptr, bytes)                                                                   \
    do {                                                                                    \
        if (hipMalloc((void **)&(ptr), (bytes)) != hipSuccess)                              \
            return cleanup(DPT_E_MEMORY, "hipMalloc failed for " #ptr);                     \
    } while (0)

    if (!P.bundle) {
        ALLOC(p->d_panels, sizeof(double) * 12 * views);
        if (hipMemcpy(p->d_panels, panels, sizeof(double) * 12 * views, hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(DPT_E_DEVICE, "copy of panels failed");
    } else {
        const size_t bytes = sizeof(double) * 3 * (size_t)pixels;
        ALLOC(p->d_ray_src, bytes);
        ALLOC(p->d_ray_end, bytes);
        if (generated) {
            ALLOC(p->d_panel_meta, sizeof(double) * 18 * views);
            ALLOC(p->d_panel_modes, sizeof(int) * views);
            p->image_cols = image_cols;
            bool ok = hipMemcpy(p->d_panel_meta, panel_meta, sizeof(double) * 18 * views, hipMemcpyHostToDevice) ==
                          hipSuccess &&
                      hipMemcpy(p->d_panel_modes, panel_modes, sizeof(int) * views, hipMemcpyHostToDevice) ==
                          hipSuccess;
            if (ok) {
                hipLaunchKernelGGL(panel_rays_kernel, dim3(grid_blocks(pixels)), dim3(kBlock), 0, 0, p->d_panel_meta,
                                   p->d_panel_modes, (int64_t)cols, image_cols, pixels, p->d_ray_src, p->d_ray_end);
                ok = hipGetLastError() == hipSuccess && hipDeviceSynchronize() == hipSuccess;
            }
            if (!ok) return cleanup(DPT_E_DEVICE, "panel ray generation failed");
        } else if (hipMemcpy(p->d_ray_src, ray_sources, bytes, hipMemcpyHostToDevice) != hipSuccess ||
                   hipMemcpy(p->d_ray_end, ray_endpoints, bytes, hipMemcpyHostToDevice) != hipSuccess) {
            return cleanup(DPT_E_DEVICE, "copy of rays failed");
        }
    }
    P.panels = p->d_panels;
    P.ray_src = p->d_ray_src;
    P.ray_end = p->d_ray_end;
    ALLOC(p->d_status, sizeof(int) * views);
    if (hipMemset(p->d_status, 0, sizeof(int) * views) != hipSuccess)
        return cleanup(DPT_E_DEVICE, "status clear failed");
    if (hipHostMalloc((void **)&p->h_status, sizeof(int32_t) * views, hipHostMallocDefault) != hipSuccess)
        return cleanup(DPT_E_MEMORY, "pinned status allocation failed");
    if (needs & DPT_POSE) ALLOC(p->d_partials, sizeof(double) * kMaxComponents * (size_t)P.wt_per_view * views);
    if (needs & DPT_VOLUME) ALLOC(p->d_acc, sizeof(double) * (size_t)voxels);
    if (p->cells) ALLOC(p->d_copy, storage == DPT_STORE_F32 ? 16 * (size_t)(planes * grid->nz)
                                                        : 16 * (size_t)(planes * std::max(grid->nz - 1, 1)));
    ALLOC(p->d_count, sizeof(unsigned long long));
    ALLOC(p->d_alpha, sizeof(float) * sample_table_entries(samples));
    {
        std::vector<float> alpha(sample_table_entries(samples));
        fill_alpha_table(alpha.data(), samples);
        if (hipMemcpy(p->d_alpha, alpha.data(), sizeof(float) * alpha.size(), hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(DPT_E_DEVICE, "copy of the sample fractions failed");
    }
    P.alpha = p->d_alpha;
    if (arithmetic == DPT_ARITH_FP64) {
        std::vector<double> alpha(2 * (size_t)samples);
        for (int k = 0; k < samples; ++k) {
            alpha[k] = ((double)k + 0.5) / (double)samples;
            alpha[(size_t)samples + k] = 1.0 - alpha[k];
        }
        ALLOC(p->d_alpha64, sizeof(double) * alpha.size());
        if (hipMemcpy(p->d_alpha64, alpha.data(), sizeof(double) * alpha.size(), hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(DPT_E_DEVICE, "copy of the sample fractions failed");
    }
    P.alpha64 = p->d_alpha64;
    for (auto &e : p->ev)
        if (hipEventCreate(&e) != hipSuccess) return cleanup(DPT_E_DEVICE, "event creation failed");
#undef ALLOC
    *out = p;
    return DPT_OK;
}

}  // namespace

extern "C" {

int dpt_plan_create(const dpt_grid_desc *grid, int32_t views, int32_t rows, int32_t cols, const double *panels,
                    const double *ray_sources, const double *ray_endpoints, int32_t samples, int32_t arithmetic,
                    int32_t storage, uint32_t needs, int32_t device, dpt_plan **out) {
    return plan_create(grid, views, rows, cols, panels, ray_sources, ray_endpoints, nullptr, nullptr, samples,
                       arithmetic, storage, needs, device, out);
}

int dpt_plan_create_panels(const dpt_grid_desc *grid, int32_t views, int32_t rows, int32_t cols,
                           const double *panel_records, const int32_t *panel_modes, int32_t samples,
                           int32_t arithmetic, int32_t storage, uint32_t needs, int32_t device, dpt_plan **out) {
    if (panel_records == nullptr) return fail(DPT_E_INVALID, "panel records are required");
    return plan_create(grid, views, rows, cols, nullptr, nullptr, nullptr, panel_records, panel_modes, samples,
                       arithmetic, storage, needs, device, out);
}

int dpt_forward(dpt_plan *p, const void *field, const double *poses, void *out, void *stream) {
    if (p == nullptr || field == nullptr || poses == nullptr || out == nullptr)
        return fail(DPT_E_INVALID, "plan, field, poses and out are required");
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    Params P = launch_params(p, poses);
    configure_tiles(P, p->forward_vb);
    switch (p->storage) {
    case DPT_STORE_F32:
        hipLaunchKernelGGL(check_field_kernel<float>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                           static_cast<const float *>(field), p->voxels, p->d_status);
        break;
    case DPT_STORE_BF16:
        hipLaunchKernelGGL(check_field_kernel<__hip_bfloat16>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                           static_cast<const __hip_bfloat16 *>(field), p->voxels, p->d_status);
        break;
    default:
        hipLaunchKernelGGL(check_field_kernel<__half>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                           static_cast<const __half *>(field), p->voxels, p->d_status);
    }
    hipLaunchKernelGGL(check_poses_kernel, dim3((P.views + 63) / 64), dim3(64), 0, s, poses, P.views, p->d_status);
    HIP_TRY(hipGetLastError());
    if (p->cells) {
        const int rc = refresh_copy(p, field, s);
        if (rc != DPT_OK) return rc;
    }
    timer_begin(p, 0, s);
    int rc;
    if (p->storage == DPT_STORE_F32)
        rc = launch_forward<float>(p, P, field, out, p->cells, s);
    else if (p->storage == DPT_STORE_BF16)
        rc = launch_forward<__hip_bfloat16>(p, P, field, out, p->cells, s);
    else
        rc = launch_forward<__half>(p, P, field, out, p->cells, s);
    timer_end(p, 0, s);
    return rc;
}

int dpt_vjp(dpt_plan *p, const void *field, const double *poses, const void *cotangent, void *grad_field,
            double *grad_pose, uint32_t flags, void *stream) {
    if (p == nullptr || field == nullptr || poses == nullptr || cotangent == nullptr)
        return fail(DPT_E_INVALID, "plan, field, poses and cotangent are required");
    const bool vol = flags & DPT_VOLUME, pose = flags & DPT_POSE;
    if (!vol && !pose) return fail(DPT_E_INVALID, "request at least one projection gradient");
    if (vol && (grad_field == nullptr || !(p->needs & DPT_VOLUME)))
        return fail(DPT_E_INVALID, "volume gradient requested without a destination or plan support");
    if (pose && (grad_pose == nullptr || !(p->needs & DPT_POSE)))
        return fail(DPT_E_INVALID, "pose gradient requested without a destination or plan support");
    if (flags & ~(uint32_t)(DPT_VOLUME | DPT_POSE | DPT_POSE_TANGENT | DPT_ACCUMULATE | DPT_NO_CHECKS |
                            DPT_VOLUME_FP64))
        return fail(DPT_E_INVALID, "unknown VJP flags");
    const bool vol64 = vol && (flags & DPT_VOLUME_FP64);
    const int components = (flags & DPT_POSE_TANGENT) ? 6 : 12;
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    Params P = launch_params(p, poses);
    P.volume_f64 = vol64 ? 1 : 0;
    configure_tiles(P, p->vjp_vb);
    const Params whole = P;
    if (vol && !p->cell_gauss) configure_segments(P);  // of the volume adjoint
    if (!(flags & DPT_NO_CHECKS)) {
        switch (p->storage) {
        case DPT_STORE_F32:
            hipLaunchKernelGGL(check_field_kernel<float>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                               static_cast<const float *>(field), p->voxels, p->d_status);
            break;
        case DPT_STORE_BF16:
            hipLaunchKernelGGL(check_field_kernel<__hip_bfloat16>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0,
                               s, static_cast<const __hip_bfloat16 *>(field), p->voxels, p->d_status);
            break;
        default:
            hipLaunchKernelGGL(check_field_kernel<__half>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                               static_cast<const __half *>(field), p->voxels, p->d_status);
        }
        hipLaunchKernelGGL(check_poses_kernel, dim3((P.views + 63) / 64), dim3(64), 0, s, poses, P.views,
                           p->d_status);
        if (p->arithmetic == DPT_ARITH_FP32)
            hipLaunchKernelGGL(check_finite_kernel<float>, dim3(grid_blocks(p->pixels)), dim3(kBlock), 0, s,
                               static_cast<const float *>(cotangent), p->pixels, p->d_status);
        else
            hipLaunchKernelGGL(check_finite_kernel<double>, dim3(grid_blocks(p->pixels)), dim3(kBlock), 0, s,
                               static_cast<const double *>(cotangent), p->pixels, p->d_status);
    }
    if (vol)
        hipLaunchKernelGGL(fill_f64_kernel, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s, p->d_acc, p->voxels);
    HIP_TRY(hipGetLastError());
    // the cell copy is rebuilt at every call: the field of this VJP may differ
    // from the last forward's
    const bool cells = p->cells && pose;
    if (cells) {
        const int rc = refresh_copy(p, field, s);
        if (rc != DPT_OK) return rc;
    }
    timer_begin(p, 1, s);
    int rc = DPT_OK;
    if (vol) rc = launch_walk(p, P, cotangent, s);
    if (rc == DPT_OK && pose) {
        if (p->storage == DPT_STORE_F32)
            rc = launch_vjp<float>(p, whole, field, cotangent, components, cells, s);
        else if (p->storage == DPT_STORE_BF16)
            rc = launch_vjp<__hip_bfloat16>(p, whole, field, cotangent, components, cells, s);
        else
            rc = launch_vjp<__half>(p, whole, field, cotangent, components, cells, s);
    }
    timer_end(p, 1, s);
    if (rc != DPT_OK) return rc;
    const int accumulate = (flags & DPT_ACCUMULATE) ? 1 : 0;
    if (pose) {
        if (components == 6)
            hipLaunchKernelGGL(pose_reduce_kernel<6>, dim3(P.views), dim3(kBlock), 0, s, p->d_partials,
                               P.wt_per_view, grad_pose, accumulate, p->d_status);
        else
            hipLaunchKernelGGL(pose_reduce_kernel<12>, dim3(P.views), dim3(kBlock), 0, s, p->d_partials,
                               P.wt_per_view, grad_pose, accumulate, p->d_status);
    }
    if (vol64)
        hipLaunchKernelGGL(finish_volume_kernel<double>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                           p->d_acc, static_cast<double *>(grad_field), p->voxels, accumulate, p->d_status);
    else if (vol)
        hipLaunchKernelGGL(finish_volume_kernel<float>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                           p->d_acc, static_cast<float *>(grad_field), p->voxels, accumulate, p->d_status);
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

}  // extern "C"

namespace {

// Per-ray VJP outputs (6 FP64 values per ray into the caller's buffer):
// mode kRayCoordinates (world source / endpoint derivatives) or kRayTangent
// (6-DoF local-right pose tangent).
int per_ray_vjp(dpt_plan *p, const void *field, const double *poses, const void *cotangent, double *out_rays,
                int mode, uint32_t flags, void *stream) {
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    Params P = launch_params(p, poses);
    configure_tiles(P, p->vjp_vb);
    if (!(flags & DPT_NO_CHECKS)) {
        switch (p->storage) {
        case DPT_STORE_F32:
            hipLaunchKernelGGL(check_field_kernel<float>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                               static_cast<const float *>(field), p->voxels, p->d_status);
            break;
        case DPT_STORE_BF16:
            hipLaunchKernelGGL(check_field_kernel<__hip_bfloat16>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0,
                               s, static_cast<const __hip_bfloat16 *>(field), p->voxels, p->d_status);
            break;
        default:
            hipLaunchKernelGGL(check_field_kernel<__half>, dim3(grid_blocks(p->voxels)), dim3(kBlock), 0, s,
                               static_cast<const __half *>(field), p->voxels, p->d_status);
        }
        hipLaunchKernelGGL(check_poses_kernel, dim3((P.views + 63) / 64), dim3(64), 0, s, poses, P.views,
                           p->d_status);
        if (p->arithmetic == DPT_ARITH_FP32)
            hipLaunchKernelGGL(check_finite_kernel<float>, dim3(grid_blocks(p->pixels)), dim3(kBlock), 0, s,
                               static_cast<const float *>(cotangent), p->pixels, p->d_status);
        else
            hipLaunchKernelGGL(check_finite_kernel<double>, dim3(grid_blocks(p->pixels)), dim3(kBlock), 0, s,
                               static_cast<const double *>(cotangent), p->pixels, p->d_status);
    }
    HIP_TRY(hipGetLastError());
    if (p->cells) {
        const int rc = refresh_copy(p, field, s);
        if (rc != DPT_OK) return rc;
    }
    p->ray_out = out_rays;
    int rc;
    if (p->storage == DPT_STORE_F32)
        rc = launch_vjp<float>(p, P, field, cotangent, mode, p->cells, s);
    else if (p->storage == DPT_STORE_BF16)
        rc = launch_vjp<__hip_bfloat16>(p, P, field, cotangent, mode, p->cells, s);
    else
        rc = launch_vjp<__half>(p, P, field, cotangent, mode, p->cells, s);
    p->ray_out = nullptr;
    return rc;
}

}  // namespace

extern "C" {

int dpt_ray_vjp(dpt_plan *p, const void *field, const double *poses, const void *cotangent, double *out_rays,
                uint32_t flags, void *stream) {
    if (p == nullptr || field == nullptr || poses == nullptr || cotangent == nullptr || out_rays == nullptr)
        return fail(DPT_E_INVALID, "plan, field, poses, cotangent and out_rays are required");
    if (flags & ~(uint32_t)DPT_NO_CHECKS) return fail(DPT_E_INVALID, "ray-coordinate VJP flags are DPT_NO_CHECKS");
    return per_ray_vjp(p, field, poses, cotangent, out_rays, kRayCoordinates, flags, stream);
}

int dpt_pose_sensitivities(dpt_plan *p, const void *field, const double *poses, const void *cotangent,
                           double *out_jacobian, uint32_t flags, void *stream) {
    if (p == nullptr || field == nullptr || poses == nullptr || cotangent == nullptr || out_jacobian == nullptr)
        return fail(DPT_E_INVALID, "plan, field, poses, cotangent and out_jacobian are required");
    if (flags & ~(uint32_t)DPT_NO_CHECKS) return fail(DPT_E_INVALID, "pose sensitivity flags are DPT_NO_CHECKS");
    return per_ray_vjp(p, field, poses, cotangent, out_jacobian, kRayTangent, flags, stream);
}

}  // extern "C"

namespace {

// Per-view sum of ray-coordinate derivatives contracted with the view's
// acquisition Jacobian: out[v, k] = sum_p sum_j rays[v, p, j] * J[v, k, j]
// (kernels/batched_projection.py:15-89, fixed-order FP64 tree per view).
__global__ __launch_bounds__(kBlock) void rays_reduce_kernel(const double *__restrict__ rays,
                                                             const double *__restrict__ jacobians, int64_t pixels,
                                                             int components, double *out, int accumulate,
                                                             int *status) {
    const int view = blockIdx.x;
    __shared__ double red[kBlock];
    const double *base = rays + (size_t)view * pixels * 6;
    for (int k = 0; k < components; ++k) {
        const double *jac = jacobians + ((size_t)view * components + k) * 6;
        double v = 0.0;
        for (int64_t i = threadIdx.x; i < pixels; i += kBlock) {
            const double *g = base + 6 * (size_t)i;
            v += g[0] * jac[0] + g[1] * jac[1] + g[2] * jac[2] + g[3] * jac[3] + g[4] * jac[4] + g[5] * jac[5];
        }
        red[threadIdx.x] = v;
        __syncthreads();
        for (int stride = kBlock / 2; stride > 0; stride >>= 1) {
            if (threadIdx.x < stride) red[threadIdx.x] += red[threadIdx.x + stride];
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            double result = red[0];
            if (accumulate) result += out[(size_t)view * components + k];
            out[(size_t)view * components + k] = result;
            if (!isfinite(result)) atomicOr(&status[view], DPT_STATUS_RANGE);
        }
        __syncthreads();
    }
}

}  // namespace

extern "C" {

int dpt_reduce_rays(dpt_plan *p, const double *rays, const double *jacobians, int32_t components, double *out,
                    uint32_t flags, void *stream) {
    if (p == nullptr || rays == nullptr || jacobians == nullptr || out == nullptr)
        return fail(DPT_E_INVALID, "plan, rays, jacobians and out are required");
    if (components < 1 || components > 16) return fail(DPT_E_INVALID, "components must be 1..16");
    if (flags & ~(uint32_t)DPT_ACCUMULATE) return fail(DPT_E_INVALID, "reduction flags are DPT_ACCUMULATE");
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t per_view = p->pixels / p->base.views;
    hipLaunchKernelGGL(rays_reduce_kernel, dim3(p->base.views), dim3(kBlock), 0, s, rays, jacobians, per_view,
                       components, out, (flags & DPT_ACCUMULATE) ? 1 : 0, p->d_status);
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

int dpt_adjoint_gather(dpt_plan *p, const double *poses, const double *cotangent, void *out, int32_t out_precision,
                       uint32_t flags, void *stream) {
    if (p == nullptr || poses == nullptr || cotangent == nullptr || out == nullptr)
        return fail(DPT_E_INVALID, "plan, poses, cotangent and out are required");
    if (p->arithmetic != DPT_ARITH_FP64 || p->cell_gauss)
        return fail(DPT_E_INVALID, "deterministic gather requires strict float64 midpoint sampling");
    if (out_precision != DPT_ARITH_FP32 && out_precision != DPT_ARITH_FP64)
        return fail(DPT_E_INVALID, "out_precision must be DPT_ARITH_FP32 or DPT_ARITH_FP64");
    if (flags & ~(uint32_t)(DPT_ACCUMULATE | DPT_NO_CHECKS))
        return fail(DPT_E_INVALID, "gather flags are DPT_ACCUMULATE and DPT_NO_CHECKS");
    DeviceGuard guard(p->device);
    if (p->d_gather_rays == nullptr) {
        if (hipMalloc((void **)&p->d_gather_rays, sizeof(GatherRay) * (size_t)p->pixels) != hipSuccess)
            return fail(DPT_E_MEMORY, "hipMalloc failed for the gather ray table");
        if (hipMalloc((void **)&p->d_gather_views, sizeof(GatherView) * (size_t)p->base.views) != hipSuccess ||
            hipMalloc((void **)&p->d_guard, sizeof(int)) != hipSuccess) {
            (void)hipFree(p->d_gather_rays);
            (void)hipFree(p->d_gather_views);
            p->d_gather_rays = nullptr;
            p->d_gather_views = nullptr;
            return fail(DPT_E_MEMORY, "hipMalloc failed for the gather view table");
        }
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Params P = launch_params(p, poses);
    timer_begin(p, 2, s);
    HIP_TRY(launch_gather(P, cotangent, p->d_gather_rays, p->d_gather_views, p->d_guard, out,
                          out_precision == DPT_ARITH_FP64, (flags & DPT_ACCUMULATE) != 0,
                          (flags & DPT_NO_CHECKS) == 0, p->d_panel_meta, p->d_panel_modes, p->image_cols, s));
    timer_end(p, 2, s);
    return DPT_OK;
}

}  // extern "C"

// ------------------------------------------------ allocation-free gather --
// Workspace of dpt_adjoint_gather_noalloc: the gather's ray table, view
// table and guard word in one file-scope device array of fixed size.  Every
// GPU the library runs on holds its own copy until the process ends; in host
// code `scratch` names a host-side stand-in, so kernels and copies only ever
// get the per-device address that hipGetSymbolAddress returns.
namespace {

constexpr size_t kScratchBytes = (size_t)DPT_GATHER_NOALLOC_BYTES;
constexpr int kScratchDevices = 64;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_scratch_lock;
unsigned char *g_scratch[kScratchDevices] = {};

size_t align256(size_t n) { return (n + 255) & ~size_t(255); }

// The device address of this device's scratch (looked up once per device,
// with that device current).
int scratch_address(int device, unsigned char **out) {
    if (device < 0 || device >= kScratchDevices) return fail(DPT_E_INVALID, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_lock);
    if (g_scratch[device] == nullptr) {
        DeviceGuard guard(device);
        void *ptr = nullptr;
        HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (ptr == nullptr) return fail(DPT_E_DEVICE, "hipGetSymbolAddress returned no address for the scratch array");
        g_scratch[device] = static_cast<unsigned char *>(ptr);
    }
    *out = g_scratch[device];
    return DPT_OK;
}

}  // namespace

extern "C" {

int dpt_adjoint_gather_noalloc(dpt_plan *p, const double *poses, const double *cotangent, void *out,
                               int32_t out_precision, uint32_t flags, void *stream) {
    if (p == nullptr || poses == nullptr || cotangent == nullptr || out == nullptr)
        return fail(DPT_E_INVALID, "plan, poses, cotangent and out are required");
    if (p->arithmetic != DPT_ARITH_FP64 || p->cell_gauss)
        return fail(DPT_E_INVALID, "deterministic gather requires strict float64 midpoint sampling");
    if (out_precision != DPT_ARITH_FP32 && out_precision != DPT_ARITH_FP64)
        return fail(DPT_E_INVALID, "out_precision must be DPT_ARITH_FP32 or DPT_ARITH_FP64");
    if (flags & ~(uint32_t)(DPT_ACCUMULATE | DPT_NO_CHECKS))
        return fail(DPT_E_INVALID, "gather flags are DPT_ACCUMULATE and DPT_NO_CHECKS");
    // [ray table | view table | guard], each 256-byte aligned
    const size_t ray_bytes = align256(sizeof(GatherRay) * (size_t)p->pixels);
    const size_t view_bytes = align256(sizeof(GatherView) * (size_t)p->base.views);
    const size_t need = ray_bytes + view_bytes + 256;
    if (need > kScratchBytes)
        return fail(DPT_E_INVALID, "the allocation-free gather needs " + std::to_string(need) +
                                       " bytes of workspace for " + std::to_string(p->pixels) + " rays and " +
                                       std::to_string(p->base.views) + " views; its fixed workspace holds " +
                                       std::to_string(kScratchBytes) + " (use dpt_adjoint_gather)");
    unsigned char *base = nullptr;
    const int rc = scratch_address(p->device, &base);
    if (rc != DPT_OK) return rc;
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    GatherRay *rays = reinterpret_cast<GatherRay *>(base);
    GatherView *views = reinterpret_cast<GatherView *>(base + ray_bytes);
    int *guard_word = reinterpret_cast<int *>(base + ray_bytes + view_bytes);
    // launch_gather clears the guard word with a kernel and rewrites both
    // tables before the voxel pass reads them
    HIP_TRY(launch_gather(launch_params(p, poses), cotangent, rays, views, guard_word, out,
                          out_precision == DPT_ARITH_FP64, (flags & DPT_ACCUMULATE) != 0,
                          (flags & DPT_NO_CHECKS) == 0, p->d_panel_meta, p->d_panel_modes, p->image_cols, s));
    return DPT_OK;
}

int dpt_plan_layout(const dpt_plan *p, int32_t *out) {
    if (p == nullptr || out == nullptr) return fail(DPT_E_INVALID, "plan and out are required");
    out[0] = p->base.walk_cap;
    out[1] = 0;
    out[2] = p->base.chunk_samples;
    out[3] = p->vjp_vb;
    out[4] = p->base.gauss_chunks;
    return DPT_OK;
}

int dpt_status(dpt_plan *p, int32_t *host_codes, int32_t clear, void *stream) {
    if (p == nullptr || host_codes == nullptr) return fail(DPT_E_INVALID, "plan and host_codes are required");
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int views = p->base.views;
    HIP_TRY(hipMemcpyAsync(p->h_status, p->d_status, sizeof(int32_t) * views, hipMemcpyDeviceToHost, s));
    if (clear) hipLaunchKernelGGL(fill_i32_kernel, dim3((views + 255) / 256), dim3(256), 0, s, p->d_status, views);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    std::memcpy(host_codes, p->h_status, sizeof(int32_t) * views);
    return DPT_OK;
}

int dpt_convert_field(const float *src, void *dst, int64_t count, int32_t storage, int32_t *status, void *stream) {
    if (src == nullptr || dst == nullptr || count < 0) return fail(DPT_E_INVALID, "src, dst and count are required");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (storage == DPT_STORE_BF16)
        hipLaunchKernelGGL(convert_kernel<__hip_bfloat16>, dim3(grid_blocks(count)), dim3(kBlock), 0, s, src,
                           static_cast<__hip_bfloat16 *>(dst), count, status);
    else if (storage == DPT_STORE_F16)
        hipLaunchKernelGGL(convert_kernel<__half>, dim3(grid_blocks(count)), dim3(kBlock), 0, s, src,
                           static_cast<__half *>(dst), count, status);
    else
        return fail(DPT_E_INVALID, "storage must be DPT_STORE_BF16 or DPT_STORE_F16");
    HIP_TRY(hipGetLastError());
    return DPT_OK;
}

int64_t dpt_cell_count(int32_t nx, int32_t ny, int32_t nz) {
    if (nx < 1 || ny < 1 || nz < 1) return fail(DPT_E_INVALID, "grid counts must be positive");
    return (int64_t)(nx > 1 ? nx - 1 : 1) * (ny > 1 ? ny - 1 : 1) * (nz > 1 ? nz - 1 : 1);
}

int dpt_convert_cells(const void *src, void *dst, int32_t nx, int32_t ny, int32_t nz, int32_t storage,
                      void *stream) {
    if (src == nullptr || dst == nullptr) return fail(DPT_E_INVALID, "src and dst are required");
    if (nx < 1 || ny < 1 || nz < 1 || (int64_t)nx * ny * nz > INT32_MAX)
        return fail(DPT_E_INVALID, "grid counts must be positive and fit signed 32-bit indexing");
    if (storage != DPT_STORE_F32 && storage != DPT_STORE_BF16 && storage != DPT_STORE_F16)
        return fail(DPT_E_INVALID, "storage must be DPT_STORE_F32, DPT_STORE_BF16 or DPT_STORE_F16");
    return launch_cells(src, dst, nx, ny, nz, storage, static_cast<hipStream_t>(stream));
}

int dpt_set_timing(dpt_plan *p, int32_t enabled) {
    if (p == nullptr) return fail(DPT_E_INVALID, "plan is required");
    p->timing = enabled != 0;
    p->timed[0] = p->timed[1] = p->timed[2] = false;
    return DPT_OK;
}

double dpt_kernel_ms(dpt_plan *p, int32_t kind) {
    if (p == nullptr || kind < 0 || kind > 2 || !p->timed[kind]) return -1.0;
    DeviceGuard guard(p->device);
    if (hipEventSynchronize(p->ev[2 * kind + 1]) != hipSuccess) return -1.0;
    float ms = -1.0f;
    if (hipEventElapsedTime(&ms, p->ev[2 * kind], p->ev[2 * kind + 1]) != hipSuccess) return -1.0;
    return (double)ms;
}

int64_t dpt_count_hit_rays(dpt_plan *p, const double *poses, void *stream) {
    if (p == nullptr || poses == nullptr) {
        fail(DPT_E_INVALID, "plan and poses are required");
        return DPT_E_INVALID;
    }
    DeviceGuard guard(p->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Params P = launch_params(p, poses);
    unsigned long long zero = 0, host = 0;
    if (hipMemcpyAsync(p->d_count, &zero, sizeof zero, hipMemcpyHostToDevice, s) != hipSuccess) return DPT_E_DEVICE;
    hipLaunchKernelGGL(count_hits_kernel, dim3(tile_grid(P)), dim3(kBlock), 0, s, P, p->d_count);
    if (hipMemcpyAsync(&host, p->d_count, sizeof host, hipMemcpyDeviceToHost, s) != hipSuccess) return DPT_E_DEVICE;
    if (hipStreamSynchronize(s) != hipSuccess) return DPT_E_DEVICE;
    return (int64_t)host;
}

}  // extern "C"
