// interp.hip -- semi-Lagrangian trajectory, plans and direct gathers (gfx950).
//
// Replaces Interp3_Plan::scatter/interpolate + optimized_interp3_ghost_xyz_p
// (src/Interp3_Plan.cpp:294-845, src/interp3.cpp:2492-2719) and the ghost
// exchange accfft_get_ghost_xyz (src/ghost.cpp:555-612) on one GPU.  The
// arithmetic per point is in gather_device.hpp.  Kernels here:
//   * the fused RK2 characteristic (Euler predictor kept in registers);
//   * the packed plan of a trajectory (12 B per point, gather_device.hpp),
//     together with the exact per-axis displacement bound that decides
//     whether the LDS-staged gathers can be used;
//   * direct gathers (one thread per point, stencil rows read from global
//     memory as unaligned 16-byte loads) for what the LDS-staged gathers do not
//     take: raw query points on small grids, displacements of more than four
//     cells on small grids or where neighbouring points go far apart, trajectories
//     with points that are not finite, and calls in a caller's own graph capture
//     (no host wait, so no displacement bound).
#include <algorithm>

#include "gather_device.hpp"

namespace claire_amd {

namespace {

using namespace gather;

constexpr int kThreads = 256;

__device__ __forceinline__ int64_t point_index(int nblocks) {
    return static_cast<int64_t>(xcd_remap(blockIdx.x, nblocks)) * kThreads + threadIdx.x;
}

// Grid indices (i1, i2, i3) of flat point i in 32-bit arithmetic (the
// gathers require nl < 2^31; 64-bit division is a long emulated sequence).
__device__ __forceinline__ void grid_index(const GatherDims& g, int64_t i, int idx[3]) {
    const uint32_t ui = static_cast<uint32_t>(i);
    const uint32_t plane = static_cast<uint32_t>(g.n2) * static_cast<uint32_t>(g.n3);
    const uint32_t i1 = ui / plane;
    const uint32_t r = ui - i1 * plane;
    const uint32_t i2 = r / static_cast<uint32_t>(g.n3);
    idx[0] = static_cast<int>(i1);
    idx[1] = static_cast<int>(i2);
    idx[2] = static_cast<int>(r - i2 * static_cast<uint32_t>(g.n3));
}

// Grid indices of a point index that advances by a fixed stride (the
// bounded-grid loops of the plan kernels): the divisions happen once per
// thread, and each step adds the stride's (i1, i2, i3) parts with carries.
struct GridWalk {
    int idx[3];
    int s[3];
    __device__ GridWalk(const GatherDims& g, int64_t i0, int64_t stride) {
        grid_index(g, i0, idx);
        grid_index(g, stride, s);  // stride = s0·n2·n3 + s1·n3 + s2, s1 < n2, s2 < n3
    }
    __device__ void advance(const GatherDims& g) {
        idx[2] += s[2];
        int c = idx[2] >= g.n3;
        if (c) idx[2] -= g.n3;
        idx[1] += s[1] + c;
        c = idx[1] >= g.n2;
        if (c) idx[1] -= g.n2;
        idx[0] += s[0] + c;
    }
};

__device__ __forceinline__ void load_q3(const float* X, int64_t i, float q[3]) {
    q[0] = X[3 * i + 0];
    q[1] = X[3 * i + 1];
    q[2] = X[3 * i + 2];
}

// Points of a trajectory: component d of point i at X[d·nl + i].
__device__ __forceinline__ void load_point(const float* X, int64_t nl, int64_t i, float q[3]) {
    q[0] = X[i];
    q[1] = X[nl + i];
    q[2] = X[2 * nl + i];
}

__global__ __launch_bounds__(kThreads) void k_gather1(GatherDims g, HH hh, const float* __restrict__ f,
                                                      const float* __restrict__ X, float* __restrict__ out, int nblocks) {
    const int64_t i = point_index(nblocks);
    if (i >= g.nl) return;
    float q[3];
    load_q3(X, i, q);
    Stencil S;
    setup_stencil(q, g, hh.h, S);
    const float* fs[1] = {f};
    float r[1];
    eval_stencil<1>(fs, S, g, r);
    out[i] = r[0];
}

struct P3 {
    const float* in[3];
    float* out[3];
};

// SemiLagrangian::ComputeTrajectoryRK2 (src/SemiLagrangian.cpp:192-288)
// with the Euler predictor kept in registers.
struct TrajParams {
    float hx[3];
    float sht;   // σ·ht
    float shth;  // σ·ht/2
};

__global__ __launch_bounds__(kThreads) void k_traj_rk2(GatherDims g, HH hh, TrajParams tp, P3 v,
                                                       float* __restrict__ X, int nblocks) {
    const int64_t i = point_index(nblocks);
    if (i >= g.nl) return;
    int idx[3];
    grid_index(g, i, idx);
    float vl[3], q[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        vl[d] = v.in[d][i];
        q[d] = foot_point(tp.hx[d], idx[d], tp.sht, vl[d]);
    }
    Stencil S;
    setup_stencil(q, g, hh.h, S);
    float vx[3];
    eval_stencil<3>(v.in, S, g, vx);
#pragma unroll
    for (int d = 0; d < 3; ++d) X[d * g.nl + i] = foot_point(tp.hx[d], idx[d], tp.shth, vx[d] + vl[d]);
}

// SemiLagrangian::ComputeTrajectoryRK4 (src/SemiLagrangian.cpp:297-459), in
// three launches, each one gather of v at the previous stage point:
//   STAGE 1: X¹ = (x − σ·ht/2·v)/2π in registers, f = v + 2·v(X¹),
//            X² = (x − σ·ht/2·v(X¹))/2π;
//   STAGE 2: f += 2·v(X²), X³ = (x − σ·ht·v(X²))/2π;
//   STAGE 3: f += v(X³), X = (x − σ·(ht/6)·f)/2π.
// f and the stage points live in F and X between launches, per component
// (stages may come from here or from the LDS-staged gathers, whichever the
// displacement of the point they read allows).  Precision follows the reference: f += 2.0·vX in
// double, the last update and every division by 2π in double.
struct Rk4Params {
    float hx[3];
    float shth;   // σ·ht/2
    float sht;    // σ·ht
    double s6;    // σ·(ht/6.0)
};

template <int STAGE>
__global__ __launch_bounds__(kThreads) void k_traj_rk4(GatherDims g, HH hh, Rk4Params tp, P3 v,
                                                       float* __restrict__ X, const float* Fin, float* Fout, int nblocks) {
    const int64_t i = point_index(nblocks);
    if (i >= g.nl) return;
    int idx[3];
    grid_index(g, i, idx);
    float vl[3], q[3];
    if constexpr (STAGE == 1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            vl[d] = v.in[d][i];
            q[d] = foot_point(tp.hx[d], idx[d], tp.shth, vl[d]);
        }
    } else {
        load_point(X, g.nl, i, q);
    }
    Stencil S;
    setup_stencil(q, g, hh.h, S);
    float vx[3];
    eval_stencil<3>(v.in, S, g, vx);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if constexpr (STAGE == 1) {
            Fout[d * g.nl + i] = static_cast<float>(static_cast<double>(vl[d]) + 2.0 * static_cast<double>(vx[d]));
            X[d * g.nl + i] = foot_point(tp.hx[d], idx[d], tp.shth, vx[d]);
        } else if constexpr (STAGE == 2) {
            Fout[d * g.nl + i] = static_cast<float>(static_cast<double>(Fin[d * g.nl + i]) + 2.0 * static_cast<double>(vx[d]));
            X[d * g.nl + i] = foot_point(tp.hx[d], idx[d], tp.sht, vx[d]);
        } else {
            X[d * g.nl + i] = foot_point_rk4(tp.hx[d], idx[d], tp.s6, Fin[d * g.nl + i] + vx[d]);
        }
    }
}

// What a block found, in one word of host memory per direction: the largest
// displacement bound above a sum of `low`, which is the same for a wave's lanes
// (the host reads lines that the device has just written, which costs it more than
// the kernel's whole fold).  Points per block stay below 2^20.
constexpr int kLowBits = 20, kTopBound = 2047;
static_assert(kPlanMaxN < kTopBound, "a bound must fit above the sum");

template <int K>
__device__ __forceinline__ void block_words_to(int (&need)[K], const int (&low)[K], int* words) {
    __shared__ int sh[2 * K][kThreads / 64];
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) need[k] = max(need[k], __shfl_xor(need[k], o, 64));
        if ((threadIdx.x & 63) == 0) {
            sh[2 * k][threadIdx.x >> 6] = min(need[k], kTopBound);
            sh[2 * k + 1][threadIdx.x >> 6] = low[k];
        }
    }
    __syncthreads();
    if (threadIdx.x < K) {
        const int* m = sh[2 * threadIdx.x];
        const int* c = sh[2 * threadIdx.x + 1];
        words[threadIdx.x * kPlanBlocks + blockIdx.x] =
            max(max(m[0], m[1]), max(m[2], m[3])) << kLowBits | (c[0] + c[1] + c[2] + c[3]);
    }
}

// Lanes of the wave whose stencil offsets o and those of the lane 32 away (half a
// wave of points is as wide as a gather tile) are kFarApart cells or more apart,
// all axes together.  An axis counts modulo 256 cells: enough for a share.
__device__ __forceinline__ int spread_lanes(const int o[3]) {
    constexpr unsigned kFarApart = 6;
    const unsigned w = ((o[0] + 128) & 255) | ((o[1] + 128) & 255) << 8 | ((o[2] + 128) & 255) << 16;
    return __popcll(__ballot(__builtin_amdgcn_sad_u8(w, __shfl_xor(w, 32, 64), 0u) >= kFarApart));
}

// Encodes the three axes of foot point q at grid index idx, stencil offsets o;
// returns the displacement bound this point needs (kNoBound when not encodable).
__device__ __forceinline__ int encode_point(const GatherDims& g, const HH& hh, const float q[3], const int idx[3],
                                            PlanPt& pt, int o[3]) {
    const int n[3] = {g.n1, g.n2, g.n3};
    int need = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float u = index_coord(q[a], n[a], hh.h[a]);
        o[a] = 0;
        if (!plan_encode(u, idx[a], n[a], pt.w[a], o[a])) {
            need = kNoBound;
            pt.w[a] = 0u;  // t = 1, o = 0: never read
            continue;
        }
        need = max(need, max(-o[a] - 1, o[a] + 1));
    }
    return need;
}

// Packed plan of a trajectory (gather_device.hpp) and the smallest D such
// that every stencil lies within [i − D − 1, i + D + 2] per axis (the window
// of the LDS-staged gathers).  Points that cannot be encoded (non-finite
// coordinates) set D to kNoBound, which routes every gather along this
// trajectory to the direct kernels on the raw foot points.
//
// Each block writes what it found into its own word of a host-resident array,
// which the host folds after the wait that it needs anyway: no word to clear
// before the launch and no copy after it.  One word for all blocks made the
// kernels wait for up to 2048 atomics on one address.  Measured with the
// division-free x/2π (gather_device.hpp): set velocity + both trajectories +
// one gather at 64³ 281 -> 188 µs, 96³ 391 -> 262, 128³ 462 -> 343, 256³
// 1703 -> 1627.
static_assert(kPlanBlocks >= 1 && kThreads == 256, "block_words_to folds four waves");

__global__ __launch_bounds__(kThreads) void k_make_plan(GatherDims g, HH hh, const float* __restrict__ X,
                                                        PlanPt* __restrict__ P, int* __restrict__ words) {
    int need[1] = {0}, count[1] = {0}, o[3];
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    GridWalk gw(g, i0, stride);
    for (int64_t i = i0; i < g.nl; i += stride, gw.advance(g)) {
        float q[3];
        load_point(X, g.nl, i, q);
        PlanPt pt;
        need[0] = max(need[0], encode_point(g, hh, q, gw.idx, pt, o));
        count[0] += spread_lanes(o);
        P[i] = pt;
    }
    block_words_to(need, count, words);
}

// Plan of the Euler predictor X̃ = (x − σ·ht·v)/2π (bounded grid, like
// k_make_plan).
//   SETV = false: the plan alone, its bound known already.
//   SETV = true:  the first pass over a new velocity, which it copies to `vout`
//                 (unless that is where it lies): the predictor's plan for σ and
//                 the bounds for σ and −σ, which differ where the extremes of v
//                 do, and whether any |v| > 0.  In place of a copy, a reduction
//                 over v and a plan launch per direction, each with a wait.
// With the foot points kept per component (no interleaved copy beside the plan),
// set velocity + both trajectories + one gather went from 187 to 134 µs at 64³,
// 342 to 285 at 128³, 1602 to 1451 at 256³ and 12.5 to 11.5 ms at 512³.
template <bool SETV>
__global__ __launch_bounds__(kThreads) void k_predictor_plan(GatherDims g, HH hh, TrajParams tp, P3 v, float* vout,
                                                             PlanPt* __restrict__ P, int* __restrict__ words) {
    int need[2] = {0, 0}, count = 0, o[3];
    bool nonzero = false;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    GridWalk gw(g, i0, stride);
    // The next point's loads are issued before this point's stores, which might alias
    // them, and are in flight while it is encoded (set velocity + state trajectory +
    // one gather at 192³ 279 -> 270 µs, at 256³ 561 -> 548).
    float vn[3] = {0.f, 0.f, 0.f};
    if (i0 < g.nl)
#pragma unroll
        for (int d = 0; d < 3; ++d) vn[d] = v.in[d][i0];
    for (int64_t i = i0; i < g.nl; i += stride, gw.advance(g)) {
        float q[3], r[3];
        const float vd[3] = {vn[0], vn[1], vn[2]};
        if (i + stride < g.nl)
#pragma unroll
            for (int d = 0; d < 3; ++d) vn[d] = v.in[d][i + stride];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            q[d] = foot_point(tp.hx[d], gw.idx[d], tp.sht, vd[d]);
            if constexpr (SETV) {
                r[d] = foot_point(tp.hx[d], gw.idx[d], -tp.sht, vd[d]);
                nonzero = nonzero || fabsf(vd[d]) > 0.0f;
                if (vout) vout[d * g.nl + i] = vd[d];
            }
        }
        PlanPt pt;
        const int a = encode_point(g, hh, q, gw.idx, pt, o);
        P[i] = pt;
        if constexpr (SETV) {
            count += spread_lanes(o);
            need[0] = max(need[0], a);
            need[1] = max(need[1], encode_point(g, hh, r, gw.idx, pt, o));
        }
    }
    if constexpr (SETV) {
        const int low[2] = {count, __ballot(nonzero) != 0};
        block_words_to(need, low, words);
    }
}

// Points given per component, interleaved: 3 floats per point.
__global__ __launch_bounds__(kThreads) void k_interleave(int64_t nl, const float* __restrict__ X,
                                                         float* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= nl) return;
    float q[3];
    load_point(X, nl, i, q);
    out[3 * i + 0] = q[0];
    out[3 * i + 1] = q[1];
    out[3 * i + 2] = q[2];
}

// Update coefficient c = 1 + ht/2·(α·dX + α·(1 + ht·α·dX)·d), d = ∇·v,
// dX = d(X).  With α = 1 on the adjoint trajectory, the SL adjoint step
// λ⁺ = λX + ht/2·(λX·dX + (λX + ht·λX·dX)·d) (src/CLAIRE.cpp:2668-2673,
// 3955-3962) is λ⁺ = c·λX; with α = ±1 on the state trajectory, the SL
// step of det(∇y^{±1}) (src/DeformationFields.cpp:714-721) is J⁺ = c·J(X).
__global__ __launch_bounds__(kThreads) void k_adjoint_coeff(GatherDims g, HH hh, const float* __restrict__ X,
                                                            const float* __restrict__ divv, float ht, float alpha,
                                                            float* __restrict__ C, int nblocks) {
    const int64_t i = point_index(nblocks);
    if (i >= g.nl) return;
    float q[3];
    load_point(X, g.nl, i, q);
    Stencil S;
    setup_stencil(q, g, hh.h, S);
    const float* fs[1] = {divv};
    float dx[1];
    eval_stencil<1>(fs, S, g, dx);
    const float d = divv[i];
    const float hthalf = 0.5f * ht;
    const float adx = alpha * dx[0];
    C[i] = 1.0f + hthalf * (adx + alpha * (1.0f + ht * adx) * d);
}

// Gather along a trajectory straight from the raw foot points (any
// displacement).
template <class Epi>
__global__ __launch_bounds__(kThreads) void k_gather_direct(GatherDims g, HH hh, const float* __restrict__ X,
                                                            const float* __restrict__ fbase, int64_t fzstride, Epi epi,
                                                            int nblocks) {
    const int64_t i = point_index(nblocks);
    if (i >= g.nl) return;
    const float* f = fbase + static_cast<int64_t>(blockIdx.y) * fzstride;
    epi.select(blockIdx.y);
    const float aux = epi.aux(i);
    float q[3];
    load_point(X, g.nl, i, q);
    Stencil S;
    setup_stencil(q, g, hh.h, S);
    const float* fs[1] = {f};
    float r[1];
    eval_stencil<1>(fs, S, g, r);
    epi.store(i, r[0], aux);
}

__global__ __launch_bounds__(kThreads) void k_body_force_static(int64_t nl, float hd, const float* __restrict__ lam,
                                                                const float* __restrict__ gm, P3 b) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= nl) return;
    const float l = lam[i];
    b.out[0][i] = (l * gm[i]) * hd;
    b.out[1][i] = (l * gm[nl + i]) * hd;
    b.out[2][i] = (l * gm[2 * nl + i]) * hd;
}

int nblocks_for(int64_t nl) { return static_cast<int>((nl + kThreads - 1) / kThreads); }

void check_gather_dims(const GatherDims& g) {
    CLR_REQUIRE(g.n1 >= 4 && g.n2 >= 4 && g.n3 >= 4, kErrInvalidArgument, "gather needs n >= 4 per axis");
    CLR_REQUIRE(static_cast<int64_t>(g.n1) * g.n2 * g.n3 == g.nl, kErrInvalidArgument, "inconsistent gather dims");
    CLR_REQUIRE(g.nl < (int64_t(1) << 31), kErrInvalidArgument, "grid too large for 32-bit stencil offsets");
}

void require_plan_size(const GatherDims& g) {
    check_gather_dims(g);
    CLR_REQUIRE(g.n1 <= kPlanMaxN && g.n2 <= kPlanMaxN && g.n3 <= kPlanMaxN, kErrUnsupportedSize,
                "trajectory plans support at most 512 points per axis");
}

TrajParams traj_params(const Dims& d, float sigma, float ht) {
    TrajParams tp;
    for (int a = 0; a < 3; ++a) tp.hx[a] = d.hx[a];
    tp.sht = sigma * ht;
    tp.shth = sigma * (0.5f * ht);
    return tp;
}

template <class Epi>
void launch_direct(const GatherDims& g, const float* X, const float* f, int64_t fz, int nz, const Epi& e,
                   hipStream_t st) {
    check_gather_dims(g);
    const int nb = nblocks_for(g.nl);
    hipLaunchKernelGGL((k_gather_direct<Epi>), dim3(nb, nz), dim3(kThreads), 0, st, g, make_hh(g), X, f, fz, e, nb);
}

}  // namespace

GatherDims gather_dims(const Dims& d) { return GatherDims{d.n[0], d.n[1], d.n[2], d.nl}; }

void launch_gather1(const GatherDims& g, const float* f, const float* X, float* out, hipStream_t st) {
    check_gather_dims(g);
    const int nb = nblocks_for(g.nl);
    hipLaunchKernelGGL(k_gather1, dim3(nb), dim3(kThreads), 0, st, g, make_hh(g), f, X, out, nb);
}

void launch_trajectory_rk2(const Dims& d, const float* const v[3], float sigma, float ht, float* X, hipStream_t st) {
    const GatherDims g = gather_dims(d);
    check_gather_dims(g);
    const int nb = nblocks_for(g.nl);
    P3 p{{v[0], v[1], v[2]}, {nullptr, nullptr, nullptr}};
    hipLaunchKernelGGL(k_traj_rk2, dim3(nb), dim3(kThreads), 0, st, g, make_hh(g), traj_params(d, sigma, ht), p, X, nb);
}

void launch_trajectory_rk4_stage(int stage, const Dims& d, const float* const v[3], float sigma, float ht, float* X,
                                 const float* Fin, float* Fout, hipStream_t st) {
    const GatherDims g = gather_dims(d);
    check_gather_dims(g);
    CLR_REQUIRE(stage >= 1 && stage <= 3, kErrInvalidArgument, "RK4 stage must be 1, 2 or 3");
    CLR_REQUIRE((stage == 1 || Fin) && (stage == 3 || Fout), kErrInvalidArgument, "RK4 stage needs its stage sums");
    const int nb = nblocks_for(g.nl);
    Rk4Params tp;
    for (int a = 0; a < 3; ++a) tp.hx[a] = d.hx[a];
    const float hthalf = 0.5f * ht;
    tp.shth = sigma * hthalf;
    tp.sht = sigma * ht;
    tp.s6 = static_cast<double>(sigma) * (static_cast<double>(ht) / 6.0);
    P3 p{{v[0], v[1], v[2]}, {nullptr, nullptr, nullptr}};
    const HH hh = make_hh(g);
    if (stage == 1)
        hipLaunchKernelGGL(k_traj_rk4<1>, dim3(nb), dim3(kThreads), 0, st, g, hh, tp, p, X, Fin, Fout, nb);
    else if (stage == 2)
        hipLaunchKernelGGL(k_traj_rk4<2>, dim3(nb), dim3(kThreads), 0, st, g, hh, tp, p, X, Fin, Fout, nb);
    else
        hipLaunchKernelGGL(k_traj_rk4<3>, dim3(nb), dim3(kThreads), 0, st, g, hh, tp, p, X, Fin, Fout, nb);
}

namespace {
// The blocks' words of one direction folded: the largest bound, and the sum.
struct PlanWords {
    int d = 0;
    int64_t sum = 0;
    PlanWords(const int* words, int nb) {
        for (int i = 0; i < nb; ++i) {
            d = std::max(d, words[i] >> kLowBits);
            sum += words[i] & ((1 << kLowBits) - 1);
        }
        if (d == kTopBound) d = kNoBound;
    }
};

void wait_for_words(hipStream_t st) {
    check_launches();  // a launch that failed wrote none
    CLR_HIP_CHECK(hipStreamSynchronize(st));
}

int plan_blocks(const GatherDims& g) {
    CLR_REQUIRE(g.nl / kPlanBlocks < (1 << kLowBits) - kThreads, kErrInvalidArgument, "grid too large for a plan");
    return std::min(nblocks_for(g.nl), kPlanBlocks);
}
}  // namespace

PlanBound launch_make_plan(const GatherDims& g, const float* X, uint32_t* P, int* words, hipStream_t st) {
    require_plan_size(g);
    const int nb = plan_blocks(g);
    hipLaunchKernelGGL(k_make_plan, dim3(nb), dim3(kThreads), 0, st, g, make_hh(g), X, reinterpret_cast<PlanPt*>(P),
                       words);
    wait_for_words(st);
    const PlanWords w(words, nb);
    return PlanBound{w.d, static_cast<float>(w.sum) / static_cast<float>(g.nl)};
}

VelocityBounds launch_set_velocity(const Dims& d, const float* v, float* vout, float ht, uint32_t* P, int* words,
                                   hipStream_t st) {
    const GatherDims g = gather_dims(d);
    require_plan_size(g);
    P3 p{{v, v + g.nl, v + 2 * g.nl}, {nullptr, nullptr, nullptr}};
    const int nb = plan_blocks(g);
    hipLaunchKernelGGL(k_predictor_plan<true>, dim3(nb), dim3(kThreads), 0, st, g, make_hh(g),
                       traj_params(d, 1.0f, ht), p, v == vout ? nullptr : vout, reinterpret_cast<PlanPt*>(P), words);
    wait_for_words(st);
    const PlanWords w0(words, nb), w1(words + kPlanBlocks, nb);
    const float spread = static_cast<float>(w0.sum) / static_cast<float>(g.nl);
    VelocityBounds b;
    b.bound[0] = PlanBound{w0.d, spread};
    b.bound[1] = PlanBound{w1.d, spread};
    b.zero = w1.sum == 0;
    return b;
}

void launch_predictor_plan(const Dims& d, const float* const v[3], float sigma, float ht, uint32_t* P,
                           hipStream_t st) {
    const GatherDims g = gather_dims(d);
    require_plan_size(g);
    P3 p{{v[0], v[1], v[2]}, {nullptr, nullptr, nullptr}};
    const int nb = std::min(nblocks_for(g.nl), kPlanBlocks);
    hipLaunchKernelGGL(k_predictor_plan<false>, dim3(nb), dim3(kThreads), 0, st, g, make_hh(g),
                       traj_params(d, sigma, ht), p, nullptr, reinterpret_cast<PlanPt*>(P), nullptr);
}

void launch_interleave(int64_t nl, const float* X, float* out, hipStream_t st) {
    hipLaunchKernelGGL(k_interleave, dim3(nblocks_for(nl)), dim3(kThreads), 0, st, nl, X, out);
}

void launch_adjoint_coeff(const GatherDims& g, const float* X, const float* divv, float ht, float alpha, float* C,
                          hipStream_t st) {
    check_gather_dims(g);
    const int nb = nblocks_for(g.nl);
    hipLaunchKernelGGL(k_adjoint_coeff, dim3(nb), dim3(kThreads), 0, st, g, make_hh(g), X, divv, ht, alpha, C, nb);
}

void launch_direct_gather(const GatherDims& g, const float* X, const float* const f[], int nf, float* const out[],
                          hipStream_t st) {
    const int64_t fz = nf > 1 ? (f[1] - f[0]) : 0;
    const int64_t oz = nf > 1 ? (out[1] - out[0]) : 0;
    for (int d = 2; d < nf; ++d)
        CLR_REQUIRE(f[d] - f[d - 1] == fz && out[d] - out[d - 1] == oz, kErrInvalidArgument,
                    "vector gather needs equally spaced components");
    launch_direct(g, X, f[0], fz, nf, EpiPlain{out[0], oz}, st);
}

void launch_direct_inc_state_step(const GatherDims& g, const float* X, const float* mt, const float* sj, float* out,
                                  int negate, hipStream_t st) {
    CLR_REQUIRE(mt != out, kErrInvalidArgument, "semi-Lagrangian step cannot run in place");
    launch_direct(g, X, mt, 0, 1, EpiIncStep{sj, out, negate ? -1.0f : 1.0f}, st);
}

void launch_direct_adjoint_step(const GatherDims& g, const float* X, const float* C, const float* lam, float* out,
                                hipStream_t st) {
    CLR_REQUIRE(lam != out, kErrInvalidArgument, "semi-Lagrangian step cannot run in place");
    launch_direct(g, X, lam, 0, 1, EpiAdjStep{C, out}, st);
}

void launch_body_force_static(int64_t nl, float hd, const float* lam, const float* gm, float* const b[3],
                              hipStream_t st) {
    const int nb = nblocks_for(nl);
    P3 p{{nullptr, nullptr, nullptr}, {b[0], b[1], b[2]}};
    hipLaunchKernelGGL(k_body_force_static, dim3(nb), dim3(kThreads), 0, st, nl, hd, lam, gm, p);
}

}  // namespace claire_amd
