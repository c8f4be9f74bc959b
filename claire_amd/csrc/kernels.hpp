// kernels.hpp -- host-side launch interface of the claire_amd HIP kernels.
#pragma once

#include <cmath>
#include <vector>

#include "common.hpp"

namespace claire_amd {

struct __align__(8) c32 {
    float x, y;
};

// ---------------------------------------------------------------------------
// FFT (fft.hip)
// ---------------------------------------------------------------------------
bool fft_size_supported(int n);

class FFTPlan3D {
  public:
    explicit FFTPlan3D(const Dims& d);
    // A plan over twiddle tables the caller keeps on the device (tw_ext[a]
    // holds n[a] values e^{-2πik/n[a]}, as fft_twiddles writes them); the
    // plan neither allocates nor frees device memory.
    FFTPlan3D(const Dims& d, c32* const tw_ext[3]);
    ~FFTPlan3D();
    FFTPlan3D(const FFTPlan3D&) = delete;
    FFTPlan3D& operator=(const FFTPlan3D&) = delete;

    // Individual passes over n fields in one launch (blockIdx.y), field f at in +
    // f·is (and out + f·os, add + f·as): a vector field's components or a time
    // series.
    static constexpr int kMaxFields = 65535;
    void x3_r2c(const float* in, int64_t is, c32* out, int64_t os, int n, hipStream_t st) const;
    // out = alpha·x + beta·add (add may be null, or equal out with as = os)
    void x3_c2r(const c32* in, int64_t is, float* out, int64_t os, int n, hipStream_t st, float alpha = 1.f,
                const float* add = nullptr, int64_t as = 0, float beta = 0.f) const;
    void x2(c32* data, int64_t ds, int n, int dir, hipStream_t st) const;
    void x1(c32* data, int dir, hipStream_t st) const;
    // Fused x1 passes (forward x1, k-space operator, inverse x1).
    void x1_multiplier(c32* data, int64_t ds, int n, const SpecParams& sp, hipStream_t st) const;
    // component d of field f's gradient at out + f·os + d·oc; in + f·is may be
    // one of the three
    void x1_grad(const c32* in, int64_t is, c32* out, int64_t os, int64_t oc, int n, hipStream_t st) const;
    // out (may equal in) = divergence of the field with components in + d·is
    void x1_div(const c32* in, int64_t is, c32* out, hipStream_t st) const;
    // Forward x1 pass that ends in a sum: per block Σ c(k3)·m(k)²·|x̂(k)|² over
    // its columns, m² the regularization norm's (sp.norm; sp.beta1 = β1 for H1,
    // √β1 for H2), so that the sum of all x1_norm_partials(n) values over N
    // is Σ_x |M x|² of the n fields.
    void x1_norm(const c32* in, int64_t is, int n, const SpecParams& sp, double* partial, hipStream_t st) const;
    int64_t x1_norm_partials(int n) const;
    // Projection of a vector field (sp.op kOpProjStokes or kOpProjRelaxed):
    // x̂_i = g_i·scale·m·(g·b̂) in place of the three spectra data + d·ds.
    void x1_project(c32* data, int64_t ds, const SpecParams& sp, hipStream_t st) const;

    Dims dims;

  private:
    c32* tw[3] = {nullptr, nullptr, nullptr};
    bool owns_tw = true;
};

// The twiddle table of an n-point transform: h[k] = e^{-2πik/n}, k < n,
// evaluated in double and rounded to FP32.
void fft_twiddles(int n, c32* h);

// Spectral gradient without device allocation (noalloc.cpp): g = ∇f with
// the launches of SpectralOps::Grad, its spectra and twiddles in a
// file-scope device array of kNoAllocScratchBytes per device.
constexpr size_t kNoAllocScratchBytes = size_t(32) << 20;
size_t noalloc_grad_bytes(const int nx[3]);
void grad_noalloc(const int nx[3], const float* f, float* g, hipStream_t st);

// ---------------------------------------------------------------------------
// Semi-Lagrangian gathers (interp.hip, gather_lds.hip).  X: foot points over
// 2π, one component per field (component d of point i at X[d·nl + i]), except
// for launch_gather1 and launch_points_gather, whose query points are
// interleaved xyz.
// ---------------------------------------------------------------------------
struct GatherDims {
    int n1, n2, n3;
    int64_t nl;
};

GatherDims gather_dims(const Dims& d);

// out = f(X), X interleaved (3 floats per point), any query points: straight from
// global memory, or (launch_points_gather) LDS-staged where the grid is large
void launch_gather1(const GatherDims& g, const float* f, const float* X, float* out, hipStream_t st);
void launch_points_gather(const GatherDims& g, const float* f, const float* X, float* out, hipStream_t st);
// out = X, interleaved
void launch_interleave(int64_t nl, const float* X, float* out, hipStream_t st);
// RK2 characteristic, Euler predictor and velocity gather fused, any
// displacement:
//   X̃ = (x − σ·ht·v)/2π,  X = (x − σ·ht/2·(v(X̃) + v))/2π
void launch_trajectory_rk2(const Dims& d, const float* const v[3], float sigma, float ht, float* X, hipStream_t st);
// Stage 1 to 3 of the RK4 characteristic, any displacement: reads v at the
// stage point in X (stage 1: at the first stage point, formed from v) and
// replaces it by the next one; stage sums as in launch_lds_traj_rk4_stage,
// except that Fout may be Fin.
void launch_trajectory_rk4_stage(int stage, const Dims& d, const float* const v[3], float sigma, float ht, float* X,
                                 const float* Fin, float* Fout, hipStream_t st);

// Packed plan of a trajectory: 3 words per point (12 B), one per axis, the
// fraction t ∈ [1,2) of the rescaled coordinate u = q·N + 3 and the offset of
// the first stencil node from the point (layout in gather_device.hpp).
// Returns the per-axis stencil displacement bound D in cells (synchronizes
// the stream); kNoBound when a foot point is not finite.  n <= 512 per axis.
// `words`: 2·kPlanBlocks ints of pinned host memory that the device can write
// (what the blocks found; one launch at a time may use them).
constexpr int kPlanBlocks = 2048;
constexpr int kNoBound = 1 << 20;
// What the choice of a gather kernel goes by.
struct PlanBound {
    int d;         // displacement bound
    float spread;  // share of the points displaced by six cells or more, all axes
                   // together, against the point 32 further on in memory
};
PlanBound launch_make_plan(const GatherDims& g, const float* X, uint32_t* P, int* words, hipStream_t st);
// RK2 characteristic through the LDS-staged gather, in three passes:
//   1. the packed plan of the Euler predictor X̃ = (x − σ·ht·v)/2π into P
//      (launch_set_velocity or launch_predictor_plan);
//   2. v gathered along it with the corrector as epilogue,
//      X = (x − σ·ht/2·(v(X̃) + v))/2π (launch_lds_traj_rk2_corrector);
//   3. the plan of X into P (launch_make_plan, which returns its bound).
// The foot points equal those of launch_trajectory_rk2.
//
// First pass over a new velocity v (3·nl): copies it to vout (unless v ==
// vout), writes the predictor's plan for σ = +1 and returns the bounds of the
// predictors for σ = +1 and −1 (whose spread is the same) and whether v is zero
// (synchronizes the stream).
struct VelocityBounds {
    PlanBound bound[2];
    bool zero;
};
VelocityBounds launch_set_velocity(const Dims& d, const float* v, float* vout, float ht, uint32_t* P, int* words,
                                   hipStream_t st);
// The predictor's plan alone.
void launch_predictor_plan(const Dims& d, const float* const v[3], float sigma, float ht, uint32_t* P,
                           hipStream_t st);
void launch_lds_traj_rk2_corrector(const Dims& d, const uint32_t* P, PlanBound bound, const float* const v[3], float sigma,
                                   float ht, float* X, hipStream_t st);
// RK4 characteristic the same way: the plan of the first stage point
// (x − σ·ht/2·v)/2π is the predictor's with ht/2; each stage gathers v along the
// previous point's plan, accumulates the stage sum f and writes
// the next point into X (the foot point at stage 3), whose plan
// launch_make_plan builds.  Stage 1
// writes f into Fout (Fin unused), stage 2 reads Fin and writes Fout (two
// distinct buffers: no launch updates an operand in place, so a gather may
// be repeated while its chunk length is tuned), stage 3 reads Fin.
void launch_lds_traj_rk4_stage(int stage, const Dims& d, const uint32_t* P, PlanBound bound, const float* const v[3],
                               float sigma, float ht, const float* Fin, float* Fout, float* X, hipStream_t st);
// Whether the gathers of nz fields along a plan of this bound run LDS-staged: the
// bound is at most kNearBound, or the points are finite, many enough for windows
// centred per block and close enough together for most to lie in them.  The direct
// kernels take the rest; the two agree up to roundings (other products are fused).
constexpr int kNearBound = 4;
bool plan_gather_lds(const GatherDims& g, PlanBound bound, int nz);
// Update coefficient per point: C = 1 + ht/2·(α·dX + α·(1 + ht·α·dX)·d)
// with d = ∇·v, dX = d(X).  α = 1 on the adjoint trajectory gives the SL
// adjoint update λ⁺ = C·λ(X_a); α = ±1 on the state trajectory gives the
// SL update of det(∇y^{±1}), J⁺ = C·J(X_s).
void launch_adjoint_coeff(const GatherDims& g, const float* X, const float* divv, float ht, float alpha, float* C,
                          hipStream_t st);

// A trajectory as the gathers see it: the packed plan, the raw foot points
// (one component per field) and the plan's bound.
struct TrajectoryPlan {
    const uint32_t* P;
    const float* X;
    PlanBound bound;
};

// Gathers along a trajectory.  Vector fields are nf equally spaced component
// pointers.  They run the LDS-staged kernels where plan_gather_lds says so, else the
// direct kernels on the raw foot points (which take the field from blockIdx.y:
// at most kMaxGatherFields of them).
//   gather:          out_d = f_d(X)
//   inc_state_step:  out = ±(f(X) − s)   (m̃^{j+1} = m̃^j(X_s) − s_j; negated for λ̃⁰ = −m̃^nt)
//   adjoint_step:    out = C·f(X)        (λ^{j+1} = C·λ^j(X_a))
constexpr int kMaxGatherFields = 65535;
void launch_plan_gather(const TrajectoryPlan& tp, const GatherDims& g, const float* const f[], int nf,
                        float* const out[], hipStream_t st);
void launch_plan_inc_state_step(const TrajectoryPlan& tp, const GatherDims& g, const float* mt, const float* sj,
                                float* out, int negate, hipStream_t st);
void launch_plan_adjoint_step(const TrajectoryPlan& tp, const GatherDims& g, const float* C, const float* lam,
                              float* out, hipStream_t st);
// launch_adjoint_coeff along a trajectory plan (LDS-staged when its bound
// allows); divv and C must not alias.
void launch_plan_adjoint_coeff(const TrajectoryPlan& tp, const GatherDims& g, const float* divv, float ht, float alpha,
                               float* C, hipStream_t st);
// Direct versions on the raw foot points X (any displacement):
void launch_direct_gather(const GatherDims& g, const float* X, const float* const f[], int nf, float* const out[],
                          hipStream_t st);
void launch_direct_inc_state_step(const GatherDims& g, const float* X, const float* mt, const float* sj, float* out,
                                  int negate, hipStream_t st);
void launch_direct_adjoint_step(const GatherDims& g, const float* X, const float* C, const float* lam, float* out,
                                hipStream_t st);

// b_d = hd·Σ_{j=0..nt} w_j·λ^j·∂_d m^{nt−j} (trapezoid weights); lam holds
// λ^0..λ^nt, gm holds ∇m^0..∇m^nt (3 fields each).
void launch_body_force(int64_t nl, int nt, float ht, float hd, const float* lam, const float* gm, float* const b[3],
                       hipStream_t st);
// Fields stored as 16-bit block floating point (the mixed form): int16
// mantissas q (field k at q + k·nl) and one power-of-two scale per block of
// 256 consecutive values of a field (field k's scales at s + k·bfp16_blocks(nl)).
struct Bfp16Fields {
    int16_t* q;
    float* s;
};
int64_t bfp16_blocks(int64_t nl);
// The same with the gradient fields in 16-bit block floating point,
// accumulated in FP32.
void launch_body_force_bfp(int64_t nl, int nt, float ht, float hd, const float* lam, const Bfp16Fields& gm,
                           float* const b[3], hipStream_t st);
// v = 0 body force: b_d = hd·λ·∂_d m
void launch_body_force_static(int64_t nl, float hd, const float* lam, const float* gm, float* const b[3],
                              hipStream_t st);
// s_j = ht/2·[(∇m^j)(X_s)·ṽX + ∇m^{j+1}·ṽ] for j = 0..nt−1 from a precomputed
// ṽX = ṽ(X_s); writes m̃¹ = −s_0 (λ̃⁰ = s_0 when nt = 1) and s_1..s_{nt−1}.
void launch_inc_state_rhs(int64_t nl, int nt, float ht, const float* const vx[3], const float* const vt[3],
                          const float* gX, const float* gm, float* s, float* mt1, hipStream_t st);

void launch_inc_state_rhs_bfp(int64_t nl, int nt, float ht, const float* const vx[3], const float* const vt[3],
                              const Bfp16Fields& gX, const Bfp16Fields& gm, float* s, float* mt1, hipStream_t st);
// nfields consecutive FP32 fields of nl values (nl a multiple of 4) into 16-bit
// block floating point: per block of 256 values, scale 2^(E−15) with
// max |v| < 2^E, mantissas rounded to nearest (error <= 2^−16 of the block's
// largest magnitude).
void launch_to_bfp16(const float* in, int64_t nl, int nfields, const Bfp16Fields& out, hipStream_t st);

// ---------------------------------------------------------------------------
// Element-wise kernels and reductions (pointwise.hip)
// ---------------------------------------------------------------------------
void launch_fill(float* x, float value, int64_t n, hipStream_t st);
void launch_copy(const float* x, float* y, int64_t n, hipStream_t st);
void launch_scale(float* x, float alpha, int64_t n, hipStream_t st);
// y = alpha·x + y
void launch_axpy(float alpha, const float* x, float* y, int64_t n, hipStream_t st);
// w = alpha·x + y
void launch_waxpy(float alpha, const float* x, const float* y, float* w, int64_t n, hipStream_t st);
// z = x − y
void launch_sub(const float* x, const float* y, float* z, int64_t n, hipStream_t st);

// FP64 reductions.  `partial` must hold kReduceBlocks doubles and `result`
// one double (device memory); the result is written to `host` too, pinned host
// memory that the host reads after a stream synchronization (no copy to queue).
constexpr int kReduceBlocks = 1024;

// Device-resident scalars of a conjugate-gradient solve (reg::Optimizer::Pcg),
// so that a run of iterations needs no host round trip: the step lengths are
// formed on the device from the reduction slots, in double, exactly as the
// host would form them, and every update is skipped once the solve has
// stopped.  Slots: 0 = pᵀw, 1 = rᵀr, 2 = rᵀz.
struct PcgState {
    double rz;     // rᵀz of the current residual
    double tol;    // stop when ‖r‖ <= tol
    double bnorm;  // ‖b‖ (divergence test ‖r‖ >= 1e6·‖b‖)
    double rnorm;  // ‖r‖ after the last iteration
    float a, na, beta;  // float(α), float(−α), float(β) for the updates
    int k;         // iterations taken
    int kmax;      // iteration limit
    int done;      // 0 while running; 1 once stopped
};
// s.rz = slots[2], s.k = 0, s.done = 0, tolerances as given
void launch_pcg_init(PcgState* s, const double* slots, double tol, double bnorm, int kmax, hipStream_t st);
// p = β·p + z unless stopped
void launch_xpay_pcg(const PcgState* s, float* p, const float* z, int64_t n, hipStream_t st);
// d += α·p and r −= α·w in one launch unless stopped
void launch_axpy2_pcg(const PcgState* s, const float* p, float* d, const float* w, float* r, int64_t n,
                      hipStream_t st);
// slots[0] = pᵀw (partial: kReduceBlocks doubles), then the α step
void launch_dot_pcg_alpha(const float* p, const float* w, int64_t n, double* partial, double* slots, PcgState* s,
                          hipStream_t st);
// slots[1] = rᵀr and slots[2] = rᵀz in one pass (partial: 2·kReduceBlocks
// doubles), then the stopping test and the β step; the state after it also
// goes to *host (pinned)
void launch_dots_pcg_beta(const float* r, const float* z, int64_t n, double* partial, double* slots, PcgState* s,
                          PcgState* host, hipStream_t st);
void launch_dot(const float* a, const float* b, int64_t n, double* partial, double* result, double* host,
                hipStream_t st);
void launch_absmax(const float* a, int64_t n, double* partial, double* result, double* host, hipStream_t st);
void launch_sqdist(const float* a, const float* b, int64_t n, double* partial, double* result, double* host,
                   hipStream_t st);
// host[0..2] = minimum, maximum and sum (partial: 3·kReduceBlocks doubles)
void launch_stats(const float* a, int64_t n, double* partial, double* host, hipStream_t st);
// result = Σ partial[0..np), in a fixed order
void launch_sum_partials(const double* partial, int np, double* result, double* host, hipStream_t st);

// ---------------------------------------------------------------------------
// Explicit RK2 transport stages (rk2.hip); each follows a spectral grad or
// div of the step (src/CLAIRE.cpp:1995-2105, 2365-2548, 2962-3135, 3504-3683)
// ---------------------------------------------------------------------------
struct Vec3Ptr {
    const float* p[3];
};
struct Vec3Out {
    float* p[3];
};
// rhs0 = −g·v, m̄ = m + ht·rhs0
void launch_rk2_state_stage1(int64_t nl, float ht, const Vec3Ptr& g, const Vec3Ptr& v, const float* m, float* rhs0,
                             float* mbar, hipStream_t st);
// m⁺ = m + ht/2·(rhs0 − g·v)
void launch_rk2_state_stage2(int64_t nl, float hthalf, const Vec3Ptr& g, const Vec3Ptr& v, const float* m,
                             const float* rhs0, float* mnext, hipStream_t st);
// rhs0 = −∇m̃·v − ∇m·ṽ, m̃̄ = m̃ + ht·rhs0 (has_gmt = false: m̃ = 0)
void launch_rk2_inc_stage1(int64_t nl, float ht, bool has_gmt, const Vec3Ptr& gmt, const Vec3Ptr& v,
                           const Vec3Ptr& gm, const Vec3Ptr& vt, const float* mt, float* rhs0, float* mtbar,
                           hipStream_t st);
// out = ±(m̃ + ht/2·(rhs1 + rhs0)), rhs1 = −∇m̃̄·v − ∇m⁺·ṽ (has_mt = false: m̃ = 0)
void launch_rk2_inc_stage2(int64_t nl, float hthalf, bool has_mt, const Vec3Ptr& gmt, const Vec3Ptr& v,
                           const Vec3Ptr& gm, const Vec3Ptr& vt, const float* mt, const float* rhs0, float* out,
                           bool negate, hipStream_t st);
// v = 0: out = ±m̃ after nt steps m̃ ← m̃ − ht·(∇m·ṽ) from m̃ = 0
void launch_rk2_inc_static(int64_t nl, int nt, float ht, const Vec3Ptr& gm, const Vec3Ptr& vt, float* out, bool negate,
                           hipStream_t st);
// w = λ·v
void launch_rk2_adj_flux(int64_t nl, const float* lam, const Vec3Ptr& v, const Vec3Out& w, hipStream_t st);
// w = v·(λ + ht·rhs0)
void launch_rk2_adj_mid(int64_t nl, float ht, const float* lam, const float* rhs0, const Vec3Ptr& v, const Vec3Out& w,
                        hipStream_t st);
// λ⁺ = λ + ht/2·(rhs0 + rhs1); next: w = λ⁺·v
void launch_rk2_adj_end(int64_t nl, float hthalf, const float* lam, const float* rhs0, const float* rhs1, float* lnext,
                        bool next, const Vec3Ptr& v, const Vec3Out& w, hipStream_t st);

}  // namespace claire_amd
