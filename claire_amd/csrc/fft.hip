// fft.hip -- hand-written 3D real FFT for gfx950 with fused k-space operators.
//
// Replaces AccFFT's accfft_execute_r2c_t / accfft_execute_c2r_t /
// accfft_grad_t / accfft_divergence_t (called e.g. at src/CLAIRE.cpp:2622,
// 3243, src/RegularizationH1.cpp:198-200,253-255; not vendored) on one GPU.
//
// Layout (same as the reference at one rank): real field [x1][x2][x3], x3
// fastest; half spectrum [k1][k2][k3], k3 in [0, n3/2], complex interleaved.
//
// A 3D transform is three passes over HBM:
//   x3 pass  rows of n3 reals, two rows packed as one complex row
//            (z = a + i·b), one complex FFT, split by Hermitian symmetry;
//   x2 pass  batched strided complex FFTs, 16 or more adjacent columns per block
//            so that each row access is a segment of 128 bytes or more;
//   x1 pass  same, and this is where k-space operators are fused: the block
//            holds complete x1 columns, so forward FFT, per-mode multiplier
//            and inverse FFT happen in one read and one write.
// Inside a block a length-N FFT is a Stockham autosort sequence of radix-16/8/
// 5/4/3/2 stages; each thread keeps V values in registers (V a multiple of
// every radix of the length) and the block swaps them through LDS between
// stages.  The inverse uses the forward radices in
// reverse order, so the forward output layout in registers is exactly the
// inverse input layout and fused forward·multiply·inverse needs no exchange.
// Twiddles come from a table generated in double precision on the host.
#include "kernels.hpp"

namespace claire_amd {

namespace {

__device__ __forceinline__ c32 cadd(c32 a, c32 b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ c32 csub(c32 a, c32 b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ c32 cmul(c32 a, c32 b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// a·(DIR·i)
template <int DIR>
__device__ __forceinline__ c32 mul_i(c32 a) { return {-DIR * a.y, DIR * a.x}; }

constexpr float kC8 = 0.70710678118654752440f;   // cos(π/4)
constexpr float kC16 = 0.92387953251128675613f;  // cos(π/8)
constexpr float kS16 = 0.38268343236508977173f;  // sin(π/8)

template <int DIR>
__device__ __forceinline__ void dft2(c32* v) {
    c32 t = v[0];
    v[0] = cadd(t, v[1]);
    v[1] = csub(t, v[1]);
}

template <int DIR>
__device__ __forceinline__ void dft4s(c32& v0, c32& v1, c32& v2, c32& v3) {
    c32 a0 = cadd(v0, v2), a1 = csub(v0, v2), a2 = cadd(v1, v3), a3 = mul_i<DIR>(csub(v1, v3));
    v0 = cadd(a0, a2);
    v2 = csub(a0, a2);
    v1 = cadd(a1, a3);
    v3 = csub(a1, a3);
}

template <int DIR>
__device__ __forceinline__ void dft4(c32* v) { dft4s<DIR>(v[0], v[1], v[2], v[3]); }

template <int DIR>
__device__ __forceinline__ void dft8(c32* v) {
    c32 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    c32 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4s<DIR>(e0, e1, e2, e3);
    dft4s<DIR>(o0, o1, o2, o3);
    // o_k *= w8^k, w8 = exp(DIR·2πi/8)
    o1 = {kC8 * (o1.x - DIR * o1.y), kC8 * (DIR * o1.x + o1.y)};
    o2 = mul_i<DIR>(o2);
    o3 = {kC8 * (-o3.x - DIR * o3.y), kC8 * (DIR * o3.x - o3.y)};
    v[0] = cadd(e0, o0);
    v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1);
    v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2);
    v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3);
    v[7] = csub(e3, o3);
}

template <int DIR>
__device__ __forceinline__ void dft16(c32* v) {
    c32 e[8], o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        e[i] = v[2 * i];
        o[i] = v[2 * i + 1];
    }
    dft8<DIR>(e);
    dft8<DIR>(o);
    // w16^k = (cos(πk/8), DIR·sin(πk/8))
    const float cs[8] = {1.f, kC16, kC8, kS16, 0.f, -kS16, -kC8, -kC16};
    const float sn[8] = {0.f, kS16, kC8, kC16, 1.f, kC16, kC8, kS16};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        c32 w = {cs[k], DIR * sn[k]};
        c32 ow = (k == 0) ? o[k] : (k == 4 ? mul_i<DIR>(o[k]) : cmul(o[k], w));
        v[k] = cadd(e[k], ow);
        v[k + 8] = csub(e[k], ow);
    }
}

constexpr float kS3 = 0.86602540378443864676f;   // sin(2π/3)
constexpr float kC51 = 0.30901699437494742410f;  // cos(2π/5)
constexpr float kC52 = -0.80901699437494742410f; // cos(4π/5)
constexpr float kS51 = 0.95105651629515357212f;  // sin(2π/5)
constexpr float kS52 = 0.58778525229247312917f;  // sin(4π/5)

// X_k = Σ_m x_m·w^{mk}, w = exp(DIR·2πi/3)
template <int DIR>
__device__ __forceinline__ void dft3(c32* v) {
    const c32 t1 = cadd(v[1], v[2]);
    const c32 t2 = {v[0].x - 0.5f * t1.x, v[0].y - 0.5f * t1.y};
    const c32 d = csub(v[1], v[2]);
    const c32 t3 = mul_i<DIR>(c32{kS3 * d.x, kS3 * d.y});
    v[0] = cadd(v[0], t1);
    v[1] = cadd(t2, t3);
    v[2] = csub(t2, t3);
}

// X_k = Σ_m x_m·w^{mk}, w = exp(DIR·2πi/5)
template <int DIR>
__device__ __forceinline__ void dft5(c32* v) {
    const c32 t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
    const c32 t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
    const c32 a1 = {v[0].x + kC51 * t1.x + kC52 * t2.x, v[0].y + kC51 * t1.y + kC52 * t2.y};
    const c32 a2 = {v[0].x + kC52 * t1.x + kC51 * t2.x, v[0].y + kC52 * t1.y + kC51 * t2.y};
    const c32 b1 = mul_i<DIR>(c32{kS51 * t3.x + kS52 * t4.x, kS51 * t3.y + kS52 * t4.y});
    const c32 b2 = mul_i<DIR>(c32{kS52 * t3.x - kS51 * t4.x, kS52 * t3.y - kS51 * t4.y});
    v[0] = cadd(v[0], cadd(t1, t2));
    v[1] = cadd(a1, b1);
    v[4] = csub(a1, b1);
    v[2] = cadd(a2, b2);
    v[3] = csub(a2, b2);
}

template <int R, int DIR>
__device__ __forceinline__ void dft(c32* v) {
    if constexpr (R == 2) dft2<DIR>(v);
    else if constexpr (R == 3) dft3<DIR>(v);
    else if constexpr (R == 4) dft4<DIR>(v);
    else if constexpr (R == 5) dft5<DIR>(v);
    else if constexpr (R == 8) dft8<DIR>(v);
    else if constexpr (R == 16) dft16<DIR>(v);
    else static_assert(R == 2 || R == 3 || R == 4 || R == 5 || R == 8 || R == 16, "unsupported radix");
}

// ---------------------------------------------------------------------------
// Stockham stage machinery.  A length-N transform is run by T = N/V threads
// per column; "virtual" butterfly j of a radix-R stage is done by thread
// j mod T.  Register convention at stage entry: v[q·R + r] = x[j + r·N/R],
// j = t + T·q.  After the last stage (span NS = N/R): v[q·R + r] = X[j + r·N/R].
// ---------------------------------------------------------------------------
template <int... R>
struct Radices {};

template <int N>
struct Plan;
// V = values per thread; Fwd radices; Inv = reverse order.  Row pairs or columns per
// block (see Geo): Row and RowWide of small and large x3 passes, Col of the x2 pass,
// X1 of the x1 passes.
template <> struct Plan<8> { static constexpr int V =  8, Row = 64, RowWide = 256, Col = 64, X1 = 64; using Fwd = Radices<8>; using Inv = Radices<8>; };
template <> struct Plan<16> { static constexpr int V = 16, Row = 64, RowWide = 256, Col = 64, X1 = 64; using Fwd = Radices<16>; using Inv = Radices<16>; };
template <> struct Plan<32> { static constexpr int V = 16, Row = 32, RowWide = 128, Col = 32, X1 = 32; using Fwd = Radices<16, 2>; using Inv = Radices<2, 16>; };
template <> struct Plan<64> { static constexpr int V = 16, Row = 16, RowWide =  64, Col = 32, X1 = 16; using Fwd = Radices<16, 4>; using Inv = Radices<4, 16>; };
template <> struct Plan<128> { static constexpr int V = 16, Row =  8, RowWide =  32, Col = 32, X1 = 16; using Fwd = Radices<16, 8>; using Inv = Radices<8, 16>; };
template <> struct Plan<256> { static constexpr int V = 16, Row = 16, RowWide =  16, Col = 32, X1 = 16; using Fwd = Radices<16, 16>; using Inv = Radices<16, 16>; };
template <> struct Plan<512> { static constexpr int V = 16, Row =  8, RowWide =   8, Col = 16, X1 =  8; using Fwd = Radices<16, 16, 2>; using Inv = Radices<2, 16, 16>; };
// lengths with factors 3 and 5
template <> struct Plan<48> { static constexpr int V = 12, Row = 16, RowWide =  64, Col = 16, X1 = 16; using Fwd = Radices<4, 4, 3>; using Inv = Radices<3, 4, 4>; };
template <> struct Plan<96> { static constexpr int V = 24, Row = 32, RowWide =  64, Col = 32, X1 = 16; using Fwd = Radices<8, 4, 3>; using Inv = Radices<3, 4, 8>; };
template <> struct Plan<150> { static constexpr int V = 30, Row = 25, RowWide =  25, Col = 25, X1 = 25; using Fwd = Radices<2, 3, 5, 5>; using Inv = Radices<5, 5, 3, 2>; };
template <> struct Plan<192> { static constexpr int V = 24, Row =  8, RowWide =  32, Col = 32, X1 = 16; using Fwd = Radices<8, 8, 3>; using Inv = Radices<3, 8, 8>; };

template <class L> struct First;
template <int R, int... RS> struct First<Radices<R, RS...>> { static constexpr int value = R; };
template <class L> struct Last;
template <int R> struct Last<Radices<R>> { static constexpr int value = R; };
template <int R, int R2, int... RS> struct Last<Radices<R, R2, RS...>> { static constexpr int value = Last<Radices<R2, RS...>>::value; };

template <int N, int V, int DIR, int NS, int R>
__device__ __forceinline__ void twiddle_butterfly(c32 (&v)[V], int t, const c32* __restrict__ tw) {
    constexpr int T = N / V;
#pragma unroll
    for (int q = 0; q < V / R; ++q) {
        const int j = t + T * q;
        if constexpr (NS > 1) {
            const int jm = j % NS;
#pragma unroll
            for (int r = 1; r < R; ++r) {
                c32 w = tw[jm * r * (N / (NS * R))];
                if constexpr (DIR > 0) w.y = -w.y;
                v[q * R + r] = cmul(v[q * R + r], w);
            }
        }
        dft<R, DIR>(&v[q * R]);
    }
}

// LDS layouts of the exchanges: lay(n, c) is the slot of element n of the
// block's column (or row pair) c.
//   ColLayout: columns interleaved with an odd pitch; the lanes of a wave run
//              over c, so any row access hits distinct banks.
//   RowLayout: each row contiguous with one pad slot per 16 elements; the
//              lanes of a wave run over n, and the radix-16 strides n = 16t + r
//              and n = t + 16r both map the 16 lanes of a row to 16 distinct
//              bank pairs.
struct ColLayout {
    int LD;
    __device__ __forceinline__ int operator()(int n, int c) const { return n * LD + c; }
};

template <int N>
struct RowLayout {
    static constexpr int CP = N + N / 16;
    __device__ __forceinline__ int operator()(int n, int c) const { return c * CP + n + (n >> 4); }
};

// Write stage outputs (span NS, radix R) to LDS, then load the inputs of the
// next radix-R2 stage.
template <int N, int V, int NS, int R, int R2, class Lay>
__device__ __forceinline__ void exchange(c32 (&v)[V], c32* s, const Lay& lay, int c, int t) {
    constexpr int T = N / V;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < V / R; ++q) {
        const int j = t + T * q;
        const int base = (j / NS) * NS * R + (j % NS);
#pragma unroll
        for (int r = 0; r < R; ++r) s[lay(base + r * NS, c)] = v[q * R + r];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < V / R2; ++q) {
        const int j = t + T * q;
#pragma unroll
        for (int r = 0; r < R2; ++r) v[q * R2 + r] = s[lay(j + r * (N / R2), c)];
    }
}

template <int N, int V, int DIR, int NS, class L>
struct Stages;

template <int N, int V, int DIR, int NS, int R>
struct Stages<N, V, DIR, NS, Radices<R>> {
    template <class Lay>
    __device__ __forceinline__ static void run(c32 (&v)[V], c32*, const Lay&, int, int t, const c32* tw) {
        twiddle_butterfly<N, V, DIR, NS, R>(v, t, tw);
    }
};

template <int N, int V, int DIR, int NS, int R, int R2, int... RS>
struct Stages<N, V, DIR, NS, Radices<R, R2, RS...>> {
    template <class Lay>
    __device__ __forceinline__ static void run(c32 (&v)[V], c32* s, const Lay& lay, int c, int t, const c32* tw) {
        twiddle_butterfly<N, V, DIR, NS, R>(v, t, tw);
        exchange<N, V, NS, R, R2>(v, s, lay, c, t);
        Stages<N, V, DIR, NS * R, Radices<R2, RS...>>::run(v, s, lay, c, t, tw);
    }
};

template <int N, int DIR, class Lay>
__device__ __forceinline__ void fft_regs(c32 (&v)[Plan<N>::V], c32* s, const Lay& lay, int c, int t,
                                         const c32* tw) {
    if constexpr (DIR < 0)
        Stages<N, Plan<N>::V, DIR, 1, typename Plan<N>::Fwd>::run(v, s, lay, c, t, tw);
    else
        Stages<N, Plan<N>::V, DIR, 1, typename Plan<N>::Inv>::run(v, s, lay, c, t, tw);
}

// Block geometry: B columns (or row pairs) per block, T threads per column.
// Blocks of one or two waves reach more CUs on small grids, wait for fewer waves at
// their barriers and leave LDS for more blocks; a column block takes at least 16
// columns, 128-byte segments, and more where they gain by it.  Against 256 threads
// per block everywhere (µs; the outputs differ by 4e-8 of their norm at most, where
// the compiler fuses other products): gradient of 32³ 27.5 -> 19.5 in all; x2 pass of
// 96³ 11.7 -> 9.3 with 32 columns for 64, of 64×64×150 8.5 -> 7.2; x1 gradient of 64³
// 9.3 -> 7.4, of 150³ 31.6 -> 28.4, of 192³ 35.8 -> 32.6 with 16 columns for 32;
// three-field rows of 256×192×150 68 -> 61 and 72 -> 65 with 25 pairs for 51.
template <int N, int B_>
struct Geo {
    static constexpr int V = Plan<N>::V;
    static constexpr int T = N / V;
    static constexpr int B = B_;
    static constexpr int THREADS = B * T;
    static constexpr int LD = B | 1;  // ColLayout pitch (odd: spreads banks)
};
template <int N, int B>
struct RowGeo : Geo<N, B> {
    static constexpr int LDS_ELEMS = B * RowLayout<N>::CP;
};
template <int N>
struct ColGeo : Geo<N, Plan<N>::Col> {
    static constexpr int LDS_ELEMS = N * Geo<N, Plan<N>::Col>::LD;
};
template <int N, int B = Plan<N>::X1>
struct X1Geo : Geo<N, B> {
    static constexpr int LDS_ELEMS = N * Geo<N, B>::LD;
};

// Blocks are dealt round-robin over the 8 XCDs; renumbered so that each XCD owns
// one contiguous range of columns and the cache lines shared by neighbouring blocks
// stay in one L2.
__device__ __forceinline__ unsigned xcd_block() {
    const unsigned nb = gridDim.x, x = blockIdx.x & 7u, r = nb & 7u;
    return x * (nb >> 3) + (x < r ? x : r) + (blockIdx.x >> 3);
}

__device__ __forceinline__ int wavenum(int k, int n) { return k > n / 2 ? k - n : (k == n / 2 ? 0 : k); }

// Per-mode real multiplier, FP32 expressions in the reference's order
// (src/RegularizationH1.cpp:222-229,373-382; src/RegularizationH2.cpp:123-128,
// 236-239,375-381; src/RegularizationH1SN.cpp:210-217,352-359;
// src/RegularizationH2SN.cpp:125-130,241-244,385-390).
__device__ __forceinline__ float spec_multiplier(const SpecParams& p, int w1, int w2, int w3) {
    const float lapik = -static_cast<float>(w1 * w1 + w2 * w2 + w3 * w3);
    const float b0 = p.beta0, b1 = p.beta1;
    switch (p.op) {
        case kOpRegApply:
            switch (p.norm) {
                case kRegH1: return p.hd * p.scale * b0 * (-lapik + b1);
                case kRegH2: return p.scale * b0 * (lapik * lapik + b1);
                case kRegH1SN: return -p.hd * p.scale * b0 * lapik;
                default: return p.hd * p.scale * b0 * (lapik * lapik);
            }
        default: {  // kOpRegInverse, kOpRegInvSqrt
            float regop;
            switch (p.norm) {
                case kRegH1: regop = b0 * (-lapik + b1); break;
                case kRegH2: regop = b0 * (lapik * lapik + b1); break;
                case kRegH1SN: regop = (fabsf(lapik) == 0.0f) ? b0 : -b0 * lapik; break;
                default: regop = (fabsf(lapik) == 0.0f) ? b0 : b0 * (lapik * lapik); break;
            }
            if (p.op == kOpRegInvSqrt) regop = sqrtf(regop);
            return p.scale / regop;
        }
    }
}

// ---------------------------------------------------------------------------
// x3 pass, real -> half complex.  Rows 2p and 2p+1 are packed as a + i·b.
// ---------------------------------------------------------------------------
// Several fields per launch, equally spaced in memory: blockIdx.y selects the
// field (a vector field's components, or the fields of a time series, go through
// one launch instead of one each).  Spacings are in elements.
struct R2CPtrs {
    const float* in;
    int64_t is;
    c32* out;
    int64_t os;
};
struct C2RPtrs {
    const c32* in;
    int64_t is;
    float* out;
    int64_t os;
    const float* add;
    int64_t as;
};
struct ColPtrs {  // in place
    c32* data;
    int64_t ds;
};

template <int N, int B>
__global__ __launch_bounds__((RowGeo<N, B>::THREADS)) void k_row_r2c(R2CPtrs ptr, int64_t nrows, const c32* __restrict__ tw) {
    const float* __restrict__ in = ptr.in + blockIdx.y * ptr.is;
    c32* __restrict__ out = ptr.out + blockIdx.y * ptr.os;
    using G = RowGeo<N, B>;
    __shared__ c32 s[G::LDS_ELEMS];
    constexpr int V = G::V, T = G::T, R0 = First<typename Plan<N>::Fwd>::value,
                  RL = Last<typename Plan<N>::Fwd>::value;
    constexpr int NH = N / 2 + 1;
    const int t = threadIdx.x % T;
    const int c = threadIdx.x / T;
    const int64_t ra = 2 * (static_cast<int64_t>(blockIdx.x) * G::B + c);
    const int64_t rb = ra + 1;
    const bool va = ra < nrows, vb = rb < nrows;
    const float* pa = in + ra * N;
    const float* pb = in + rb * N;
    c32 v[V];
#pragma unroll
    for (int q = 0; q < V / R0; ++q) {
        const int j = t + T * q;
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int n = j + r * (N / R0);
            v[q * R0 + r] = {va ? pa[n] : 0.f, vb ? pb[n] : 0.f};
        }
    }
    const RowLayout<N> lay;
    fft_regs<N, -1>(v, s, lay, c, t, tw);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < V / RL; ++q) {
        const int j = t + T * q;
#pragma unroll
        for (int r = 0; r < RL; ++r) s[lay(j + r * (N / RL), c)] = v[q * RL + r];
    }
    __syncthreads();
    c32* oa = out + ra * NH;
    c32* ob = out + rb * NH;
    for (int k = t; k < NH; k += T) {
        const c32 zk = s[lay(k, c)];
        const c32 zm = s[lay(k == 0 ? 0 : N - k, c)];
        if (va) oa[k] = {0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y)};
        if (vb) ob[k] = {0.5f * (zk.y + zm.y), 0.5f * (zm.x - zk.x)};
    }
}

// ---------------------------------------------------------------------------
// x3 pass, half complex -> real, with epilogue out = alpha·x + beta·add.
// The imaginary parts of the k3 = 0 and k3 = n3/2 coefficients are ignored
// (FFTW c2r convention).
// ---------------------------------------------------------------------------
// Calls use(e, load(e)) for the e < n of this thread's part of [0, MOST), in
// batches whose loads are all issued before the first value is used.
template <int MOST, int THREADS, class Load, class Use>
__device__ __forceinline__ void flat_copy(int n, Load&& load, Use&& use) {
    constexpr int ITER = (MOST + THREADS - 1) / THREADS, BATCH = 15;
#pragma unroll 1
    for (int i0 = 0; i0 < ITER; i0 += BATCH) {
        decltype(load(0)) x[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int e = threadIdx.x + THREADS * (i0 + i);
            if (e < n) x[i] = load(e);
        }
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int e = threadIdx.x + THREADS * (i0 + i);
            if (e < n) use(e, x[i]);
        }
    }
}

// ADD: some field has an added term (its values are loaded before the
// transform, in registers the plain pass does not need).
template <int N, int B, bool ADD>
__global__ __launch_bounds__((RowGeo<N, B>::THREADS)) void k_row_c2r(C2RPtrs ptr, int64_t nrows,
                                                                     const c32* __restrict__ tw, float alpha,
                                                                     float beta) {
    const c32* __restrict__ in = ptr.in + blockIdx.y * ptr.is;
    float* __restrict__ out = ptr.out + blockIdx.y * ptr.os;
    const float* __restrict__ add = ADD ? ptr.add + blockIdx.y * ptr.as : nullptr;
    using G = RowGeo<N, B>;
    __shared__ c32 s[G::LDS_ELEMS];
    constexpr int V = G::V, T = G::T, R0 = First<typename Plan<N>::Inv>::value,
                  RL = Last<typename Plan<N>::Inv>::value;
    constexpr int NH = N / 2 + 1;
    const int t = threadIdx.x % T;
    const int c = threadIdx.x / T;
    const int64_t ra = 2 * (static_cast<int64_t>(blockIdx.x) * G::B + c);
    const int64_t rb = ra + 1;
    const bool va = ra < nrows, vb = rb < nrows;
    const c32* ha = in + ra * NH;
    const c32* hb = in + rb * NH;
    c32 v[V];
    // the epilogue's added field, loaded before the transform so that its
    // latency overlaps the butterflies (three-field pass with the add at
    // 256³: 115.7 -> 113.0 µs, outputs identical)
    constexpr int NQ = (N % 4 == 0) ? (N / 4 + T - 1) / T : 1;
    float4 qa[NQ], qb[NQ];
    if constexpr (N % 4 == 0) {
        const float* aa0 = add ? add + ra * N : nullptr;
        const float* ab0 = add ? add + rb * N : nullptr;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int m = t + T * i;
            if (aa0 && va && m < N / 4) qa[i] = reinterpret_cast<const float4*>(aa0)[m];
            if (ab0 && vb && m < N / 4) qb[i] = reinterpret_cast<const float4*>(ab0)[m];
        }
    }
#pragma unroll
    for (int q = 0; q < V / R0; ++q) {
        const int j = t + T * q;
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int k = j + r * (N / R0);
            const bool mirror = k > N / 2;
            const int kk = mirror ? N - k : k;
            c32 A = va ? ha[kk] : c32{0.f, 0.f};
            c32 Bv = vb ? hb[kk] : c32{0.f, 0.f};
            if (kk == 0 || kk == N / 2) {
                A.y = 0.f;
                Bv.y = 0.f;
            }
            if (mirror) {
                A.y = -A.y;
                Bv.y = -Bv.y;
            }
            v[q * R0 + r] = {A.x - Bv.y, A.y + Bv.x};
        }
    }
    const RowLayout<N> lay;
    fft_regs<N, +1>(v, s, lay, c, t, tw);
    float* oa = out + ra * N;
    float* ob = out + rb * N;
    const float* aa = add ? add + ra * N : nullptr;
    const float* ab = add ? add + rb * N : nullptr;
    if constexpr (N % 4 == 0) {
        // Stage the result through LDS so that each lane writes 4 consecutive
        // reals (16-byte stores) of both rows.
        __syncthreads();
#pragma unroll
        for (int q = 0; q < V / RL; ++q) {
            const int j = t + T * q;
#pragma unroll
            for (int r = 0; r < RL; ++r) s[lay(j + r * (N / RL), c)] = v[q * RL + r];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int m = t + T * i;
            if (m >= N / 4) break;
            const c32 z0 = s[lay(4 * m, c)], z1 = s[lay(4 * m + 1, c)], z2 = s[lay(4 * m + 2, c)],
                      z3 = s[lay(4 * m + 3, c)];
            if (va) {
                float4 o = make_float4(alpha * z0.x, alpha * z1.x, alpha * z2.x, alpha * z3.x);
                if (aa) {
                    const float4 x = qa[i];
                    o = make_float4(o.x + beta * x.x, o.y + beta * x.y, o.z + beta * x.z, o.w + beta * x.w);
                }
                reinterpret_cast<float4*>(oa)[m] = o;
            }
            if (vb) {
                float4 o = make_float4(alpha * z0.y, alpha * z1.y, alpha * z2.y, alpha * z3.y);
                if (ab) {
                    const float4 x = qb[i];
                    o = make_float4(o.x + beta * x.x, o.y + beta * x.y, o.z + beta * x.z, o.w + beta * x.w);
                }
                reinterpret_cast<float4*>(ob)[m] = o;
            }
        }
    } else if constexpr (ADD) {
        // Rows that are no multiple of 16 bytes, with an added field: the
        // block's rows, contiguous in memory, are staged through LDS and
        // written value by value with consecutive lanes on consecutive values,
        // as the added field is read.  (Written from the registers, in runs of
        // 5 values with a dependent read of the added field each, the
        // three-field pass took 171 µs at 256×192×150, where moving its bytes
        // takes about 50; the Hessian matvec there 1113 -> 1014 µs.  Without
        // the added field staging gains nothing there and loses 4% at
        // 64×64×150, and the passes' other accesses lose up to 10% by it at
        // every length whose rows have fewer than 16 threads.)
        __syncthreads();
#pragma unroll
        for (int q = 0; q < V / RL; ++q) {
            const int j = t + T * q;
#pragma unroll
            for (int r = 0; r < RL; ++r) s[lay(j + r * (N / RL), c)] = v[q * RL + r];
        }
        __syncthreads();
        const int64_t r0 = 2 * static_cast<int64_t>(blockIdx.x) * G::B;
        const int rows = nrows - r0 < 2 * G::B ? static_cast<int>(nrows - r0) : 2 * G::B;
        const float* sf = reinterpret_cast<const float*>(s);
        float* dst = out + r0 * N;
        const float* ad = add ? add + r0 * N : nullptr;
        auto value = [&](int e) {
            const int row = e / N;
            return alpha * sf[2 * lay(e - row * N, row >> 1) + (row & 1)];
        };
        if (ad)  // may be dst: each value is read before it is written
            flat_copy<2 * G::B * N, G::THREADS>(
                rows * N, [&](int e) { return ad[e]; }, [&](int e, float x) { dst[e] = value(e) + beta * x; });
        else
            for (int e = threadIdx.x; e < rows * N; e += G::THREADS) dst[e] = value(e);
    } else {
#pragma unroll
        for (int q = 0; q < V / RL; ++q) {
            const int j = t + T * q;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const int n = j + r * (N / RL);
                const c32 z = v[q * RL + r];
                if (va) oa[n] = alpha * z.x;
                if (vb) ob[n] = alpha * z.y;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Strided column pass (x2 or x1), plain forward or inverse, in place allowed.
// Column cg starts at (cg / inner)·outer + cg % inner; elements are estride
// apart.
// ---------------------------------------------------------------------------
struct ColGeom {
    int64_t ncols, inner, outer, estride;
};

// Offset of column cg's first element; column counts and the inner extent
// fit 32 bits (64-bit division is a long emulated sequence).
template <int N>
__device__ __forceinline__ int64_t col_base(const ColGeom& g, int64_t cg) {
    const uint32_t c = static_cast<uint32_t>(cg), in = static_cast<uint32_t>(g.inner);
    const uint32_t q = c / in;
    return static_cast<int64_t>(q) * g.outer + static_cast<int64_t>(c - q * in);
}

// Raw buffer access to one field of a complex spectrum of `elems` values: a
// per-lane byte offset (the lane's column and row) plus a uniform one (the
// element's stride multiple), both 32-bit, so a column pass keeps one address
// register per lane instead of a 64-bit address per element.  The launchers
// require fields under 2 GiB.
using spec_rsrc_t = __amdgpu_buffer_rsrc_t;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ spec_rsrc_t spec_rsrc(const c32* p, int64_t elems) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<c32*>(p), 0, static_cast<int>(elems * 8), 0x00020000);
}
__device__ __forceinline__ c32 bload_c(spec_rsrc_t r, uint32_t voff, uint32_t soff) {
    const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
    return {__uint_as_float(w.x), __uint_as_float(w.y)};
}
__device__ __forceinline__ void bstore_c(spec_rsrc_t r, c32 v, uint32_t voff, uint32_t soff) {
    u32x2 w;
    w.x = __float_as_uint(v.x);
    w.y = __float_as_uint(v.y);
    __builtin_amdgcn_raw_buffer_store_b64(w, r, voff, soff, 0);
}

template <int N, int DIR>
__global__ __launch_bounds__(ColGeo<N>::THREADS) void k_col(ColPtrs ptr, ColGeom geo, const c32* __restrict__ tw) {
    c32* data = ptr.data + blockIdx.y * ptr.ds;  // in place
    using G = ColGeo<N>;
    __shared__ c32 s[G::LDS_ELEMS];
    using L = typename std::conditional<(DIR < 0), typename Plan<N>::Fwd, typename Plan<N>::Inv>::type;
    constexpr int V = G::V, T = G::T, R0 = First<L>::value, RL = Last<L>::value;
    const int c = threadIdx.x % G::B;
    const int t = threadIdx.x / G::B;
    // x2 rows are never 128-byte aligned (nh is odd), so neighbouring blocks share
    // cache lines (renumbered only where 8 divided the number of blocks, the
    // three-field pass of 192³ took 41 µs, now 29)
    const int64_t cg = static_cast<int64_t>(xcd_block()) * G::B + c;
    const bool valid = cg < geo.ncols;
    const int64_t base = valid ? col_base<N>(geo, cg) : 0;
    c32 v[V];
    const spec_rsrc_t rio = spec_rsrc(data, geo.ncols * N);
    const uint32_t es8 = static_cast<uint32_t>(geo.estride) * 8u;
    const uint32_t lane = static_cast<uint32_t>(base) * 8u + static_cast<uint32_t>(t) * es8;
#pragma unroll
    for (int q = 0; q < V / R0; ++q)
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const c32 x = bload_c(rio, lane, static_cast<uint32_t>(T * q + r * (N / R0)) * es8);
            v[q * R0 + r] = valid ? x : c32{0.f, 0.f};
        }
    fft_regs<N, DIR>(v, s, ColLayout{G::LD}, c, t, tw);
    if (valid) {
#pragma unroll
        for (int q = 0; q < V / RL; ++q)
#pragma unroll
            for (int r = 0; r < RL; ++r)
                bstore_c(rio, v[q * RL + r], lane, static_cast<uint32_t>(T * q + r * (N / RL)) * es8);
    }
}

// ---------------------------------------------------------------------------
// Fused x1 pass: forward x1 FFT, k-space operator, inverse x1 FFT.
//   kFuseMult  out[d] = F1⁻¹(m(k)·F1(in[d]))         d = blockIdx.y
//   kFuseGrad  out[d] = F1⁻¹(i·w_d·scale·F1(in[0]))   d = 0..2
//   kFuseDiv   out[0] = F1⁻¹(Σ_d i·w_d·scale·F1(in[d]))
// Columns of the x1 pass are (k2, k3) with cg = k2·nh + k3.
// ---------------------------------------------------------------------------
enum FuseMode { kFuseMult = 0, kFuseGrad = 1, kFuseDiv = 2, kFuseProject = 3 };

// Per-mode factor m of the models' projections, FP32/FP64 exactly as the
// reference writes it: ĉ = scale·m·(g·b̂), x̂_i = g_i·ĉ, b ← b + F⁻¹x̂.
//   Stokes (src/CLAIREStokes.cpp:457-462): m = −1/|w|², the Nyquist index
//   kept at +n/2 in |w|², −1 at w = 0.
//   Relaxed (src/CLAIREDivReg.cpp:362-404): lapik = −|g|² (Nyquist zeroed),
//   m = opik·(1/lapik), opik = 1/(β0·(1/(β2·(−lapik + 1))) + 1).
__device__ __forceinline__ float proj_factor(const SpecParams& p, int k1, int k2, int k3, int n1, int n2, int n3) {
    const int x1 = k1 > n1 / 2 ? k1 - n1 : k1, x2 = k2 > n2 / 2 ? k2 - n2 : k2, x3 = k3 > n3 / 2 ? k3 - n3 : k3;
    if (p.op == kOpProjStokes) {
        const float lap = static_cast<float>(static_cast<long>(x1) * x1 + static_cast<long>(x2) * x2 +
                                             static_cast<long>(x3) * x3);
        return lap == 0.0f ? -1.0f : static_cast<float>(-1.0 / static_cast<double>(lap));
    }
    const int z1 = k1 == n1 / 2 ? 0 : x1, z2 = k2 == n2 / 2 ? 0 : x2, z3 = k3 == n3 / 2 ? 0 : x3;
    const float lapik = -static_cast<float>(static_cast<long>(z1) * z1 + static_cast<long>(z2) * z2 +
                                            static_cast<long>(z3) * z3);
    const float lapinvik = lapik == 0.0f ? -1.0f : static_cast<float>(1.0 / static_cast<double>(lapik));
    float opik = static_cast<float>(1.0 / (static_cast<double>(p.beta2) * (static_cast<double>(-lapik) + 1.0)));
    opik = static_cast<float>(1.0 / (static_cast<double>(p.beta0) * static_cast<double>(opik) + 1.0));
    return opik * lapinvik;
}

// Field f of a pass at in + f·is and out + f·os; in grad mode field f's three
// components go to out + f·os + d·oc, in div mode the components come from
// in + d·is.
struct X1Ptrs {
    const c32* in;
    int64_t is;
    c32* out;
    int64_t os;
    int64_t oc;
};

// The columns of an x1 pass lie side by side, so blocks of 16 share lines only where
// the planes are not 128-byte aligned: there the blocks are renumbered (128×150×128,
// multiplier of three fields 20.5 -> 18.2 µs), elsewhere neighbouring blocks are
// better on different XCDs (512³ gradient, in two stages of 32 and 16: 717 against 768
// µs).
__device__ __forceinline__ unsigned x1_block(const ColGeom& g) {
    return g.estride % 16 != 0 ? xcd_block() : blockIdx.x;
}

template <int N, int MODE, int B>
__global__ __launch_bounds__((X1Geo<N, B>::THREADS)) void k_x1_fused(X1Ptrs ptr, ColGeom geo, const c32* __restrict__ tw,
                                                                   SpecParams sp, int n2, int n3, int nh) {
    using G = X1Geo<N, B>;
    __shared__ c32 s[G::LDS_ELEMS];
    using LF = typename Plan<N>::Fwd;
    constexpr int V = G::V, T = G::T, R0 = First<LF>::value, RL = Last<LF>::value;
    const int c = threadIdx.x % G::B;
    const int t = threadIdx.x / G::B;
    const unsigned blk = x1_block(geo);
    const int64_t cg = static_cast<int64_t>(blk) * G::B + c;
    const bool valid = cg < geo.ncols;
    const int64_t base = valid ? cg : 0;
    const int k2 = static_cast<int>(static_cast<uint32_t>(cg) / static_cast<uint32_t>(nh));
    const int k3 = static_cast<int>(cg) - k2 * nh;
    const int w2 = wavenum(k2, n2), w3 = wavenum(k3, n3);

    const uint32_t es8 = static_cast<uint32_t>(geo.estride) * 8u;
    const uint32_t lane = static_cast<uint32_t>(base) * 8u + static_cast<uint32_t>(t) * es8;
    auto load_fwd = [&](const c32* src, c32 (&v)[V]) {
        const spec_rsrc_t r_in = spec_rsrc(src, geo.ncols * N);
#pragma unroll
        for (int q = 0; q < V / R0; ++q)
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const c32 x = bload_c(r_in, lane, static_cast<uint32_t>(T * q + r * (N / R0)) * es8);
                v[q * R0 + r] = valid ? x : c32{0.f, 0.f};
            }
        fft_regs<N, -1>(v, s, ColLayout{G::LD}, c, t, tw);
    };
    // After the forward pass v[q·RL + r] = X[k1], k1 = j + r·N/RL; the
    // inverse plan starts with radix RL and expects the same layout.
    auto inv_store = [&](c32 (&v)[V], c32* dst) {
        fft_regs<N, +1>(v, s, ColLayout{G::LD}, c, t, tw);
        constexpr int RI = Last<typename Plan<N>::Inv>::value;
        if (valid) {
            const spec_rsrc_t r_out = spec_rsrc(dst, geo.ncols * N);
#pragma unroll
            for (int q = 0; q < V / RI; ++q)
#pragma unroll
                for (int r = 0; r < RI; ++r)
                    bstore_c(r_out, v[q * RI + r], lane, static_cast<uint32_t>(T * q + r * (N / RI)) * es8);
        }
    };

    if constexpr (MODE == kFuseMult) {
        c32 v[V];
        load_fwd(ptr.in + blockIdx.y * ptr.is, v);
#pragma unroll
        for (int q = 0; q < V / RL; ++q) {
            const int j = t + T * q;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const int w1 = wavenum(j + r * (N / RL), N);
                const float m = spec_multiplier(sp, w1, w2, w3);
                v[q * RL + r] = {v[q * RL + r].x * m, v[q * RL + r].y * m};
            }
        }
        inv_store(v, ptr.out + blockIdx.y * ptr.os);
    } else if constexpr (MODE == kFuseGrad) {
        c32 x[V];
        load_fwd(ptr.in + blockIdx.y * ptr.is, x);
        const float sc = sp.scale;
#pragma unroll 1
        for (int d = 0; d < 3; ++d) {
            c32 v[V];
#pragma unroll
            for (int q = 0; q < V / RL; ++q) {
                const int j = t + T * q;
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int w = (d == 0) ? wavenum(j + r * (N / RL), N) : (d == 1 ? w2 : w3);
                    const float wd = static_cast<float>(w);
                    const c32 a = x[q * RL + r];
                    v[q * RL + r] = {-wd * a.y * sc, wd * a.x * sc};
                }
            }
            inv_store(v, ptr.out + blockIdx.y * ptr.os + d * ptr.oc);
        }
    } else if constexpr (MODE == kFuseDiv) {
        c32 acc[V];
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = {0.f, 0.f};
#pragma unroll 1
        for (int d = 0; d < 3; ++d) {
            c32 v[V];
            load_fwd(ptr.in + d * ptr.is, v);
#pragma unroll
            for (int q = 0; q < V / RL; ++q) {
                const int j = t + T * q;
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int w = (d == 0) ? wavenum(j + r * (N / RL), N) : (d == 1 ? w2 : w3);
                    const float wd = static_cast<float>(w);
                    const c32 a = v[q * RL + r];
                    // Σ_d i·w_d·a_d, accumulated as the oracle and AccFFT order the terms
                    acc[q * RL + r].x += -wd * a.y;
                    acc[q * RL + r].y += wd * a.x;
                }
            }
        }
        const float sc = sp.scale;
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = {acc[i].x * sc, acc[i].y * sc};
        inv_store(acc, ptr.out);
    } else {
        // projection of a vector field: all three components at every mode
        c32 a[V], b[V], e[V];
        load_fwd(ptr.in, a);
        load_fwd(ptr.in + ptr.is, b);
        load_fwd(ptr.in + 2 * ptr.is, e);
        const float sc = sp.scale;
        const float g2 = static_cast<float>(w2), g3 = static_cast<float>(w3);
#pragma unroll
        for (int q = 0; q < V / RL; ++q) {
            const int j = t + T * q;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const int k1 = j + r * (N / RL);
                const float g1 = static_cast<float>(wavenum(k1, N));
                const float m = proj_factor(sp, k1, k2, k3, N, n2, n3);
                const int i = q * RL + r;
                float cre = -sc * (g1 * a[i].x + g2 * b[i].x + g3 * e[i].x);
                float cim = sc * (g1 * a[i].y + g2 * b[i].y + g3 * e[i].y);
                cre *= m;
                cim *= m;
                b[i] = {-g2 * cre, g2 * cim};
                e[i] = {-g3 * cre, g3 * cim};
                a[i] = {cre * -g1, cim * g1};
            }
        }
        inv_store(a, ptr.out);
        inv_store(b, ptr.out + ptr.os);
        inv_store(e, ptr.out + 2 * ptr.os);
    }
}

// ---------------------------------------------------------------------------
// Norms of the regularization functionals from the spectrum.  By Parseval
//   Σ_x |M v|² = (1/N)·Σ_k c(k3)·m(k)²·|v̂(k)|²,
// with c = 2 for the half spectrum's columns 0 < k3 < n3/2, which stand for
// their mirror images too, and 1 for the others.  The block holds complete x1
// columns after the forward pass, so it folds them in FP64 and writes one
// partial sum instead of a spectrum; no inverse transform, gradient field or
// dot product is left (objective at 192³ 1570 -> 1132 µs, of which the functional
// 570 -> about 125; at 64³ 423 -> 282).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double norm_factor(const SpecParams& p, double k2) {
    switch (p.norm) {  // m² without the constants the host applies
        case kRegH1: return k2 + static_cast<double>(p.beta1);   // ‖∇v‖² + β1·‖v‖²
        case kRegH1SN: return k2;                                // ‖∇v‖²
        case kRegH2: {                                           // ‖(Δ + √β1)v‖²
            const double m = static_cast<double>(p.beta1) - k2;  // β1 holds √β1
            return m * m;
        }
        default: return k2 * k2;                                 // ‖Δv‖²
    }
}

template <int N>
__global__ __launch_bounds__(X1Geo<N>::THREADS) void k_x1_norm(X1Ptrs ptr, ColGeom geo, const c32* __restrict__ tw,
                                                             SpecParams sp, int n2, int n3, int nh,
                                                             double* __restrict__ partial) {
    using G = X1Geo<N>;
    __shared__ c32 s[G::LDS_ELEMS];
    using LF = typename Plan<N>::Fwd;
    constexpr int V = G::V, T = G::T, R0 = First<LF>::value, RL = Last<LF>::value;
    const int c = threadIdx.x % G::B;
    const int t = threadIdx.x / G::B;
    const unsigned blk = x1_block(geo);
    const int64_t cg = static_cast<int64_t>(blk) * G::B + c;
    const bool valid = cg < geo.ncols;
    const int64_t base = valid ? cg : 0;
    const int k2 = static_cast<int>(static_cast<uint32_t>(cg) / static_cast<uint32_t>(nh));
    const int k3 = static_cast<int>(cg) - k2 * nh;
    const int w2 = wavenum(k2, n2), w3 = wavenum(k3, n3);
    const uint32_t es8 = static_cast<uint32_t>(geo.estride) * 8u;
    const uint32_t lane = static_cast<uint32_t>(base) * 8u + static_cast<uint32_t>(t) * es8;
    const spec_rsrc_t r_in = spec_rsrc(ptr.in + blockIdx.y * ptr.is, geo.ncols * N);
    c32 v[V];
#pragma unroll
    for (int q = 0; q < V / R0; ++q)
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const c32 x = bload_c(r_in, lane, static_cast<uint32_t>(T * q + r * (N / R0)) * es8);
            v[q * R0 + r] = valid ? x : c32{0.f, 0.f};
        }
    fft_regs<N, -1>(v, s, ColLayout{G::LD}, c, t, tw);
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < V / RL; ++q) {
        const int j = t + T * q;
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const int w1 = wavenum(j + r * (N / RL), N);
            const double x = static_cast<double>(v[q * RL + r].x), y = static_cast<double>(v[q * RL + r].y);
            acc += norm_factor(sp, static_cast<double>(w1 * w1 + w2 * w2 + w3 * w3)) * (x * x + y * y);
        }
    }
    if (k3 != 0 && 2 * k3 != n3) acc *= 2.0;
    // block sum in a fixed order (the thread count need not be a multiple of
    // a wave): one value per thread through LDS, folded by the first wave
    static_assert(G::LDS_ELEMS >= G::THREADS, "one double per thread must fit the exchange buffer");
    double* sh = reinterpret_cast<double*>(s);
    __syncthreads();
    sh[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    double sum = 0.0;
    for (int i = threadIdx.x; i < G::THREADS; i += 64) sum += sh[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (threadIdx.x == 0) partial[static_cast<int64_t>(blockIdx.y) * gridDim.x + blk] = sum;
}

// ---------------------------------------------------------------------------
// Host-side dispatch on the (runtime) transform length.
// ---------------------------------------------------------------------------
template <template <int> class F, class... A>
void dispatch_n(int n, A&&... a) {
    switch (n) {
        case 8: F<8>::go(a...); break;
        case 16: F<16>::go(a...); break;
        case 32: F<32>::go(a...); break;
        case 64: F<64>::go(a...); break;
        case 128: F<128>::go(a...); break;
        case 256: F<256>::go(a...); break;
        case 512: F<512>::go(a...); break;
        case 48: F<48>::go(a...); break;
        case 96: F<96>::go(a...); break;
        case 150: F<150>::go(a...); break;
        case 192: F<192>::go(a...); break;
        default: throw Error(kErrUnsupportedSize, "FFT length " + std::to_string(n) + " not supported");
    }
}

// Row pairs of a launch from which the row passes take blocks of 256 threads.
// Rows of the spectrum are not whole cache lines, so blocks share them at both ends,
// which small blocks do more often: forward rows of 512×192×192 (147456 pairs in
// three fields) take 115 µs with 32 pairs per block, 131 with 8, and of 512×128×128
// (98304) 49 and 53.  Below, the launch is bound by latency and by CUs without a
// block: 32³ 8.0 and 4.6 µs, 96³ 8.6 and 7.0 (one field), 192³ 44 and 39 (inverse).
constexpr int64_t kWideRowPairs = int64_t(1) << 16;

template <int N>
struct RowR2C {
    static void go(const R2CPtrs& p, int ncomp, int64_t nrows, const c32* tw, hipStream_t st) {
        if ((nrows + 1) / 2 * ncomp >= kWideRowPairs)
            launch<Plan<N>::RowWide>(p, ncomp, nrows, tw, st);
        else
            launch<Plan<N>::Row>(p, ncomp, nrows, tw, st);
    }

    template <int B>
    static void launch(const R2CPtrs& p, int ncomp, int64_t nrows, const c32* tw, hipStream_t st) {
        const int64_t blocks = ((nrows + 1) / 2 + B - 1) / B;
        hipLaunchKernelGGL((k_row_r2c<N, B>), dim3(static_cast<unsigned>(blocks), ncomp), dim3(RowGeo<N, B>::THREADS), 0, st,
                           p, nrows, tw);
    }
};

template <int N>
struct RowC2R {
    static void go(const C2RPtrs& p, int ncomp, int64_t nrows, const c32* tw, float alpha, float beta, hipStream_t st) {
        if ((nrows + 1) / 2 * ncomp >= kWideRowPairs)
            launch<Plan<N>::RowWide>(p, ncomp, nrows, tw, alpha, beta, st);
        else
            launch<Plan<N>::Row>(p, ncomp, nrows, tw, alpha, beta, st);
    }

    template <int B>
    static void launch(const C2RPtrs& p, int ncomp, int64_t nrows, const c32* tw, float alpha, float beta,
                       hipStream_t st) {
        const dim3 grid(static_cast<unsigned>(((nrows + 1) / 2 + B - 1) / B), ncomp), block(RowGeo<N, B>::THREADS);
        if (p.add)
            hipLaunchKernelGGL((k_row_c2r<N, B, true>), grid, block, 0, st, p, nrows, tw, alpha, beta);
        else
            hipLaunchKernelGGL((k_row_c2r<N, B, false>), grid, block, 0, st, p, nrows, tw, alpha, beta);
    }
};

template <int N>
struct ColPass {
    static void go(const ColPtrs& p, int ncomp, ColGeom geo, int dir, const c32* tw, hipStream_t st) {
        using G = ColGeo<N>;
        CLR_REQUIRE(geo.ncols * N * 8 < (int64_t(1) << 31), kErrInvalidArgument,
                    "spectrum field too large for 32-bit buffer offsets");
        const dim3 grid(static_cast<unsigned>((geo.ncols + G::B - 1) / G::B), ncomp);
        if (dir < 0)
            hipLaunchKernelGGL((k_col<N, -1>), grid, dim3(G::THREADS), 0, st, p, geo, tw);
        else
            hipLaunchKernelGGL((k_col<N, +1>), grid, dim3(G::THREADS), 0, st, p, geo, tw);
    }
};

// columns of an x1 pass of 512 from which its blocks take 16 of them
constexpr int64_t kWideX1Columns = int64_t(1) << 15;

template <int N>
struct X1Fused {
    static void go(int mode, X1Ptrs p, ColGeom geo, const c32* tw, SpecParams sp, int n2, int n3, int nh, int nfields,
                   hipStream_t st) {
        CLR_REQUIRE(geo.ncols * N * 8 < (int64_t(1) << 31), kErrInvalidArgument,
                    "spectrum field too large for 32-bit buffer offsets");
        switch (mode) {
            case kFuseMult: launch<kFuseMult>(p, geo, tw, sp, n2, n3, nh, nfields, st); break;
            case kFuseGrad: launch<kFuseGrad>(p, geo, tw, sp, n2, n3, nh, nfields, st); break;
            case kFuseProject: launch<kFuseProject>(p, geo, tw, sp, n2, n3, nh, 1, st); break;
            default: launch<kFuseDiv>(p, geo, tw, sp, n2, n3, nh, 1, st); break;
        }
    }

    template <int MODE>
    static void launch(const X1Ptrs& p, const ColGeom& geo, const c32* tw, const SpecParams& sp, int n2, int n3, int nh,
                       int nfields, hipStream_t st) {
        // At 512 points a column has 32 threads: 8 columns make a block of 256 threads
        // with 64-byte segments, 16 one of 512 with 128-byte segments.  The wide block
        // is better once the launch is bound by memory (multiplier of three fields /
        // gradient, µs: 512³ 1150 -> 915 / 789 -> 654, 512×256×256 394 -> 328 / 194 ->
        // 187), the narrow one below (512×192×192 128 : 132 / 92 : 101, 512×96×96
        // projection 58 : 64).
        if constexpr (N == 512) {
            if (geo.ncols >= kWideX1Columns) return launch_b<MODE, 16>(p, geo, tw, sp, n2, n3, nh, nfields, st);
        }
        launch_b<MODE, Plan<N>::X1>(p, geo, tw, sp, n2, n3, nh, nfields, st);
    }

    template <int MODE, int B>
    static void launch_b(const X1Ptrs& p, const ColGeom& geo, const c32* tw, const SpecParams& sp, int n2, int n3, int nh,
                         int nfields, hipStream_t st) {
        const dim3 grid(static_cast<unsigned>((geo.ncols + B - 1) / B), nfields);
        hipLaunchKernelGGL((k_x1_fused<N, MODE, B>), grid, dim3(X1Geo<N, B>::THREADS), 0, st, p, geo, tw, sp, n2, n3, nh);
    }
};

template <int N>
struct X1Blocks {
    static void go(int64_t ncols, int64_t* blocks) { *blocks = (ncols + X1Geo<N>::B - 1) / X1Geo<N>::B; }
};

template <int N>
struct X1Norm {
    static void go(X1Ptrs p, ColGeom geo, const c32* tw, SpecParams sp, int n2, int n3, int nh, int ncomp, double* partial,
                   hipStream_t st) {
        using G = X1Geo<N>;
        CLR_REQUIRE(geo.ncols * N * 8 < (int64_t(1) << 31), kErrInvalidArgument,
                    "spectrum field too large for 32-bit buffer offsets");
        const dim3 grid(static_cast<unsigned>((geo.ncols + G::B - 1) / G::B), ncomp);
        hipLaunchKernelGGL(k_x1_norm<N>, grid, dim3(G::THREADS), 0, st, p, geo, tw, sp, n2, n3, nh, partial);
    }
};

ColGeom geom_x2(const Dims& d) {
    // columns (i1, k3): cg = i1·nh + k3, start i1·n2·nh + k3, stride nh
    return ColGeom{static_cast<int64_t>(d.n[0]) * d.nh, d.nh, static_cast<int64_t>(d.n[1]) * d.nh, d.nh};
}
ColGeom geom_x1(const Dims& d) {
    // columns (k2, k3): cg = k2·nh + k3, start cg, stride n2·nh
    const int64_t plane = static_cast<int64_t>(d.n[1]) * d.nh;
    return ColGeom{plane, plane, 0, plane};
}

}  // namespace

bool fft_size_supported(int n) {
    return n == 8 || n == 16 || n == 32 || n == 64 || n == 128 || n == 256 || n == 512 || n == 48 || n == 96 ||
           n == 150 || n == 192;
}

void fft_twiddles(int n, c32* h) {
    for (int k = 0; k < n; ++k) {
        const double ang = -2.0 * 3.14159265358979323846 * static_cast<double>(k) / static_cast<double>(n);
        h[k] = {static_cast<float>(std::cos(ang)), static_cast<float>(std::sin(ang))};
    }
}

namespace {
void require_fft_sizes(const Dims& d) {
    for (int a = 0; a < 3; ++a)
        CLR_REQUIRE(fft_size_supported(d.n[a]), kErrUnsupportedSize,
                    "grid size " + std::to_string(d.n[a]) +
                        " not supported (powers of two 8..512, and 48, 96, 150, 192)");
}
}  // namespace

FFTPlan3D::FFTPlan3D(const Dims& d) : dims(d) {
    require_fft_sizes(d);
    for (int a = 0; a < 3; ++a) {
        std::vector<c32> h(d.n[a]);
        fft_twiddles(d.n[a], h.data());
        CLR_HIP_CHECK(hipMalloc(&tw[a], sizeof(c32) * d.n[a]));
        CLR_HIP_CHECK(hipMemcpy(tw[a], h.data(), sizeof(c32) * d.n[a], hipMemcpyHostToDevice));
    }
}

FFTPlan3D::FFTPlan3D(const Dims& d, c32* const tw_ext[3]) : dims(d), owns_tw(false) {
    require_fft_sizes(d);
    for (int a = 0; a < 3; ++a) {
        CLR_REQUIRE(tw_ext[a] != nullptr, kErrInvalidArgument, "missing twiddle table");
        tw[a] = tw_ext[a];
    }
}

FFTPlan3D::~FFTPlan3D() {
    if (!owns_tw) return;
    for (int a = 0; a < 3; ++a)
        if (tw[a]) (void)hipFree(tw[a]);
}

void FFTPlan3D::x3_r2c(const float* in, int64_t is, c32* out, int64_t os, int n, hipStream_t st) const {
    CLR_REQUIRE(n >= 1 && n <= kMaxFields, kErrInvalidArgument, "1 to 65535 fields per FFT pass");
    const R2CPtrs p{in, is, out, os};
    dispatch_n<RowR2C>(dims.n[2], p, n, static_cast<int64_t>(dims.n[0]) * dims.n[1], tw[2], st);
}
void FFTPlan3D::x3_c2r(const c32* in, int64_t is, float* out, int64_t os, int n, hipStream_t st, float alpha,
                       const float* add, int64_t as, float beta) const {
    CLR_REQUIRE(n >= 1 && n <= kMaxFields, kErrInvalidArgument, "1 to 65535 fields per FFT pass");
    const C2RPtrs p{in, is, out, os, add, as};
    dispatch_n<RowC2R>(dims.n[2], p, n, static_cast<int64_t>(dims.n[0]) * dims.n[1], tw[2], alpha, beta, st);
}
void FFTPlan3D::x2(c32* data, int64_t ds, int n, int dir, hipStream_t st) const {
    CLR_REQUIRE(n >= 1 && n <= kMaxFields, kErrInvalidArgument, "1 to 65535 fields per FFT pass");
    const ColPtrs p{data, ds};
    dispatch_n<ColPass>(dims.n[1], p, n, geom_x2(dims), dir, tw[1], st);
}
void FFTPlan3D::x1(c32* data, int dir, hipStream_t st) const {
    const ColPtrs p{data, 0};
    dispatch_n<ColPass>(dims.n[0], p, 1, geom_x1(dims), dir, tw[0], st);
}

void FFTPlan3D::x1_multiplier(c32* data, int64_t ds, int n, const SpecParams& sp, hipStream_t st) const {
    const X1Ptrs p{data, ds, data, ds, 0};
    dispatch_n<X1Fused>(dims.n[0], static_cast<int>(kFuseMult), p, geom_x1(dims), tw[0], sp, dims.n[1], dims.n[2],
                        dims.nh, n, st);
}

int64_t FFTPlan3D::x1_norm_partials(int ncomp) const {
    int64_t blocks = 0;
    dispatch_n<X1Blocks>(dims.n[0], geom_x1(dims).ncols, &blocks);
    return blocks * ncomp;
}

void FFTPlan3D::x1_norm(const c32* in, int64_t is, int n, const SpecParams& sp, double* partial,
                        hipStream_t st) const {
    const X1Ptrs p{in, is, nullptr, 0, 0};
    dispatch_n<X1Norm>(dims.n[0], p, geom_x1(dims), tw[0], sp, dims.n[1], dims.n[2], dims.nh, n, partial, st);
}

void FFTPlan3D::x1_grad(const c32* in, int64_t is, c32* out, int64_t os, int64_t oc, int n, hipStream_t st) const {
    CLR_REQUIRE(n >= 1 && n <= kMaxFields, kErrInvalidArgument, "1 to 65535 fields per FFT pass");
    const X1Ptrs p{in, is, out, os, oc};
    SpecParams sp{};
    sp.scale = dims.scale;
    dispatch_n<X1Fused>(dims.n[0], static_cast<int>(kFuseGrad), p, geom_x1(dims), tw[0], sp, dims.n[1], dims.n[2],
                        dims.nh, n, st);
}

void FFTPlan3D::x1_project(c32* data, int64_t ds, const SpecParams& sp, hipStream_t st) const {
    CLR_REQUIRE(sp.op == kOpProjStokes || sp.op == kOpProjRelaxed, kErrInvalidArgument, "not a projection");
    const X1Ptrs p{data, ds, data, ds, 0};
    dispatch_n<X1Fused>(dims.n[0], static_cast<int>(kFuseProject), p, geom_x1(dims), tw[0], sp, dims.n[1], dims.n[2],
                        dims.nh, 1, st);
}

void FFTPlan3D::x1_div(const c32* in, int64_t is, c32* out, hipStream_t st) const {
    const X1Ptrs p{in, is, out, 0, 0};
    SpecParams sp{};
    sp.scale = dims.scale;
    dispatch_n<X1Fused>(dims.n[0], static_cast<int>(kFuseDiv), p, geom_x1(dims), tw[0], sp, dims.n[1], dims.n[2],
                        dims.nh, 1, st);
}

}  // namespace claire_amd
