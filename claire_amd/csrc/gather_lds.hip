// gather_lds.hip -- LDS-staged semi-Lagrangian gathers and the streaming
// transport kernels of the Hessian matvec (gfx950).
//
// Same arithmetic as the direct gather (tricubic Lagrange weights of
// src/interp3.cpp:2508-2533 on the rescaled plan points, modular ghost
// indexing), but the field is read through LDS:
//
//   * a block owns a 16 (x2) × 32 or 64 (x3) tile of output points and
//     marches along x1 over a chunk of planes ("2.5D" streaming), the chunk
//     length chosen per launch so that the blocks fill whole rounds of the
//     GPU;
//   * LDS holds a ring of input planes, each the tile plus a halo of D+1
//     (low side) and D+2 (high side) cells in x2 and x3, where D is the exact
//     per-axis stencil displacement bound of the plan (D <= 2 covers CFL 2),
//     so every stencil of the tile lies inside the ring by construction; larger
//     displacements, and raw query points, take windows centred per block on
//     large grids, and the points outside them are read from global memory (see
//     PointMode; centred_windows and launch_points_gather say when);
//   * the ring has one spare slot: while the block evaluates plane x1 the
//     global loads of plane x1+D+3 and of the next plane's query points are
//     in flight and land in the spare slot / registers afterwards, so each
//     plane costs one barrier and no exposed HBM latency;
//   * every input element is read from HBM/L2 once per (tile, chunk); the 64
//     stencil values per point come from LDS (ds_read2_b32 pairs).
// Blocks are remapped so that each XCD streams one contiguous range of
// tiles and keeps the shared halo rows in its own L2.
#include <algorithm>
#include <cstdlib>
#include <limits>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "gather_device.hpp"

namespace claire_amd {

namespace {

using namespace gather;

constexpr int kLT2 = 16;        // tile extent in x2
constexpr int kLThreads = 512;  // 8 waves; wave w covers tile rows 2w and 2w+1

// LDS plane geometry of the one-value layout for displacement bound D.  A plane
// holds E2 rows of E3 valid columns at a row pitch that is a multiple of 32
// dwords: a wave reads two tile rows of 32 points each (one row per half-wave),
// so lanes whose stencils start on different rows or planes still hit different
// banks unless their columns collide mod 32.
//   D <= 2: a 16 × 32 tile, one point per thread, 53 KB of LDS -- three
//           blocks (24 waves) per CU;
//   D <= 4: a 16 × 64 tile, two points per thread 32 columns apart, 135 KB.
template <int D>
struct LdsGeo {
    static constexpr int LT3 = (D <= 2) ? 32 : 64;  // tile extent in x3
    static constexpr int PTS = LT3 / 32;             // points per thread and plane
    static constexpr int WAVES_PER_EU = (D <= 2) ? 6 : 2;
    static constexpr int HLO = D + 1, HHI = D + 2;
    static constexpr int E2 = kLT2 + HLO + HHI, E3 = LT3 + HLO + HHI;
    static constexpr int PITCH = (E3 + 31) / 32 * 32;
    static constexpr int P = E2 * PITCH;       // dwords per LDS plane
    static constexpr int NV = E2 * E3;         // valid elements per plane
    static constexpr int WIN = HLO + HHI + 1;  // planes read while evaluating one output plane
    static constexpr int W = WIN + 1;          // ring slots (one spare for the prefetch)
    static constexpr int FILL = (NV + kLThreads - 1) / kLThreads;
};

__device__ __forceinline__ int pmod(int a, int n) {
    int r = a % n;
    return r < 0 ? r + n : r;
}

// Raw buffer accesses: a 32-bit per-lane byte offset plus a uniform byte
// offset (the plane), against a resource that bounds the array (reads past
// it return 0, writes past it are dropped).  Word 3 of a gfx9 raw buffer
// resource: 32-bit data, no swizzle.
using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr int kBufferWord3 = 0x00020000;

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), kBufferWord3);
}
// Cache policy of the buffer loads: 0 for the field planes (neighbouring
// tiles re-read their halo rows from L2), kNonTemporal for the plan words and
// the per-point coefficients, which are read once.
constexpr int kNonTemporal = 2;
__device__ __forceinline__ float bload(rsrc_t r, uint32_t voff, uint32_t soff) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ float bload_once(rsrc_t r, uint32_t voff, uint32_t soff) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, kNonTemporal));
}
__device__ __forceinline__ void bstore(rsrc_t r, float v, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, voff, soff, 0);
}
__device__ __forceinline__ PlanPt bload_plan(rsrc_t r, uint32_t voff, uint32_t soff) {
    typedef unsigned int u3 __attribute__((ext_vector_type(3)));
    const u3 w = __builtin_amdgcn_raw_buffer_load_b96(r, voff, soff, kNonTemporal);
    PlanPt p;
    p.w[0] = w.x;
    p.w[1] = w.y;
    p.w[2] = w.z;
    return p;
}

// Keeps the compiler from splitting an LDS base address into a register part
// plus a constant too large for the ds_read2 offset fields; the stencil's row
// and column offsets then all fit the instruction's immediates.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

template <class Epi>
__device__ __forceinline__ float* out2_of(const Epi& e) {
    if constexpr (Epi::kOut2)
        return e.outp2();
    else
        return e.outp();
}

template <int D, class Epi>
__global__ __launch_bounds__(kLThreads) __attribute__((amdgpu_waves_per_eu(LdsGeo<D>::WAVES_PER_EU))) void k_gather_lds(
    GatherDims g, const PlanPt* __restrict__ plan, const float* __restrict__ fbase, int64_t fzstride, Epi epi,
    int nblocks, int chunk) {
    using G = LdsGeo<D>;
    constexpr int PTS = G::PTS;
    __shared__ float lds[G::W * G::P];
    const int tid = threadIdx.x;
    const int nt3 = (g.n3 + G::LT3 - 1) / G::LT3;
    const int nt2 = (g.n2 + kLT2 - 1) / kLT2;
    // one block per (tile, chunk, field), a tile's fields adjacent (as in
    // k_gather_lds_pair)
    const int nz = static_cast<int>(gridDim.x) / nblocks;
    const int Lz = xcd_remap(blockIdx.x, nblocks * nz);
    const int z = Lz % nz;
    const int L = Lz / nz;
    const int t3 = L % nt3;
    const int t2 = (L / nt3) % nt2;
    const int ch = L / (nt3 * nt2);
    const float* f = fbase + static_cast<int64_t>(z) * fzstride;
    epi.select(z);
    // Byte sizes fit 32 bits: the host requires nl < 2^28 (12 B per point).
    const uint32_t fbytes = static_cast<uint32_t>(g.nl) * 4u;
    const rsrc_t rf = make_rsrc(f, fbytes);
    const rsrc_t rp = make_rsrc(plan, 3u * fbytes);
    const rsrc_t ra = make_rsrc(Epi::kHasAux ? epi.auxp() : f, fbytes);
    const rsrc_t ro = make_rsrc(epi.outp(), fbytes);
    const rsrc_t ro2 = make_rsrc(out2_of(epi), fbytes);
    const uint32_t plane4 = static_cast<uint32_t>(g.n2) * static_cast<uint32_t>(g.n3) * 4u;  // bytes per plane
    const int x1s = ch * chunk;
    const int x1e = min(x1s + chunk, g.n1);
    const int r2 = t2 * kLT2 - G::HLO;
    const int r3 = t3 * G::LT3 - G::HLO;

    // Offsets (within a global plane and within an LDS plane) of the tile
    // elements this thread loads; elements past the tile reload element
    // NV−1 (never stored).
    uint32_t foff[G::FILL];
    int loff[G::FILL];
#pragma unroll
    for (int k = 0; k < G::FILL; ++k) {
        const int e = min(tid + kLThreads * k, G::NV - 1);
        const int e2 = e / G::E3;
        const int e3 = e - e2 * G::E3;
        foff[k] = 4u * static_cast<uint32_t>(pmod(r2 + e2, g.n2) * g.n3 + pmod(r3 + e3, g.n3));  // bytes
        loff[k] = e2 * G::PITCH + e3;
    }

    // This thread's two output points within a plane: wave w covers tile rows
    // 2w and 2w+1, 32 columns each, and the two points are 32 columns apart.
    // Invalid points load point 0 of the plane and skip the store.  rc4 is
    // the byte offset of the point's own cell in an LDS plane.
    const int lane = tid & 63;
    const int lx2 = 2 * (tid >> 6) + (lane >> 5);
    const int x2 = t2 * kLT2 + lx2;
    uint32_t off[PTS];
    int rc4[PTS];
    bool valid[PTS];
    int x3s[PTS];
#pragma unroll
    for (int k = 0; k < PTS; ++k) {
        const int lx3 = (lane & 31) + 32 * k;
        const int x3 = t3 * G::LT3 + lx3;
        x3s[k] = x3;
        valid[k] = x2 < g.n2 && x3 < g.n3;
        off[k] = valid[k] ? 4u * static_cast<uint32_t>(x2 * g.n3 + x3) : 0u;  // bytes of a float
        rc4[k] = 4 * ((lx2 + G::HLO) * G::PITCH + lx3 + G::HLO);
    }

    // prologue: planes x1s−HLO … x1s+HHI into ring slots 0 … WIN−1, and the
    // query points of plane x1s
    // All loads of the prologue are issued before the first one is landed:
    // landing each plane before loading the next costs a memory round trip
    // per plane, which no other block hides on a small grid (measured for the
    // pair kernel below).
    {
        float pro[G::WIN][G::FILL];
        int xw = pmod(x1s - G::HLO, g.n1);
#pragma unroll
        for (int k = 0; k < G::WIN; ++k) {
            const uint32_t src = static_cast<uint32_t>(xw) * plane4;
            xw = (xw + 1 == g.n1) ? 0 : xw + 1;
#pragma unroll
            for (int q = 0; q < G::FILL; ++q) pro[k][q] = bload(rf, foff[q], src);
        }
#pragma unroll
        for (int k = 0; k < G::WIN; ++k)
#pragma unroll
            for (int q = 0; q < G::FILL; ++q)
                if (tid + kLThreads * q < G::NV) lds[k * G::P + loff[q]] = pro[k][q];
    }
    // Query points of plane x1 live in (qa, aa) or (qb, ab); the loop below
    // alternates the two so that the prefetch of the next plane's points
    // needs no register copies.
    PlanPt qa[PTS], qb[PTS];
    float aa[PTS], ab[PTS];
    {
        const uint32_t pb = static_cast<uint32_t>(x1s) * plane4;
#pragma unroll
        for (int k = 0; k < PTS; ++k) {
            qa[k] = bload_plan(rp, 3u * off[k], 3u * pb);
            aa[k] = Epi::kHasAux ? bload_once(ra, off[k], pb) : 0.0f;
        }
    }
    __syncthreads();

    constexpr int P4 = 4 * G::P;  // bytes per ring slot
    const char* ldsb = reinterpret_cast<const char*>(lds);
    int cs = 0;  // ring slot of plane x1 − HLO
    // Input planes are loaded two steps before they are landed: step x1
    // lands plane x1 + HHI + 1 (in pa or pb, loaded by step x1 − 1) and
    // loads plane x1 + HHI + 2 into the other set.
    float pa[G::FILL], pb2[G::FILL];
    {
        const uint32_t src = static_cast<uint32_t>(pmod(x1s + G::HHI + 1, g.n1)) * plane4;
#pragma unroll
        for (int q = 0; q < G::FILL; ++q) pa[q] = bload(rf, foff[q], src);
    }
    // periodic index of plane x1 + HHI + 2, advanced by one per step (a
    // scalar modulo per step costs about 20 scalar instructions)
    int xf = pmod(x1s + G::HHI + 2, g.n1);
    auto step = [&](int x1, const PlanPt (&cur)[PTS], const float (&caux)[PTS], PlanPt (&nxt)[PTS],
                    float (&naux)[PTS], const float (&pre)[G::FILL], float (&pnext)[G::FILL]) {
        // Prefetch for the next steps, unconditionally (past the chunk end it
        // reloads a plane of this chunk; the values are never used).
        const int xn = (x1 + 1 < x1e) ? x1 + 1 : x1;
        {
            const uint32_t src = static_cast<uint32_t>(xf) * plane4;
            xf = (xf + 1 == g.n1) ? 0 : xf + 1;
#pragma unroll
            for (int q = 0; q < G::FILL; ++q) pnext[q] = bload(rf, foff[q], src);
        }
        {
            const uint32_t pb = static_cast<uint32_t>(xn) * plane4;
#pragma unroll
            for (int k = 0; k < PTS; ++k) {
                nxt[k] = bload_plan(rp, 3u * off[k], 3u * pb);
                naux[k] = Epi::kHasAux ? bload_once(ra, off[k], pb) : 0.0f;
            }
        }

        // Stencils: weights and the LDS byte addresses of rows 0 and 3 of the
        // four planes of each point.  The plan's bound keeps every offset
        // within the ring; the clamps only pin LDS addresses inside the
        // allocation.
        float w1[PTS][4], w2[PTS][4], w3[PTS][4];
        int base[PTS][4], base3[PTS][4];
#pragma unroll
        for (int k = 0; k < PTS; ++k) {
            lagrange_weights(plan_t(cur[k].w[0]), w1[k]);
            lagrange_weights(plan_t(cur[k].w[1]), w2[k]);
            lagrange_weights(plan_t(cur[k].w[2]), w3[k]);
            const int lb4 = min(max(rc4[k] + plan_off(cur[k].w[1]) * (4 * G::PITCH) + 4 * plan_off(cur[k].w[2]), 0),
                                4 * (G::P - 3 * G::PITCH - 4));
            int sw = min(max(cs + G::HLO + plan_off(cur[k].w[0]), 0), 2 * G::W - 4);
            sw -= (sw >= G::W) ? G::W : 0;  // ring slot of the first stencil plane
            base[k][0] = opaque(sw * P4 + lb4);
#pragma unroll
            for (int a = 1; a < 4; ++a) base[k][a] = opaque(base[k][a - 1] + ((sw + a == G::W) ? P4 - G::W * P4 : P4));
            // rows 0-2 fit the 8-bit dword offsets of ds_read2_b32 from base;
            // row 3 (3·PITCH + 3 dwords away) needs its own base
#pragma unroll
            for (int a = 0; a < 4; ++a) base3[k][a] = opaque(base[k][a] + 3 * 4 * G::PITCH);
        }
        float v[PTS];
#pragma unroll
        for (int k = 0; k < PTS; ++k) v[k] = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            float sa[PTS];
#pragma unroll
            for (int k = 0; k < PTS; ++k) sa[k] = 0.f;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
#pragma unroll
                for (int k = 0; k < PTS; ++k) {
                    const float* p = (b < 3) ? reinterpret_cast<const float*>(ldsb + base[k][a]) + b * G::PITCH
                                             : reinterpret_cast<const float*>(ldsb + base3[k][a]);
                    // spelled out: left to the compiler, one row of the second point
                    // of the bound-4 kernel was summed in another order
                    sa[k] = fmaf(w2[k][b], row_sum(w3[k], p[0], p[1], p[2], p[3]), sa[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < PTS; ++k) v[k] = fmaf(w1[k][a], sa[k], v[k]);
        }
        {
            const uint32_t pb = static_cast<uint32_t>(x1) * plane4;
#pragma unroll
            for (int k = 0; k < PTS; ++k) {
                if (!valid[k]) continue;
                if constexpr (Epi::kCoord)
                    bstore(ro, epi.apply_at(v[k], caux[k], x1, x2, x3s[k]), off[k], pb);
                else
                    bstore(ro, epi.apply(v[k], caux[k]), off[k], pb);
                if constexpr (Epi::kOut2) bstore(ro2, epi.apply2(v[k], caux[k]), off[k], pb);
            }
        }

        // land the prefetched plane (x1 + HHI + 1) in the spare ring slot
        const int spare = (cs == 0) ? G::W - 1 : cs - 1;
        float* dst = lds + spare * G::P;
#pragma unroll
        for (int q = 0; q < G::FILL; ++q)
            if (tid + kLThreads * q < G::NV) dst[loff[q]] = pre[q];
        cs = (cs + 1 == G::W) ? 0 : cs + 1;
        __syncthreads();
    };

    int x1 = x1s;
    for (; x1 + 1 < x1e; x1 += 2) {
        step(x1, qa, aa, qb, ab, pa, pb2);
        step(x1 + 1, qb, ab, qa, aa, pb2, pa);
    }
    if (x1 < x1e) step(x1, qa, aa, qb, ab, pa, pb2);
}

// Pair layout, D = 2 around a centre.  Entry c of an LDS row holds the two consecutive
// values (f[c], f[c+1]) of the tile row, so the four values of a stencil row
// starting at column c are the 8-byte entries c and c + 2: one ds_read2_b64
// per stencil row instead of two ds_read2_b32, with no alignment condition
// on c.  The price is twice the LDS per plane.  A block keeps a ring of
// W = WIN + 2·PERIOD − 1 planes and synchronizes once per PERIOD = 2 output
// planes (the planes of two consecutive stencil windows stay resident while
// the next two are landed in slots neither window reads): 11 planes of a
// 16 × 32 tile with its halo at a row pitch of 80 dwords take 79.1 KB, two
// blocks (16 waves) per CU.  The pitch of 96 dwords that a one-plane period
// affords has a third of the bank conflicts (8 k against 22 k cycles per CU
// and launch at 256³), but the halved barriers gain more (adjoint step
// 107.2 → 105.1 µs; at one plane per barrier the pitch of 80 alone costs
// 6 µs).
struct PairGeo {
    static constexpr int D = 2;
    static constexpr int LT3 = 32;
    static constexpr int WAVES_PER_EU = 4;
    static constexpr int HLO = D + 1, HHI = D + 2;
    static constexpr int E2 = kLT2 + HLO + HHI, E3 = LT3 + HLO + HHI;
    static constexpr int NE3 = E3 - 1;                   // entries per row (the last column only fills entry E3 − 2)
    static constexpr int PITCH = (2 * NE3 + 15) / 16 * 16;  // dwords per row
    static constexpr int P = E2 * PITCH;                 // dwords per LDS plane
    static constexpr int NV = E2 * NE3;                  // entries per plane
    static constexpr int WIN = HLO + HHI + 1;            // planes of one output plane's stencils
    static constexpr int PERIOD = 2;                     // output planes per barrier
    static constexpr int W = WIN + 2 * PERIOD - 1;       // ring slots
    static constexpr int FILL = (NV + kLThreads - 1) / kLThreads;
    // every ds_read2_b64 of a stencil (rows 0-3, entries c and c + 2) is
    // within the instruction's 8-bit offsets (in 8-byte units) of the base
    static_assert((3 * 4 * PITCH + 16) / 8 <= 255, "row 3 out of ds_read2_b64 offset range");
    // the kernel's steps are unrolled by four and barriers close periods
    static_assert(4 % PERIOD == 0, "the period must divide the unroll of four");
    // two blocks (16 waves) per CU in the 160 KB of LDS
    static_assert(2 * W * P * 4 <= 160 * 1024, "ring too large for two blocks per CU");
};

// Which points a launch takes:
//   kPtsNear  plan words with a bound D <= 2: every stencil lies in the window;
//   kPtsPlan  plan words of any displacement;
//   kPtsRaw   raw query points (3 floats per point over 2π, any value), turned
//             into plan words as they are used.
// For the last two the window of a block is centred on the mean offset of a
// sample of its points (a smooth deformation is nearly rigid over a tile), and a
// point whose stencil is not inside reads it from global memory, in the
// arithmetic of the direct kernels.  A block with less than 60% of its sample
// inside (scattered points) stages nothing and takes the direct way throughout:
// with 75% the gather at points of 256³ moved by noise of ±2.5 cells took 599 µs,
// 556 with 60, and for ±3 cells 601, 655 with 60.
enum PointMode { kPtsNear = 0, kPtsPlan = 1, kPtsRaw = 2 };
// most planes per block of the last two (one bit of a mask each; raw points keep
// to 32 bits and to input planes one step ahead, or the kernel runs out of
// registers)
constexpr int far_chunk(int mode) { return mode == kPtsRaw ? 32 : 64; }

template <class Epi, int MODE>
__global__ __launch_bounds__(kLThreads) __attribute__((amdgpu_waves_per_eu(PairGeo::WAVES_PER_EU))) void
k_gather_lds_pair(GatherDims g, HH hh, const PlanPt* __restrict__ plan, const float* __restrict__ fbase,
                  int64_t fzstride, Epi epi, int nblocks, int chunk) {
    using G = PairGeo;
    __shared__ __align__(16) float lds[G::W * G::P];
    const int tid = threadIdx.x;
    const int nt3 = (g.n3 + G::LT3 - 1) / G::LT3;
    const int nt2 = (g.n2 + kLT2 - 1) / kLT2;
    // One block per (tile, chunk, field) on a 1D grid.  The fields of a tile
    // are neighbours in each XCD's range, so the plan words one of them loads
    // are L2 hits for the others (three-field gather at 256³ 288.0 -> 285.4
    // µs, outputs identical).
    const int nz = static_cast<int>(gridDim.x) / nblocks;
    const int Lz = xcd_remap(blockIdx.x, nblocks * nz);
    const int z = Lz % nz;
    const int L = Lz / nz;
    const int t3 = L % nt3;
    const int t2 = (L / nt3) % nt2;
    const int ch = L / (nt3 * nt2);
    const float* f = fbase + static_cast<int64_t>(z) * fzstride;
    epi.select(z);
    const uint32_t fbytes = static_cast<uint32_t>(g.nl) * 4u;
    const rsrc_t rf = make_rsrc(f, fbytes);
    const rsrc_t rp = make_rsrc(plan, 3u * fbytes);
    const rsrc_t ra = make_rsrc(Epi::kHasAux ? epi.auxp() : f, fbytes);
    const rsrc_t ro = make_rsrc(epi.outp(), fbytes);
    const rsrc_t ro2 = make_rsrc(out2_of(epi), fbytes);
    const uint32_t plane4 = static_cast<uint32_t>(g.n2) * static_cast<uint32_t>(g.n3) * 4u;
    const int x1s = ch * chunk;
    const int x1e = min(x1s + chunk, g.n1);
    // Wave w covers tile rows 2w and 2w + 1, 32 columns each.
    struct Column {
        int lx2, lx3, x2, x3;
        bool valid;
        uint32_t off;  // bytes of a float within a plane (0 where not valid)
    };
    auto column = [&](int t) {
        Column c;
        c.lx2 = 2 * (t >> 6) + ((t & 63) >> 5);
        c.lx3 = t & 31;
        c.x2 = t2 * kLT2 + c.lx2;
        c.x3 = t3 * G::LT3 + c.lx3;
        c.valid = c.x2 < g.n2 && c.x3 < g.n3;
        c.off = c.valid ? 4u * static_cast<uint32_t>(c.x2 * g.n3 + c.x3) : 0u;
        return c;
    };
    const int lane = tid & 63;
    const Column me = column(tid);

    // Plan words of a loaded point of plane x1; false when a raw point has none
    // (a coordinate that is not finite).
    auto decode = [&](const PlanPt& p, int x1, const Column& c, uint32_t (&w)[3]) {
        if constexpr (MODE != kPtsRaw) {
            w[0] = p.w[0];
            w[1] = p.w[1];
            w[2] = p.w[2];
            return true;
        } else {
            int o;
            w[0] = w[1] = w[2] = 0u;
            const bool a = plan_encode(index_coord(__uint_as_float(p.w[0]), g.n1, hh.h[0]), x1, g.n1, w[0], o);
            const bool b = plan_encode(index_coord(__uint_as_float(p.w[1]), g.n2, hh.h[1]), c.x2, g.n2, w[1], o);
            const bool e = plan_encode(index_coord(__uint_as_float(p.w[2]), g.n3, hh.h[2]), c.x3, g.n3, w[2], o);
            return a && b && e;
        }
    };
    auto store_point = [&](int x1, const Column& c, float v, float a) {
        const uint32_t pb = static_cast<uint32_t>(x1) * plane4;
        if constexpr (Epi::kCoord)
            bstore(ro, epi.apply_at(v, a, x1, c.x2, c.x3), c.off, pb);
        else
            bstore(ro, epi.apply(v, a), c.off, pb);
        if constexpr (Epi::kOut2) bstore(ro2, epi.apply2(v, a), c.off, pb);
    };
    // a point of plane x1 read straight from global memory, and stored
    auto direct_point = [&](int x1, const Column& c) {
        const uint32_t pb = static_cast<uint32_t>(x1) * plane4;
        const PlanPt p = bload_plan(rp, 3u * c.off, 3u * pb);
        const float a = Epi::kHasAux ? bload_once(ra, c.off, pb) : 0.0f;
        Stencil st;
        if constexpr (MODE == kPtsRaw) {
            const float q[3] = {__uint_as_float(p.w[0]), __uint_as_float(p.w[1]), __uint_as_float(p.w[2])};
            setup_stencil(q, g, hh.h, st);
        } else {
            plan_stencil(p.w, x1, c.x2, c.x3, g, st);
        }
        const float* fs[1] = {f};
        float r[1];
        eval_stencil<1>(fs, st, g, r);
        store_point(x1, c, r[0], a);
    };
    // Window: stencil offsets o with o − c in [−D − 1, D − 1] on every axis.
    int c1 = 0, c2 = 0, c3 = 0;
    auto in_window = [&](const uint32_t (&w)[3]) {
        return static_cast<uint32_t>(plan_off(w[0]) - c1 + G::D + 1) <= 2u * G::D &&
               static_cast<uint32_t>(plan_off(w[1]) - c2 + G::D + 1) <= 2u * G::D &&
               static_cast<uint32_t>(plan_off(w[2]) - c3 + G::D + 1) <= 2u * G::D;
    };
    if constexpr (MODE != kPtsNear) {
        // sample: this thread's column at a quarter and three quarters of the chunk
        uint32_t w[2][3];
        bool ok[2];
        PlanPt p[2];
        const int xs[2] = {x1s + (x1e - x1s) / 4, x1s + 3 * (x1e - x1s) / 4};
#pragma unroll
        for (int k = 0; k < 2; ++k) p[k] = bload_plan(rp, 3u * me.off, 3u * (static_cast<uint32_t>(xs[k]) * plane4));
        int m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            ok[k] = decode(p[k], xs[k], me, w[k]) && me.valid;
            if (ok[k]) {
                m[0] += plan_off(w[k][0]);
                m[1] += plan_off(w[k][1]);
                m[2] += plan_off(w[k][2]);
                m[3] += 1;
            }
        }
        int* sh = reinterpret_cast<int*>(lds);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) m[a] += __shfl_xor(m[a], o, 64);
            if (lane == 0) sh[4 * (tid >> 6) + a] = m[a];
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            m[a] = 0;
#pragma unroll
            for (int k = 0; k < kLThreads / 64; ++k) m[a] += sh[4 * k + a];
        }
        const float inv = 1.0f / static_cast<float>(max(m[3], 1));
        // offsets of −1 (a point on its own node's cell) sit at the window's middle
        c1 = __builtin_amdgcn_readfirstlane(__float2int_rn(static_cast<float>(m[0]) * inv)) + 1;
        c2 = __builtin_amdgcn_readfirstlane(__float2int_rn(static_cast<float>(m[1]) * inv)) + 1;
        c3 = __builtin_amdgcn_readfirstlane(__float2int_rn(static_cast<float>(m[2]) * inv)) + 1;
        const int mine = __popcll(__ballot(ok[0] && in_window(w[0]))) + __popcll(__ballot(ok[1] && in_window(w[1])));
        if (lane == 0) sh[64 + (tid >> 6)] = mine;
        __syncthreads();
        int inside = 0;
#pragma unroll
        for (int k = 0; k < kLThreads / 64; ++k) inside += sh[64 + k];
        __syncthreads();  // the staging below reuses sh
        if (5 * __builtin_amdgcn_readfirstlane(inside) < 3 * __builtin_amdgcn_readfirstlane(m[3])) {
            if (me.valid)
                for (int x = x1s; x < x1e; ++x) direct_point(x, me);
            return;
        }
    }
    const int r2 = t2 * kLT2 - G::HLO + c2;
    const int r3 = t3 * G::LT3 - G::HLO + c3;
    const int xw0 = x1s - G::HLO + c1;  // the first input plane

    // Entries this thread fills: the byte offsets (within a global plane) of
    // the entry's two values and the entry's dword offset in an LDS plane.
    // Entries past the plane reload entry NV−1 (never stored).
    uint32_t foff[G::FILL][2];
    int loff[G::FILL];
#pragma unroll
    for (int k = 0; k < G::FILL; ++k) {
        const int e = min(tid + kLThreads * k, G::NV - 1);
        const int e2 = e / G::NE3;
        const int e3 = e - e2 * G::NE3;
        const int row = pmod(r2 + e2, g.n2) * g.n3;
        foff[k][0] = 4u * static_cast<uint32_t>(row + pmod(r3 + e3, g.n3));
        foff[k][1] = 4u * static_cast<uint32_t>(row + pmod(r3 + e3 + 1, g.n3));
        loff[k] = e2 * G::PITCH + 2 * e3;
    }

    // byte offset of the point's own cell (its entry) in an LDS plane, less the
    // window's centre
    const int rc = 4 * ((me.lx2 + G::HLO - c2) * G::PITCH + 2 * (me.lx3 + G::HLO - c3));

    auto store2 = [&](float* dst, int q, float a, float b) {
        *reinterpret_cast<float2*>(dst + loff[q]) = make_float2(a, b);
    };
    // Loads run ahead of their use: while plane x1 is evaluated, the plan
    // words (and the epilogue operand) of plane x1 + LA_PT and the input
    // plane x1 + HHI + PERIOD + LA_PL are issued.  Q[k & 3] / A[k & 3] hold
    // the plan words and operand of step k; PRE[k % NPRE] the input plane
    // that step k lands in a free ring slot.  Measured at 256³ (outputs
    // identical): plane loads two steps ahead instead of one take the steps
    // from 104.5 to 103.7 µs for 8 more VGPRs (123); plan words three steps
    // ahead instead of two are slower (105 µs).
    constexpr int LA_PT = 2;  // steps between a plan word load and its use
    constexpr int LA_PL = MODE == kPtsRaw ? 1 : 2;  // steps between an input plane load and its landing
    constexpr int NPRE = (LA_PL == 1) ? 2 : 4;
    PlanPt Q[4];
    float A[4];
    float PRE[NPRE][G::FILL][2];
    auto load_point = [&](int x, PlanPt& q, float& a) {
        const int xc = min(x, x1e - 1);  // past the chunk end: a plane of this chunk, never used
        const uint32_t pb = static_cast<uint32_t>(xc) * plane4;
        q = bload_plan(rp, 3u * me.off, 3u * pb);
        a = Epi::kHasAux ? bload_once(ra, me.off, pb) : 0.0f;
    };
    auto load_plane = [&](int xw, float (&pre)[G::FILL][2]) {  // xw: plane index in [0, n1)
        const uint32_t src = static_cast<uint32_t>(xw) * plane4;
#pragma unroll
        for (int q = 0; q < G::FILL; ++q) {
            pre[q][0] = bload(rf, foff[q][0], src);
            pre[q][1] = bload(rf, foff[q][1], src);
        }
    };
    // prologue: input planes x1s − HLO … x1s + HHI + PERIOD − 1 (the stencils
    // of the first PERIOD output planes) into ring slots 0 … WIN + PERIOD − 2
    // with all loads issued before the first one is landed (36 registers,
    // free until the main loop).  Landed one by one, as 18 dependent memory
    // round trips, the prologue was most of a short block's time: one-field
    // gather at 64³ 9.2 -> 8.1 µs, at 256³ (32 planes) 94.8 -> 89.4 µs; matvec at
    // 64³ 149.7 -> 122.8 µs, at 256³ 2.01 -> 1.95 ms; outputs identical.
    {
        constexpr int NPRO = G::WIN + G::PERIOD - 1;
        float pro[NPRO][G::FILL][2];
        int xw = pmod(xw0, g.n1);
#pragma unroll
        for (int k = 0; k < NPRO; ++k) {
            load_plane(xw, pro[k]);
            xw = (xw + 1 == g.n1) ? 0 : xw + 1;
        }
#pragma unroll
        for (int k = 0; k < NPRO; ++k)
#pragma unroll
            for (int q = 0; q < G::FILL; ++q)
                if (tid + kLThreads * q < G::NV) store2(lds + k * G::P, q, pro[k][q][0], pro[k][q][1]);
    }
    for (int k = 0; k < LA_PT; ++k) load_point(x1s + k, Q[k], A[k]);
    for (int k = 0; k < LA_PL; ++k) load_plane(pmod(xw0 + G::HLO + G::HHI + G::PERIOD + k, g.n1), PRE[k]);
    // periodic index of the input plane the next step loads, advanced by one
    // per step (a scalar modulo per step costs about 20 scalar instructions)
    int xf = pmod(xw0 + G::HLO + G::HHI + G::PERIOD + LA_PL, g.n1);
    __syncthreads();

    constexpr int P4 = 4 * G::P;
    constexpr uint32_t kLast = 4u * (G::W * G::P - 3 * G::PITCH - 6);  // last address a stencil plane can start at
    const char* ldsb = reinterpret_cast<const char*>(lds);
    uint32_t cs4 = G::HLO * P4;  // (ring slot of plane x1 - HLO, plus HLO)·P4
    // Stencil rows kept in registers across output planes.  A point's
    // stencil spans input planes x1 + o1 … x1 + o1 + 3; when the next plane's
    // point has the same offsets (o1, o2, o3) -- about 95% of points on a
    // CFL-2 trajectory -- its planes 0..2 are this point's planes 1..3, so
    // only its plane 3 is read from LDS.  S[k & 3] holds the rows of the
    // plane that step k reads as its plane 3; step k's plane a lives in
    // S[(k + a) & 3], which is the set step k + 1 uses for plane a − 1.
    // Lanes whose offsets changed (and every lane on a chunk's first plane)
    // read all four planes.  The values and their order of summation are
    // those of the LDS reads, so results are unchanged bit for bit.
    float2 S[4][4][2];
    int prev_key = std::numeric_limits<int>::min();
    // planes of the chunk whose point of this thread is outside the window
    using Mask = typename std::conditional<(far_chunk(MODE) > 32), uint64_t, uint32_t>::type;
    Mask outside = 0;
    auto step = [&](auto kconst, int x1) {
        constexpr int K = decltype(kconst)::value;
        const PlanPt cur = Q[K & 3];
        const float caux = A[K & 3];
        load_point(x1 + LA_PT, Q[(K + LA_PT) & 3], A[(K + LA_PT) & 3]);
        load_plane(xf, PRE[(K + LA_PL) % NPRE]);  // plane x1 + HHI + PERIOD + LA_PL
        xf = (xf + 1 == g.n1) ? 0 : xf + 1;
        // land input plane x1 + HHI + PERIOD (loaded LA_PL steps earlier) in
        // the slot of plane x1 + HHI + PERIOD − W, which no step between
        // this period's barriers reads.  Landing it before the point's
        // stencil is read, not after the point is stored, lets the writes
        // drain while the point is evaluated, and a wave reaches the
        // period's barrier with no landing pending (measured at 256³,
        // outputs identical: adjoint step 103.9 -> 103.1 µs, three-field
        // gather 289.4 -> 287.3 µs).
        uint32_t spare = cs4 + (G::WIN + G::PERIOD - 1 - G::HLO) * P4;
        spare -= (spare >= G::W * P4) ? G::W * P4 : 0;
        float* dst = lds + spare / 4;
#pragma unroll
        for (int q = 0; q < G::FILL; ++q)
            if (tid + kLThreads * q < G::NV) store2(dst, q, PRE[K % NPRE][q][0], PRE[K % NPRE][q][1]);
        uint32_t word[3];
        bool inside = decode(cur, x1, me, word);
        if constexpr (MODE != kPtsNear) inside = inside && in_window(word);
        float w1[4], w2[4], w3[4];
        lagrange_weights(plan_t(word[0]), w1);
        lagrange_weights(plan_t(word[1]), w2);
        lagrange_weights(plan_t(word[2]), w3);
        // Byte address of the stencil's first row, counted from the ring slot
        // of plane x1 - HLO as if the ring did not end: o1·P4 plus the cell's
        // address within a plane (below P4, so equal keys are equal offsets).
        const int key = (plan_off(word[0]) - c1) * P4 +
                        (rc + plan_off(word[1]) * (4 * G::PITCH) + 8 * plan_off(word[2]));
        const bool reuse = key == prev_key;  // never on a chunk's first plane
        prev_key = key;
        // Stencil plane a starts at x = key + (slot + a)·P4, less the ring's
        // length W·P4 when it has run past the end: as unsigned numbers the
        // smaller of the two.  The third operand of the minimum only pins the
        // address inside the allocation (the plan's bound keeps it there).
        const uint32_t x0 = static_cast<uint32_t>(key) + cs4;
        // 156 instead of 161 vector instructions per point and step against
        // comparing and selecting per plane on ring-slot numbers (one-field
        // gather at 256³ 94.7 -> 94.4 µs, at 128³ 18.8 -> 18.4 µs; 256³ matvec
        // 1.957 -> 1.944 ms; outputs identical): a step waits on LDS more than
        // it issues.
        auto ring = [&](int a) {
            const uint32_t x = x0 + static_cast<uint32_t>(a * P4);
            return opaque(static_cast<int>(min(min(x, x - static_cast<uint32_t>(G::W * P4)), kLast)));
        };
        auto read_plane = [&](int a, float2 (&R)[4][2]) {
            const int base = ring(a);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const char* row = ldsb + base + b * 4 * G::PITCH;
                R[b][0] = *reinterpret_cast<const float2*>(row);
                R[b][1] = *reinterpret_cast<const float2*>(row + 16);
            }
        };
        // The stencil reads are issued at raised wave priority, so that a
        // wave's reads go out ahead of the other waves' contractions and
        // their LDS latency overlaps that work (outputs identical; at 256³
        // adjoint step 103.4 -> 101.1 µs, inc-state step 104.1 -> 101.0 µs,
        // three-field gather 285.6 -> 287.2 µs, matvec +0.9%; priority 3
        // instead of 1, or raised from the landing on, gained no more).
        __builtin_amdgcn_s_setprio(1);
        if (!reuse) {
            read_plane(0, S[K & 3]);
            read_plane(1, S[(K + 1) & 3]);
            read_plane(2, S[(K + 2) & 3]);
        }
        read_plane(3, S[(K + 3) & 3]);
        __builtin_amdgcn_s_setprio(0);
        float v = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            float sa = 0.f;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const float2 lo = S[(K + a) & 3][b][0];
                const float2 hi = S[(K + a) & 3][b][1];
                if constexpr (MODE != kPtsNear || Epi::kRowFrom1)
                    sa += w2[b] * row_sum(w3, lo.x, lo.y, hi.x, hi.y);
                else
                    sa += w2[b] * fmaf(w3[3], hi.y, fmaf(w3[2], hi.x, fmaf(w3[1], lo.y, w3[0] * lo.x)));
            }
            v += w1[a] * sa;
        }
        if constexpr (MODE == kPtsNear) {
            if (me.valid) store_point(x1, me, v, caux);
        } else {
            if (me.valid && inside) store_point(x1, me, v, caux);
            if (__ballot(me.valid && !inside))
                outside |= static_cast<Mask>(me.valid && !inside) << (x1 - x1s);
        }
        cs4 = (cs4 == (G::W - 1 + G::HLO) * P4) ? G::HLO * P4 : cs4 + P4;
        if constexpr (K % G::PERIOD == G::PERIOD - 1) __syncthreads();
    };
    using K0 = std::integral_constant<int, 0>;
    using K1 = std::integral_constant<int, 1>;
    using K2 = std::integral_constant<int, 2>;
    using K3 = std::integral_constant<int, 3>;

    // four planes per trip (the register sets rotate once)
    int x1 = x1s;
    for (; x1 + 3 < x1e; x1 += 4) {
        step(K0{}, x1);
        step(K1{}, x1 + 1);
        step(K2{}, x1 + 2);
        step(K3{}, x1 + 3);
    }
    // the last 0-3 planes continue the rotation
    if (x1 < x1e) step(K0{}, x1);
    if (x1 + 1 < x1e) step(K1{}, x1 + 1);
    if (x1 + 2 < x1e) step(K2{}, x1 + 2);
    // The points outside the window.  They lie together, so a few waves would have
    // most of them, one memory round trip each: they are shared out through the
    // ring's memory.  Where kDense lanes of a wave or more are outside on a plane,
    // the whole group goes to a wave, whose loads stay on neighbouring addresses;
    // the others are listed one by one and fill waves.  (All one by one, a scalar
    // gather along smooth displacements of up to 9 cells at 256³ took 397 µs,
    // shared out 204, by the direct kernel 362; groups of 16 lanes or more 224.
    // Within the steps, the global stencil beside the rows kept for the next
    // plane spills registers.)
    if constexpr (MODE != kPtsNear) {
        static_assert(far_chunk(MODE) <= 8 * static_cast<int>(sizeof(Mask)), "one bit per plane");
        constexpr int kDense = 32, kWaves = kLThreads / 64, kMost = far_chunk(MODE) * kWaves;
        struct Outside {
            int groups, points;
            struct {
                uint64_t lanes;
                int plane, wave;
            } group[kMost];
            int point[(kDense - 1) * kMost];  // plane · kLThreads + thread
        };
        static_assert(sizeof(Outside) <= sizeof(lds), "lists exceed the ring");
        Outside& sh = *reinterpret_cast<Outside*>(lds);
        const int wave = tid >> 6;
        __syncthreads();  // the ring is no longer read
        if (tid == 0) sh.groups = sh.points = 0;
        __syncthreads();
        // one trip per plane on which a lane of this wave is outside
        while (const uint64_t left = __ballot(outside != 0)) {
            const int lowest = __builtin_ctzll(outside | (static_cast<uint64_t>(1) << 63));
            const int k = __builtin_amdgcn_readlane(lowest, __builtin_ctzll(left));
            const bool out = (outside >> k) & 1;
            outside &= ~(static_cast<Mask>(1) << k);
            const uint64_t lanes = __ballot(out);
            if (__popcll(lanes) >= kDense) {
                if (lane == 0) {
                    const int at = atomicAdd(&sh.groups, 1);
                    sh.group[at].lanes = lanes;
                    sh.group[at].plane = k;
                    sh.group[at].wave = wave;
                }
            } else if (out) {
                sh.point[atomicAdd(&sh.points, 1)] = k * kLThreads + tid;
            }
        }
        __syncthreads();
        for (int e = wave; e < sh.groups; e += kWaves)
            if ((sh.group[e].lanes >> lane) & 1) direct_point(x1s + sh.group[e].plane, column(64 * sh.group[e].wave + lane));
        for (int e = tid; e < sh.points; e += kLThreads)
            direct_point(x1s + sh.point[e] / kLThreads, column(sh.point[e] % kLThreads));
    }
}

// Incremental state right-hand sides, streamed with 16-byte accesses:
//   s_j = ht/2·[(∇m^j)(X_s)·ṽ(X_s) + ∇m^{j+1}·ṽ],  j = 0..nt−1
// (the two decrements of src/CLAIRE.cpp:3253-3273);
// writes m̃¹ = −s_0 (λ̃⁰ = s_0 when nt = 1) and s_1..s_{nt−1}.
// 4 consecutive values as float4.
// 16-byte (FP32) or 8-byte (16-bit) streaming loads with the non-temporal
// hint: every element of these arrays is read once per launch, and the hint
// keeps the streams from displacing reusable lines (measured on a read-8,
// write-1 stream at 256³: 5.84 TB/s with the hint, 5.19 TB/s without).
using f4v = float __attribute__((ext_vector_type(4)));
using u2v = unsigned __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float4 ld4(const float* a, int64_t i) {
    const f4v v = __builtin_nontemporal_load(reinterpret_cast<const f4v*>(a) + i);
    return make_float4(v.x, v.y, v.z, v.w);
}

// Sources of the Newton-invariant gradient fields, field k at offset k·nl:
//   SrcF32  FP32 (the plain form);
//   SrcBfp  16-bit block floating point (the mixed form): int16 mantissas
//           with one power-of-two scale per block of 256 consecutive values
//           of a field (kBfpBlock4 float4 groups, one wave of the streaming
//           kernels); value = q·scale exactly.
constexpr int kBfpBlock4 = 64;
struct SrcF32 {
    const float* p;
    __device__ float4 load(int k, int64_t nl, int64_t i) const { return ld4(p + k * nl, i); }
};
struct SrcBfp {
    const int16_t* q;
    const float* s;
    int64_t nblk;  // scale blocks per field
    __device__ float4 load(int k, int64_t nl, int64_t i) const {
        const u2v bits = __builtin_nontemporal_load(reinterpret_cast<const u2v*>(q + k * nl) + i);
        const float sc = s[k * nblk + i / kBfpBlock4];
        const int16_t a = static_cast<int16_t>(bits.x & 0xFFFFu), b = static_cast<int16_t>(bits.x >> 16);
        const int16_t c = static_cast<int16_t>(bits.y & 0xFFFFu), d = static_cast<int16_t>(bits.y >> 16);
        return make_float4(static_cast<float>(a) * sc, static_cast<float>(b) * sc, static_cast<float>(c) * sc,
                           static_cast<float>(d) * sc);
    }
};

template <class Src>
struct RhsP {
    const float* vx[3];
    const float* vt[3];
    Src gX;
    Src gm;
    float* s;
    float* mt1;
};

// Src = SrcF32 (plain) or SrcBfp (mixed form: the Newton-invariant gradient
// fields stored as 16-bit block floating point, accumulated in FP32).
// On large grids each wave of the streaming kernels covers K = 2 consecutive runs of 64
// float4 (1 KB of FP32) of every stream, lane l taking float4 l of each run,
// so each of the 30-odd streams is read in 2 KB bursts.  Measured at 256³
// (outputs identical): k_inc_state_rhs 399 → 367 µs and k_body_force 256 →
// 243 µs with two runs per wave; four runs (227 VGPRs for the right-hand
// sides) were slower than two.  A microbenchmark of 30 read and 4 write
// streams gave 5.6, 6.2 and 6.6 TB/s for one, two and four runs.
__device__ __forceinline__ int64_t stream_base(int k) {
    return static_cast<int64_t>(blockIdx.x) * 256 * k + (threadIdx.x >> 6) * 64 * k + (threadIdx.x & 63);
}

template <class Src, int K>
__global__ __launch_bounds__(256) void k_inc_state_rhs(int64_t nl4, int nt, float hthalf, RhsP<Src> p) {
    const int64_t i0 = stream_base(K);
    const int64_t nl = nl4 * 4;
    float4 x0[K], x1[K], x2[K], v0[K], v1[K], v2[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int64_t i = min(i0 + 64 * k, nl4 - 1);  // past the end: reload the last group, never stored
        x0[k] = ld4(p.vx[0], i); x1[k] = ld4(p.vx[1], i); x2[k] = ld4(p.vx[2], i);
        v0[k] = ld4(p.vt[0], i); v1[k] = ld4(p.vt[1], i); v2[k] = ld4(p.vt[2], i);
    }
    // blockIdx.y selects a group of consecutive time steps (one group on large grids)
    const int jn = (nt + gridDim.y - 1) / gridDim.y, j0 = blockIdx.y * jn, j1 = min(j0 + jn, nt);
    for (int j = j0; j < j1; ++j) {
        float4 a0[K], a1[K], a2[K], c0[K], c1[K], c2[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int64_t i = min(i0 + 64 * k, nl4 - 1);
            a0[k] = p.gX.load(3 * j, nl, i); a1[k] = p.gX.load(3 * j + 1, nl, i); a2[k] = p.gX.load(3 * j + 2, nl, i);
            c0[k] = p.gm.load(3 * (j + 1), nl, i); c1[k] = p.gm.load(3 * (j + 1) + 1, nl, i);
            c2[k] = p.gm.load(3 * (j + 1) + 2, nl, i);
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int64_t i = i0 + 64 * k;
            if (i >= nl4) continue;
            float4 s;
            s.x = hthalf * (a0[k].x * x0[k].x + a1[k].x * x1[k].x + a2[k].x * x2[k].x) +
                  hthalf * (c0[k].x * v0[k].x + c1[k].x * v1[k].x + c2[k].x * v2[k].x);
            s.y = hthalf * (a0[k].y * x0[k].y + a1[k].y * x1[k].y + a2[k].y * x2[k].y) +
                  hthalf * (c0[k].y * v0[k].y + c1[k].y * v1[k].y + c2[k].y * v2[k].y);
            s.z = hthalf * (a0[k].z * x0[k].z + a1[k].z * x1[k].z + a2[k].z * x2[k].z) +
                  hthalf * (c0[k].z * v0[k].z + c1[k].z * v1[k].z + c2[k].z * v2[k].z);
            s.w = hthalf * (a0[k].w * x0[k].w + a1[k].w * x1[k].w + a2[k].w * x2[k].w) +
                  hthalf * (c0[k].w * v0[k].w + c1[k].w * v1[k].w + c2[k].w * v2[k].w);
            if (j == 0) {
                if (nt != 1) s = make_float4(-s.x, -s.y, -s.z, -s.w);
                reinterpret_cast<float4*>(p.mt1)[i] = s;
            } else {
                reinterpret_cast<float4*>(p.s + static_cast<int64_t>(j) * nl)[i] = s;
            }
        }
    }
}

// Body force b_d = hd·Σ_{j=0..nt} w_j·λ^j·∂_d m^{nt−j} with trapezoid weights
// w_0 = w_nt = ht/2, w_j = ht, accumulated in the reference's order
// (src/CLAIRE.cpp:2668-2709 and 3940-3999, scaled by hd at :2341/:3471).
// Streamed with 16-byte accesses; lam holds λ^0..λ^nt.
template <class Src>
struct BodyP {
    const float* lam;
    Src gm;
    float* b[3];
};

template <class Src, int K, int J>
__global__ __launch_bounds__(256) void k_body_force(int64_t nl4, int nt, float ht, float hd, BodyP<Src> p) {
    const int64_t i0 = stream_base(K);
    const int64_t nl = nl4 * 4;
    float4 s[K][3];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) s[k][d] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j0 = 0; j0 <= nt; j0 += J) {  // J time steps in flight
        float4 l[J][K], g[J][K][3];
#pragma unroll
        for (int jj = 0; jj < J; ++jj) {
            const int j = min(j0 + jj, nt);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int64_t i = min(i0 + 64 * k, nl4 - 1);  // past the end: reload the last group, never stored
                l[jj][k] = ld4(p.lam + static_cast<int64_t>(j) * nl, i);
#pragma unroll
                for (int d = 0; d < 3; ++d) g[jj][k][d] = p.gm.load(3 * (nt - j) + d, nl, i);
            }
        }
#pragma unroll
        for (int jj = 0; jj < J; ++jj) {
            const int j = j0 + jj;
            if (j > nt) break;
            const float w = (j == 0 || j == nt) ? 0.5f * ht : ht;
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    s[k][d].x += w * g[jj][k][d].x * l[jj][k].x;
                    s[k][d].y += w * g[jj][k][d].y * l[jj][k].y;
                    s[k][d].z += w * g[jj][k][d].z * l[jj][k].z;
                    s[k][d].w += w * g[jj][k][d].w * l[jj][k].w;
                }
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int64_t i = i0 + 64 * k;
        if (i >= nl4) continue;
#pragma unroll
        for (int d = 0; d < 3; ++d)
            reinterpret_cast<float4*>(p.b[d])[i] =
                make_float4(s[k][d].x * hd, s[k][d].y * hd, s[k][d].z * hd, s[k][d].w * hd);
    }
}

// FP32 → 16-bit block floating point, field blockIdx.y, 4 values per thread.
// A wave (64 threads, 256 values) shares one scale 2^(E−15), E the binary
// exponent of its largest magnitude (max |v| < 2^E), so every mantissa
// q = round(v / 2^(E−15)) fits int16 (clamped to ±32767 at the top); the
// rounding error is at most 2^−16 of the block's largest magnitude.  Blocks
// whose largest magnitude is below 2^−100 are stored as zero.
__global__ __launch_bounds__(256) void k_to_bfp16(const float* __restrict__ in, int16_t* __restrict__ q,
                                                  float* __restrict__ s, int64_t nl4, int64_t nblk) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t field = blockIdx.y;
    const int64_t nl = nl4 * 4;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < nl4) a = reinterpret_cast<const float4*>(in + field * nl)[i];
    float m = fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w)));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    float scale = 1.0f, inv = 0.0f;
    if (m >= 0x1p-100f) {
        int e = 0;
        (void)frexpf(m, &e);  // m = f·2^e, f ∈ [0.5, 1)
        scale = ldexpf(1.0f, e - 15);
        inv = ldexpf(1.0f, 15 - e);
    }
    auto quant = [&](float v) {
        const float r = rintf(v * inv);
        return static_cast<int16_t>(fminf(fmaxf(r, -32767.0f), 32767.0f));
    };
    const int64_t blk = i / kBfpBlock4;
    if (i < nl4) {
        const uint32_t lo = static_cast<uint16_t>(quant(a.x)) | (static_cast<uint32_t>(static_cast<uint16_t>(quant(a.y))) << 16);
        const uint32_t hi = static_cast<uint16_t>(quant(a.z)) | (static_cast<uint32_t>(static_cast<uint16_t>(quant(a.w))) << 16);
        u2v bits;
        bits.x = lo;
        bits.y = hi;
        reinterpret_cast<u2v*>(q + field * nl)[i] = bits;
        if (i % kBfpBlock4 == 0) s[field * nblk + blk] = scale;
    }
}

int num_cus() {
    // one device per process; the first call (any thread) queries it
    static const int cus = [] {
        int dev = 0, n = 0;
        CLR_HIP_CHECK(hipGetDevice(&dev));
        CLR_HIP_CHECK(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
        return n > 0 ? n : 1;
    }();
    return cus;
}

// CLAIRE_AMD_GATHER_CHUNK (planes, >= 1) overrides the choice, for tuning.
int chunk_override() {
    // read at every launch (not cached) so that a process can switch it
    const char* e = std::getenv("CLAIRE_AMD_GATHER_CHUNK");
    return e ? std::atoi(e) : 0;
}

// CLAIRE_AMD_GATHER_PAIR=0 selects the one-value-per-entry layout for every
// D <= 2 gather (three blocks per CU) instead of the pair layout (two), for
// comparison.
bool pair_layout() {
    static const bool on = [] {
        const char* e = std::getenv("CLAIRE_AMD_GATHER_PAIR");
        return !(e && std::atoi(e) == 0);
    }();
    return on;
}

// Chunk lengths (planes per block) worth trying, the most promising first, by
// a model of the launch: with nch chunks a CU runs k = ceil(tiles·nch/CUs)
// blocks, `per_cu` of them at a time (their LDS decides it), and a block costs
// its planes plus a prologue worth about kPrologue planes.  A CU that holds
// fewer blocks than it could is faster per block but slower overall: share[m]
// is the time of a plane with m resident blocks over that with per_cu
// (measured: pair layout 0.85 against 1.25 µs, one-value layout 1.0, 1.7 and
// 2.35 µs).  Against the measured times of 64³ to 512³ the model is within
// about 10%, so the tuner below times its best few.  What it finds: one full
// round of long chunks on large grids (256³, one field: 64 planes 90 µs, 32
// planes 91, 24 planes 97; 512³: 64 planes 626 µs, 24 planes 697, since a
// chunk re-reads the planes around it), and enough short chunks to reach every
// CU on small ones (64³: 2 planes 6.7 µs, 4 planes 8.2, 8 planes 11.3).
constexpr int kMaxChunk = 128;
constexpr int kCandidates = 6;

std::vector<int> chunk_candidates(int n1, int64_t tiles, int per_cu, int most) {
    static const double share[4][4] = {
        {0, 0, 0, 0}, {0, 1.0, 0, 0}, {0, 0.68, 1.0, 0}, {0, 0.43, 0.72, 1.0}};
    constexpr double kPrologue = 3.0;
    std::vector<std::pair<double, int>> cost;
    for (int nch = 1; nch <= n1; ++nch) {
        const int chunk = (n1 + nch - 1) / nch;
        if (chunk > most || (!cost.empty() && cost.back().second == chunk)) continue;
        const int64_t blocks = tiles * ((n1 + chunk - 1) / chunk);
        const int64_t k = (blocks + num_cus() - 1) / num_cus();
        const double rounds = static_cast<double>(k / per_cu) + share[per_cu][k % per_cu];
        cost.emplace_back(rounds * (chunk + kPrologue), chunk);
    }
    std::sort(cost.begin(), cost.end());
    std::vector<int> c;
    for (size_t i = 0; i < cost.size() && i < static_cast<size_t>(kCandidates); ++i) c.push_back(cost[i].second);
    return c;
}

// Chunk-length autotuning of the kernels with a fixed window.  The first launch
// of a gather shape (bound D, grid, number of fields) times the candidates on
// the launch stream, each kTuneRuns times in turn, and keeps the one with the
// shortest run for every later launch of that shape (a single run each had kept
// a length up to 10% slower than the best).  The chunk length only changes how the
// planes are split among blocks, not the arithmetic of any point, so every
// candidate writes the same output; repeating a launch is harmless because no
// gather writes a buffer it reads (the launchers check it: the steps refuse to run
// in place, and the RK4 stage sums ping-pong between two buffers).  Tuning is
// skipped while the stream is being captured into a graph;
// CLAIRE_AMD_GATHER_TUNE=0 turns it off (the model's first choice is used).
// Launches with centred windows always take the model's first choice: how long
// a length takes there depends on the points (how far they drift over a chunk),
// so the first call's points would decide for all later ones, and a call at raw
// points would wait for its stream.  Over smooth maps of CFL 2.5 to 9 at 96³ to
// 512³ that choice is 2.8% (geometric mean) off the best length of each input
// and within 6% of the one timed at CFL 2.5; at CFL 13 shorter chunks, which drift
// less, would win (three fields of 128³ 86 µs with 13 planes, 109 with its choice).
constexpr int kTuneRuns = 3;
struct ShapeKey {
    int d, n1, n2, n3, nz;
    bool operator<(const ShapeKey& o) const {
        return std::tie(d, n1, n2, n3, nz) < std::tie(o.d, o.n1, o.n2, o.n3, o.nz);
    }
};
std::mutex g_tune_mu;
std::map<ShapeKey, int> g_tuned;

bool tuning_enabled() {
    static const bool on = [] {
        const char* e = std::getenv("CLAIRE_AMD_GATHER_TUNE");
        return !(e && std::atoi(e) == 0);
    }();
    return on;
}

// Launches through `launch(chunk)` with the chunk length of `key`: timed on the
// first launch of that shape, or (tune = false) the model's first choice.
template <class Launch>
void chunked_launch(const ShapeKey& key, int64_t tiles, int per_cu, int most, bool tune, hipStream_t st,
                    Launch&& launch) {
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        const auto it = g_tuned.find(key);
        if (it != g_tuned.end()) return launch(it->second);
    }
    const std::vector<int> cand = chunk_candidates(key.n1, tiles, per_cu, most);
    if (!tune) {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        return launch(g_tuned[key] = cand[0]);
    }
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (!tuning_enabled() || hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
        return launch(cand[0]);
    launch(cand[0]);  // warm-up; its output is the result
    int best = cand[0];
    if (cand.size() > 1) {
        hipEvent_t ev[2];
        CLR_HIP_CHECK(hipEventCreate(&ev[0]));
        CLR_HIP_CHECK(hipEventCreate(&ev[1]));
        float best_ms = std::numeric_limits<float>::max();
        for (int run = 0; run < kTuneRuns; ++run)
            for (int c : cand) {
                CLR_HIP_CHECK(hipEventRecord(ev[0], st));
                launch(c);
                CLR_HIP_CHECK(hipEventRecord(ev[1], st));
                CLR_HIP_CHECK(hipEventSynchronize(ev[1]));
                float ms = 0.f;
                CLR_HIP_CHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
                if (ms < best_ms) {
                    best_ms = ms;
                    best = c;
                }
            }
        (void)hipEventDestroy(ev[0]);
        (void)hipEventDestroy(ev[1]);
    }
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tuned[key] = best;
}

// One-value layout for bound −MODE (MODE < 0) or pair layout with the points of
// MODE.
template <int MODE, class Epi>
void launch_lds(const GatherDims& g, const void* pts, const float* f, int64_t fzstride, int nz, const Epi& epi,
                hipStream_t st) {
    constexpr bool kPair = MODE >= 0;
    constexpr int D = kPair ? PairGeo::D : -MODE;
    const int nt3 = (g.n3 + LdsGeo<D>::LT3 - 1) / LdsGeo<D>::LT3;
    const int nt2 = (g.n2 + kLT2 - 1) / kLT2;
    const PlanPt* P = static_cast<const PlanPt*>(pts);
    auto launch = [&](int chunk) {
        const int nch = (g.n1 + chunk - 1) / chunk;
        const int nb = nt3 * nt2 * nch;
        if constexpr (kPair)
            hipLaunchKernelGGL((k_gather_lds_pair<Epi, MODE>), dim3(nb * nz), dim3(kLThreads), 0, st, g, make_hh(g), P,
                               f, fzstride, epi, nb, chunk);
        else
            hipLaunchKernelGGL((k_gather_lds<D, Epi>), dim3(nb * nz), dim3(kLThreads), 0, st, g, P, f, fzstride, epi,
                               nb, chunk);
    };
    constexpr int kPerCu = kPair ? 2 : (D <= 2 ? 3 : 1);
    constexpr int kMost = MODE > kPtsNear ? far_chunk(MODE) : kMaxChunk;
    const int64_t tiles = static_cast<int64_t>(nt3) * nt2 * nz;
    if (chunk_override() >= 1) return launch(std::min({chunk_override(), g.n1, kMost}));
    chunked_launch(ShapeKey{MODE, g.n1, g.n2, g.n3, nz}, tiles, kPerCu, kMost, MODE <= kPtsNear, st, launch);
}

void check_lds_dims(const GatherDims& g) {
    CLR_REQUIRE(g.n1 >= 4 && g.n2 >= 4 && g.n3 >= 4, kErrInvalidArgument, "gather needs n >= 4 per axis");
    CLR_REQUIRE(g.nl < (int64_t(1) << 28), kErrInvalidArgument, "grid too large for 32-bit buffer byte offsets");
}

// Points of a launch from which bounds above 2 take centred windows (kPtsPlan).
// Finding the centres costs a block about 2 µs, which small launches, one block
// per CU, do not hide.  Centred windows against the kernel they replace (D <= 4 up
// to CFL 4, else the direct one), one field: 64³ 8.5 : 6.8 µs (CFL 4); 96³ 14.5 :
// 15.5 (CFL 3.5) and 20.9 : 20.9 (CFL 6); 128³ 21.6 : 23.6 and 27 : 41; 256³ 102 :
// 152 and 130 : 266.  Three fields: 64³ 13.7 : 13.7 (CFL 4); 96³ 28 : 38 and 36 :
// 56; 128³ 47 : 61 and 62 : 117; 256³ 301 : 419 and 360 : 792.
constexpr int64_t kFarPoints = int64_t(1) << 19;
// Share of far-apart points (PlanBound::spread) up to which they are the faster
// ones, by the kernel they replace: one that a bound of 4 cells suffices for, or
// the direct one.  In µs against that kernel, scalar and three fields, for smooth
// fields of up to so many cells and for noise:
//   bound 4    96³  3.5 smooth (spread 0.03) 14.5 : 15.5  28 : 38
//             128³  the same (0.02) 21.6 : 23.6  47 : 61, noise 2.8 36 : 31  101 : 87
//             256³  the same (0.00) 102 : 152  301 : 419, noise 2.8 273 : 205  751 : 610
//   above 4    96³  8 smooth (0.4 to 0.45) 25.3 : 22.3  51 : 60, 9 (0.5 to 0.55) 29 : 22.6  62 : 60
//             128³  9 smooth (0.45 to 0.5) 40 : 43  114 : 123, 20 (> 0.65) 81 : 51  209 : 147
//       192×150×256 10 smooth (< 0.4) 114 : 110  280 : 322, 12 (0.5 to 0.55) 146 : 113  351 : 333
//             256³  9 smooth (< 0.4) 204 : 278  500 : 826, 12 (0.5 to 0.55) 399 : 285  743 : 857
//        noise 5 (0.5 to 0.55)  128³ 83 : 70  251 : 207, 256³ 610 : 627  1873 : 2001
constexpr float kMostSpread[2] = {0.05f, 0.5f};

bool centred_windows(const GatherDims& g, PlanBound b, int nz) {
    return g.nl * nz >= kFarPoints && b.spread <= kMostSpread[b.d > kNearBound];
}

template <class Epi>
void dispatch(PlanBound bound, const GatherDims& g, const uint32_t* P, const float* f, int64_t fzstride, int nz,
              const Epi& epi, hipStream_t st) {
    check_lds_dims(g);
    CLR_REQUIRE(plan_gather_lds(g, bound, nz), kErrInvalidArgument, "displacement bound too large for the LDS gather");
    if (bound.d > 2) {
        if (centred_windows(g, bound, nz)) return launch_lds<kPtsPlan>(g, P, f, fzstride, nz, epi, st);
        return launch_lds<-4>(g, P, f, fzstride, nz, epi, st);
    }
    // The pair layout (two blocks per CU) is faster than the one-value layout
    // (three) for one field per launch (the solves' steps: 110 µs against 115
    // at 256³, before later changes to both kernels), for plain three-field
    // gathers, and for the trajectory stages from about 80³ points on: set
    // velocity + state trajectory + one gather 615 -> 580 µs at 256³, 4.63 ->
    // 4.35 ms at 512³, 125 -> 121 µs at 128³, 89.9 -> 89.0 at 96³.  Below, the
    // third resident block counts for more: 58.6 against 56.9 µs at 64³.
    constexpr bool kPlain = std::is_same<Epi, EpiPlain>::value;
    constexpr int64_t kPairStagePoints = int64_t(1) << 19;
    if ((nz == 1 || kPlain || g.nl >= kPairStagePoints) && pair_layout())
        launch_lds<kPtsNear>(g, P, f, fzstride, nz, epi, st);
    else
        launch_lds<-2>(g, P, f, fzstride, nz, epi, st);
}

bool use_lds(const TrajectoryPlan& tp, const GatherDims& g, int nz) { return plan_gather_lds(g, tp.bound, nz); }

}  // namespace

bool plan_gather_lds(const GatherDims& g, PlanBound b, int nz) {
    if (b.d < 0 || b.d > kPlanMaxN) return false;  // no plan: a point is not finite
    return b.d <= kNearBound || centred_windows(g, b, nz);
}

void launch_points_gather(const GatherDims& g, const float* f, const float* X, float* out, hipStream_t st) {
    // Raw points cost the centred windows their encoding too.  Smooth maps in µs
    // against the direct kernel: 64³ CFL 2 10.1 : 7.7; 96³ CFL 2 18.0 : 18.9, CFL 8
    // 25.8 : 21.3; 128³ CFL 3 26 : 38, CFL 9 40 : 42; 192×150×256 CFL 3 67 : 99, CFL 9
    // 88 : 102; 256³ CFL 3 134 : 259, CFL 9 163 : 263.  The points stay on the device,
    // so nothing is known of them here, and each block decides for itself.  Blocks of
    // 512 threads with an equal count of planes balance direct reads worse than the
    // direct kernel's small blocks do, so scattered points pay for it.  At 128³,
    // 192×150×256 and 256³: noise of ±2 cells 35 : 68, 105 : 199, 203 : 473; ±4 86 :
    // 71, 348 : 255, 720 : 647; ±8 107 : 118, 570 : 424, 1150 : 1044; one point in ten
    // anywhere 62 : 46, 271 : 214, 630 : 530; all anywhere 319 : 316, 1886 : 1857, 4923 :
    // 4917; folding maps of CFL 20 77 : 50, 193 : 110, 368 : 301.
    if (g.nl < (int64_t(1) << 20)) return launch_gather1(g, f, X, out, st);
    check_lds_dims(g);
    launch_lds<kPtsRaw>(g, X, f, 0, 1, EpiPlain{out, 0}, st);
}

void launch_plan_gather(const TrajectoryPlan& tp, const GatherDims& g, const float* const f[], int nf,
                        float* const out[], hipStream_t st) {
    if (!use_lds(tp, g, nf)) return launch_direct_gather(g, tp.X, f, nf, out, st);
    const int64_t fz = nf > 1 ? (f[1] - f[0]) : 0;
    const int64_t oz = nf > 1 ? (out[1] - out[0]) : 0;
    for (int d = 2; d < nf; ++d)
        CLR_REQUIRE(f[d] - f[d - 1] == fz && out[d] - out[d - 1] == oz, kErrInvalidArgument,
                    "vector gather needs equally spaced components");
    dispatch(tp.bound, g, tp.P, f[0], fz, nf, EpiPlain{out[0], oz}, st);
}

void launch_plan_inc_state_step(const TrajectoryPlan& tp, const GatherDims& g, const float* mt, const float* sj,
                                float* out, int negate, hipStream_t st) {
    if (!use_lds(tp, g, 1)) return launch_direct_inc_state_step(g, tp.X, mt, sj, out, negate, st);
    CLR_REQUIRE(mt != out, kErrInvalidArgument, "semi-Lagrangian step cannot run in place");
    dispatch(tp.bound, g, tp.P, mt, 0, 1, EpiIncStep{sj, out, negate ? -1.0f : 1.0f}, st);
}

void launch_plan_adjoint_step(const TrajectoryPlan& tp, const GatherDims& g, const float* C, const float* lam,
                              float* out, hipStream_t st) {
    if (!use_lds(tp, g, 1)) return launch_direct_adjoint_step(g, tp.X, C, lam, out, st);
    CLR_REQUIRE(lam != out, kErrInvalidArgument, "semi-Lagrangian step cannot run in place");
    dispatch(tp.bound, g, tp.P, lam, 0, 1, EpiAdjStep{C, out}, st);
}

void launch_plan_adjoint_coeff(const TrajectoryPlan& tp, const GatherDims& g, const float* divv, float ht, float alpha,
                               float* C, hipStream_t st) {
    if (!use_lds(tp, g, 1)) return launch_adjoint_coeff(g, tp.X, divv, ht, alpha, C, st);
    CLR_REQUIRE(divv != C, kErrInvalidArgument, "coefficient cannot overwrite ∇·v");
    dispatch(tp.bound, g, tp.P, divv, 0, 1, EpiAdjCoeff{divv, C, ht, alpha}, st);
}

void launch_lds_traj_rk2_corrector(const Dims& d, const uint32_t* P, PlanBound bound, const float* const v[3], float sigma,
                                   float ht, float* X, hipStream_t st) {
    const GatherDims g = gather_dims(d);
    const int64_t vz = v[1] - v[0];
    CLR_REQUIRE(v[2] - v[1] == vz && vz == g.nl, kErrInvalidArgument, "velocity components must be contiguous");
    EpiTrajRk2 e{v[0], X, g.nl, d.hx[0], d.hx[1], d.hx[2], sigma * (0.5f * ht), 0};
    dispatch(bound, g, P, v[0], vz, 3, e, st);
}

void launch_lds_traj_rk4_stage(int stage, const Dims& d, const uint32_t* P, PlanBound bound, const float* const v[3],
                               float sigma, float ht, const float* Fin, float* Fout, float* X, hipStream_t st) {
    const GatherDims g = gather_dims(d);
    const int64_t vz = v[1] - v[0];
    CLR_REQUIRE(v[2] - v[1] == vz && vz == g.nl, kErrInvalidArgument, "velocity components must be contiguous");
    // the tuner may repeat a launch: no stage may overwrite what it reads
    CLR_REQUIRE(stage == 1 || Fin != nullptr, kErrInvalidArgument, "RK4 stage needs the previous stage sum");
    CLR_REQUIRE(stage == 3 || (Fout != nullptr && Fout != Fin), kErrInvalidArgument,
                "RK4 stage sum must go to a buffer distinct from its input");
    const float hx[3] = {d.hx[0], d.hx[1], d.hx[2]};
    const float hthalf = 0.5f * ht;
    const double s6 = static_cast<double>(sigma) * (static_cast<double>(ht) / 6.0);
    switch (stage) {
        case 1: {
            EpiTrajRk4<1> e{v[0], X, Fout, g.nl, hx[0], hx[1], hx[2], sigma * hthalf, s6, 0};
            return dispatch(bound, g, P, v[0], vz, 3, e, st);
        }
        case 2: {
            EpiTrajRk4<2> e{Fin, X, Fout, g.nl, hx[0], hx[1], hx[2], sigma * ht, s6, 0};
            return dispatch(bound, g, P, v[0], vz, 3, e, st);
        }
        case 3: {
            EpiTrajRk4<3> e{Fin, X, X, g.nl, hx[0], hx[1], hx[2], 0.0f, s6, 0};  // no second output
            return dispatch(bound, g, P, v[0], vz, 3, e, st);
        }
        default:
            throw Error(kErrInvalidArgument, "RK4 stage must be 1, 2 or 3");
    }
}

// Points from which the streaming kernels are bound by memory and take two runs per
// wave.  Below, they wait for their loads with too few waves to hide them: one run per
// wave, four of the body force's time steps in flight at once, and the right-hand
// sides' time steps shared out over up to four groups of blocks (each time step is
// independent of the others).  Body force 6.4 -> 4.4 µs at 32³, 10.3 -> 6.6 at 64³;
// right-hand sides 6.9 -> 2.9 and 9.8 -> 8.4, but 21.8 -> 27.5 at 96³ and 157 -> 241
// at 192³, where every group reads the velocities again.
constexpr int64_t kStreamPoints = int64_t(1) << 19;
unsigned stream_blocks(int64_t nl4, int k) { return static_cast<unsigned>((nl4 + 256 * k - 1) / (256 * k)); }

template <class Src>
void body_force(int64_t nl, int nt, float ht, float hd, const float* lam, const Src& gm, float* const b[3],
                hipStream_t st) {
    CLR_REQUIRE(nl % 4 == 0, kErrInvalidArgument, "grid size must be a multiple of 4 points");
    const int64_t nl4 = nl / 4;
    BodyP<Src> p{lam, gm, {b[0], b[1], b[2]}};
    if (nl < kStreamPoints)
        hipLaunchKernelGGL((k_body_force<Src, 1, 4>), dim3(stream_blocks(nl4, 1)), dim3(256), 0, st, nl4, nt, ht, hd, p);
    else
        hipLaunchKernelGGL((k_body_force<Src, 2, 1>), dim3(stream_blocks(nl4, 2)), dim3(256), 0, st, nl4, nt, ht, hd, p);
}

template <class Src>
void inc_state_rhs(int64_t nl, int nt, float ht, const float* const vx[3], const float* const vt[3], const Src& gX,
                   const Src& gm, float* s, float* mt1, hipStream_t st) {
    CLR_REQUIRE(nl % 4 == 0, kErrInvalidArgument, "grid size must be a multiple of 4 points");
    CLR_REQUIRE(nt >= 1, kErrInvalidArgument, "nt must be >= 1");
    const int64_t nl4 = nl / 4;
    RhsP<Src> p{{vx[0], vx[1], vx[2]}, {vt[0], vt[1], vt[2]}, gX, gm, s, mt1};
    if (nl < kStreamPoints)
        hipLaunchKernelGGL((k_inc_state_rhs<Src, 1>), dim3(stream_blocks(nl4, 1), std::min(nt, 4)), dim3(256), 0, st, nl4,
                           nt, 0.5f * ht, p);
    else
        hipLaunchKernelGGL((k_inc_state_rhs<Src, 2>), dim3(stream_blocks(nl4, 2)), dim3(256), 0, st, nl4, nt, 0.5f * ht, p);
}

int64_t bfp16_blocks(int64_t nl) { return (nl / 4 + kBfpBlock4 - 1) / kBfpBlock4; }

namespace {

SrcBfp bfp_src(const Bfp16Fields& f, int64_t nl) { return SrcBfp{f.q, f.s, bfp16_blocks(nl)}; }

}  // namespace

void launch_body_force(int64_t nl, int nt, float ht, float hd, const float* lam, const float* gm, float* const b[3],
                       hipStream_t st) {
    body_force(nl, nt, ht, hd, lam, SrcF32{gm}, b, st);
}

void launch_body_force_bfp(int64_t nl, int nt, float ht, float hd, const float* lam, const Bfp16Fields& gm,
                           float* const b[3], hipStream_t st) {
    body_force(nl, nt, ht, hd, lam, bfp_src(gm, nl), b, st);
}

void launch_inc_state_rhs(int64_t nl, int nt, float ht, const float* const vx[3], const float* const vt[3],
                          const float* gX, const float* gm, float* s, float* mt1, hipStream_t st) {
    inc_state_rhs(nl, nt, ht, vx, vt, SrcF32{gX}, SrcF32{gm}, s, mt1, st);
}

void launch_inc_state_rhs_bfp(int64_t nl, int nt, float ht, const float* const vx[3], const float* const vt[3],
                              const Bfp16Fields& gX, const Bfp16Fields& gm, float* s, float* mt1, hipStream_t st) {
    inc_state_rhs(nl, nt, ht, vx, vt, bfp_src(gX, nl), bfp_src(gm, nl), s, mt1, st);
}

void launch_to_bfp16(const float* in, int64_t nl, int nfields, const Bfp16Fields& out, hipStream_t st) {
    CLR_REQUIRE(nl % 4 == 0, kErrInvalidArgument, "field length must be a multiple of 4");
    CLR_REQUIRE(nfields >= 1 && nfields <= 65535, kErrInvalidArgument, "1 to 65535 fields");
    const int64_t nl4 = nl / 4;
    const int nb = static_cast<int>((nl4 + 255) / 256);
    hipLaunchKernelGGL(k_to_bfp16, dim3(nb, nfields), dim3(256), 0, st, in, out.q, out.s, nl4, bfp16_blocks(nl));
}

}  // namespace claire_amd
