// scaled.hip.h -- first-order sweeps (value, marginals, parameter gradients) in the
// linear domain: alpha is held as a 64-bit float a with alpha = T ln(2) (log2 a + K),
// K a per-lane integer exponent that is renewed once per chunk.
//
// The recurrences are sums of products there (soft Smith-Waterman:
//   a[i,j] = E[i,j] (a[i-1,j-1] + 1) + g (a[i-1,j] + a[i,j-1]),  E = 2^(s c), g = 2^(gap c),
//   c = log2(e) / T),
// so a cell costs one exponential and four 64-bit fmas where the log domain pays an
// exponential per candidate and a logarithm, and its dependency chain is two fmas and a
// lane shift.  The reverse sweep needs no alpha: with b[i,j] the weight of all paths
// from (i, j) on,
//   b[i,j] = 1 + E[i+1,j+1] b[i+1,j+1] + g (b[i+1,j] + b[i,j+1]),
// and the marginal is P = E (a[i-1,j-1] + 1) b / Z.  The forward keeps one checkpoint per
// 16-step chunk (the state that enters it) instead of a table, and the reverse sweep
// rebuilds the chunk's values from it in registers, in the scale that makes a b / Z the
// marginal itself.  E carries a 32-bit rounding; values, flows and gap sums are in 64 bits;
// the sum of P s takes P as it is stored, in 32 bits, and is in 32 bits over the 16 steps of a
// chunk (with helper waves it takes s from E, log2 E / c) and in 64 bits beyond.
//
// Range.  Scores that move a lane's values up by more than about 60 bits a step take them
// beyond 2^1023 of its chunk's scale: they become infinite or NaN, which the sweeps detect.
// They set redo[b], the reverse sweep is left out where the forward found it, and the log-domain
// sweeps recompute that element, in the launch shape that they would have taken.
// Downwards nothing becomes infinite.  E is 0 below 2^-149 (and rounded below 2^-126), and
// values below 2^-1022 of the scale are lost.  Where two gaps go round any match (linear
// gaps, and global affine ones, whose gaps follow each other in either order) they bound both:
// a gap costs at most kMaxGapBits, which the host checks, so what is left out weighs less than
// 2^(80 - 126) of what goes round it.  Local affine alignment has to match through the cell: the
// forward keeps the largest factor below 2^-126 that it met, and element_partition() says
// whether it can be left out (a mask: yes) or the element is out of range.
//
// Pipeline.  Stripes of 64 rows, one wave each, a lane per row, one anti-diagonal per
// step (wavefront.hip.h); at most 8 stripes per workgroup.  Longer elements, and
// elements of small batches, are split into parts.  A part's boundary row reaches the
// next part through global memory: an exporting wave copies the last stripe's ring
// out and an importing wave copies it into the next part's first ring, so that the
// sweeping waves wait on LDS progress words only and never on a global load of their
// own.
//
// What bounds them.  Few elements: the pipeline, (L2 / 16 + 4 + 5 (stripes - 1)) chunk
// periods of some 2000 (forward) and 2500 (reverse) cycles, most of them the 16 dependent
// steps.  Enough elements to fill the chip: instruction issue.  Memory is far from it
// (scores read twice, marginals written once: 0.8 GB at [256, 512, 512], 0.13 ms).
// Log-domain sweeps before, these after, microseconds (forward + reverse), one call among
// others:
//   SW [2, 100, 120]             32 + 44    46 in one launch
//   SW [256, 512, 512]         168 + 228   104 + 231
//   SW [48, 300, 411] ragged     81 + 118    49 + 85
//   NW [96, 301, 277]            99 + 161    56 + 83
// Largest error of values, marginals and gradients against 64 bits, relative (2-norm):
// 3e-5 before, 1e-7 after at [256, 512, 512].
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wavefront.hip.h"

namespace d2p_amd {
namespace sc {

using namespace wf;

constexpr int P = 16;               // steps per chunk
constexpr int NT = 4;               // score tiles of a forward wave: loads three chunks ahead
constexpr int RCH = 16;             // chunks a ring holds
constexpr int RING = RCH * P;       // its slots
constexpr int LEAD = 5;             // chunks a stripe runs behind its producer
constexpr int MAXW = 8;             // waves per workgroup
constexpr int MAXS_SPLIT = 6;       // stripes per part beside the two copying waves
constexpr double kMaxGapBits = 40.0;
// log2 of the least factor E that 32 bits hold in full
constexpr float kMinBits = -126.0f;
// local affine elements with smaller factors (element_partition): log2 of Z at most, and log2 of
// the share of Z of the paths through one such cell at most (2^20 cells: 2^-40 in all)
constexpr int kMaxMaskedExp = 850;
constexpr float kNoShare = -60.0f;
// exponent of the SW scale: below it the restart term 1 would overflow
constexpr int kMinExp = -900;

enum Fam { SW, NW, AFF, NWAFF };

template <Fam F>
struct Traits {
    static constexpr bool AFFINE = F == AFF || F == NWAFF;
    static constexpr bool LOCAL = F == SW || F == AFF;      // restart and end anywhere
    static constexpr int NV = AFFINE ? 3 : 1;               // own state: a, or M, I, D
    static constexpr int NP = AFFINE ? 2 : 1;               // values passed down a row
    static constexpr int NQ = AFFINE ? 2 : 1;               // values passed up a row
};

struct Consts {
    float c;           // log2(e) / T
    double g, o, e;    // linear gap, open, extend factors
    double gc, oc, ec; // their base-2 exponents
};

// Chunks of a stripe.
__host__ __device__ inline int chunks(int L2) { return (L2 + 63 + P - 1) / P; }

// ---- per-call memory, carved from the table area of the workspace (every entry
// point's table is larger): checkpoints, exponents, last rows, reverse flows.
struct Mem {
    double* ck;     // [B][stripe][chunk][lane][NV + 1]
    int* kx;        // [B][stripe][chunk][64] exponents entering the chunk
    double* brow;   // [B][stripe][plane NP][16 (nch + 1)] last row by step + 1
    int* kexp;      // [B][part][nch] forward boundary exponents (split)
    double* flow;   // [B][part][plane NQ][16 nch] reverse flows by step (split)
    int* kflow;     // [B][part][nch] their exponents
    double* zpart;  // [B][part][3] partition (mantissa, exponent), log2 of the largest E left out
    size_t bytes;
};

template <Fam F>
__host__ inline Mem carve(void* base, int B, int max_L1, int max_L2, int G) {
    using Tr = Traits<F>;
    const size_t ns = ((size_t)max_L1 + 63) / 64, nch = (size_t)chunks(max_L2);
    const size_t st = (size_t)B * ns, pt = (size_t)B * G;
    char* p = (char*)base;
    Mem m;
    auto take = [&](size_t n) {
        char* q = p;
        p += round256(n);
        return q;
    };
    m.ck = (double*)take(st * nch * 64 * (Tr::NV + 1) * 8);
    m.kx = (int*)take(st * nch * 64 * 4);
    m.brow = (double*)take(st * Tr::NP * P * (nch + 1) * 8);
    m.kexp = (int*)take(pt * nch * 4);
    m.flow = (double*)take(pt * Tr::NQ * P * nch * 8);
    m.kflow = (int*)take(pt * nch * 4);
    m.zpart = (double*)take(pt * 3 * 8);
    m.bytes = (size_t)(p - (char*)base);
    return m;
}

struct Args {
    const float* m;       // scores [B][L1max][L2max]
    const int* lengths;   // [B][2] or null
    float* out;           // marginals
    float* value;
    float* grad0;         // gap / open (null: none)
    float* grad1;         // extend (affine)
    float* gradT;
    int* status;
    int* redo;
    uint64_t* fflag;
    uint64_t* bflag;
    double* bpart;        // [B][part][4]
    Mem mem;
    Consts k;
    double gap, ext, T;   // parameters in their own units
    int B, L1max, L2max, NSmax, G, SPW;
    uint32_t epoch;
};

// ---------------------------------------------------------------- device helpers

__device__ __forceinline__ double shr1(double v, double old) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), 0x138, 0xf,
                                               0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), 0x138, 0xf,
                                               0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double shl1(double v, double old) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), 0x130, 0xf,
                                               0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), 0x130, 0xf,
                                               0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ int shr1(int v, int old) {
    return __builtin_amdgcn_update_dpp(old, v, 0x138, 0xf, 0xf, false);
}
__device__ __forceinline__ int shl1(int v, int old) {
    return __builtin_amdgcn_update_dpp(old, v, 0x130, 0xf, 0xf, false);
}
__device__ __forceinline__ double scale2(double v, int e) { return __builtin_amdgcn_ldexp(v, e); }
// exponent of a non-negative number: 1024 for infinities and NaN, -1023 for 0
__device__ __forceinline__ int exponent(double v) {
    return (int)(((uint32_t)__double2hiint(v) >> 20) & 0x7ff) - 1023;
}

__device__ __forceinline__ void store_sys_f64(double* p, double v) {
    store_sys2(reinterpret_cast<float2*>(p),
               make_float2(__int_as_float(__double2loint(v)), __int_as_float(__double2hiint(v))));
}
__device__ __forceinline__ void store_sys_i32(int* p, int v) {
    store_sys(reinterpret_cast<float*>(p), __int_as_float(v));
}

// LDS of one workgroup.  Ring r of the forward is written by the producer of wave r
// (ring 0 by the importing wave) and read by wave r; of the reverse sweep, ring r is
// written by wave r and read by wave r - 1 (ring `stripes` by the importing wave).
template <int N>
struct Ring {
    double v[N][RING];
    int k[RCH];
    int pad[RCH];
};

// Marks an element for the log-domain sweeps.  The bits tell what the forward found, which every
// part of the reverse sweep sees, from what a part of the reverse sweep found, which the
// others may or may not.
enum { REDO_FWD = 1, REDO_BWD = 2 };
static_assert((REDO_FWD | REDO_BWD) < 1 << REDO_BITS, "below the count of parts");
__device__ __forceinline__ void flag_redo(int* redo_b, int bit) {
    __hip_atomic_fetch_or(redo_b, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The quads of one chunk of the stripe, clamped only where the 16-byte loads could
// leave the tensor: `room` is the number of floats from the stripe's first row to the
// tensor's end.  Cells outside the stripe's rows or columns read a neighbouring row's
// values, which the sweeps mask.  (Offsets from the stripe's first row are never
// negative: lane r's lowest column is t_first - r of row r.)
__device__ __forceinline__ void stage_chunk(f32x4 (&sq)[P / 4], const float* sbase, long long room,
                                            int L1left, int L2max, int lane, int t_first) {
    using Q = QuadTile<P>;
    const long long last = 63LL * (L2max - 1) + t_first + P;
    if (last <= room && t_first + P <= room) {
        const char* cbase = reinterpret_cast<const char*>(sbase);
        uint32_t off = quad_offset0<P, 1>(L2max, lane, t_first);
        const uint32_t step = (uint32_t)(Q::ROWS_X4 * (L2max - 1)) * 4u;
#pragma unroll
        for (int i = 0; i < Q::NQ; ++i) {
            sq[i] = *reinterpret_cast<const f32x4*>(cbase + off);
            off += step;
        }
    } else {
        int l = lane;
        __asm__ volatile("" : "+v"(l));   // (rare: its offsets are not kept across chunks)
#pragma unroll
        for (int i = 0; i < Q::NQ; ++i) {
            const int r = Q::ROWS_X4 * i + l / Q::NQ;
            const int c0 = t_first + 4 * ((l % Q::NQ) ^ Q::swz(r)) - r;
            const float* row = sbase + (size_t)min(r, L1left - 1) * L2max;
#pragma unroll
            for (int e = 0; e < 4; ++e) sq[i][e] = row[min(max(c0 + e, 0), L2max - 1)];
        }
    }
}
__device__ __forceinline__ void put_chunk(float* tile, const f32x4 (&sq)[P / 4], int lane) {
#pragma unroll
    for (int i = 0; i < P / 4; ++i) reinterpret_cast<f32x4*>(tile)[64 * i + lane] = sq[i];
}

// The same chunk straight into an LDS quad tile (4 asynchronous operations, or P at the
// tensor's end); completion is waited for with wait_vmcnt.
__device__ __forceinline__ void dma_chunk(uint32_t tile_lds, const float* sbase, long long room,
                                          int L1left, int L2max, int lane, int t_first) {
    using Q = QuadTile<P>;
    const long long last = 63LL * (L2max - 1) + t_first + P;
    if (last <= room && t_first + P <= room) {
        uint32_t voff = quad_offset0<P, 1>(L2max, lane, t_first);
        const uint32_t vstep = (uint32_t)(Q::ROWS_X4 * (L2max - 1)) * 4u;
#pragma unroll
        for (int i = 0; i < Q::NQ; ++i) lds_dma_dwordx4<1024>(sbase, voff, tile_lds, vstep);
    } else {
        int l = lane;
        __asm__ volatile("" : "+v"(l));
#pragma unroll
        for (int j = 0; j < P; ++j) {
            int r, col;
            quad_cell<P, 1>(64 * j + l, t_first, r, col);
            uint32_t voff =
                (uint32_t)(min(r, L1left - 1) * L2max + min(max(col, 0), L2max - 1)) * 4u;
            lds_dma_dword<256>(sbase, voff, tile_lds, 0u);
        }
    }
}

// Progress words.  A wave's LDS operations execute in order, so the word written after
// the ring data is seen after it: no wait in between, only an order for the compiler.
__device__ __forceinline__ void post(int* prog, int wave, int value) {
    __asm__ volatile("" ::: "memory");
    __hip_atomic_store(prog + wave, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __asm__ volatile("" ::: "memory");
}

// Waits of a stripe's own waves on each other: as wait_for, with shorter sleeps and without its
// wait for this wave's own LDS operations, which execute in order.
__device__ __forceinline__ void wait_own(int* prog, int w, int need, int* status_b) {
    if (prog_load(prog, w) < need) {
        const int limit = __builtin_amdgcn_readfirstlane(g_spin_limit);
        int spins = 0;
        do {
            __builtin_amdgcn_s_sleep(1);
            if (++spins >= limit) {
                atomicOr(status_b, 1);
                break;
            }
        } while (prog_load(prog, w) < need);
    }
    __asm__ volatile("" ::: "memory");
}

// ---------------------------------------------------------------- cell recurrences

// One forward cell: E its factor, d the diagonal input and u the inputs from above (in
// the scale of the lane above, f converts), v the lane's own state (its left cell).
// t1: the diagonal sum; the marginal is t1 E b / Z.
template <Fam F>
struct FwdIn {
    double f, gf;       // 2^(K_above - K), and (linear gaps) times the gap factor
    double one;         // the restart term in this lane's scale
};

template <Fam F>
__device__ __forceinline__ void fwd_cell(const Consts& k, const FwdIn<F>& in, double E, double d,
                                         const double* u, double* v, double& t1, double& t3) {
    if constexpr (F == SW || F == NW) {
        t1 = F == SW ? __builtin_fma(in.f, d, in.one) : in.f * d;
        t3 = __builtin_fma(in.gf, u[0], k.g * v[0]);
        v[0] = __builtin_fma(E, t1, t3);
    } else {
        // v = M, I, D; u[1] = the I state that the cell above feeds
        t1 = F == AFF ? __builtin_fma(in.f, d, in.one) : in.f * d;
        double lm = k.o * v[0];
        if (F == NWAFF) lm = __builtin_fma(k.o, v[1], lm);
        v[2] = __builtin_fma(k.e, v[2], lm);
        v[0] = E * t1;
        v[1] = in.f * u[1];
        t3 = 0.0;
    }
}
// The values a cell passes to the row below.
template <Fam F>
__device__ __forceinline__ void fwd_pass(const Consts& k, const double* v, double* p) {
    if constexpr (Traits<F>::AFFINE) {
        p[0] = (v[0] + v[1]) + v[2];
        double t = __builtin_fma(k.e, v[1], k.o * v[0]);
        if (F == NWAFF) t = __builtin_fma(k.o, v[2], t);
        p[1] = t;
    } else {
        p[0] = v[0];
    }
}

}  // namespace sc
}  // namespace d2p_amd
