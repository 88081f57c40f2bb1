// scaled_sweeps.hip.h -- the forward and reverse sweep kernels of scaled.hip.h and
// their launches, one instantiation per family.
#pragma once
#include <float.h>
#include <limits.h>
#include <stdlib.h>

#include <type_traits>

#include "../../include/d2p_amd.h"
#include "capi_util.hip.h"
#include "scaled.hip.h"

namespace d2p_amd {
namespace sc {

// log2 of the boundary cell x of row 0 / column 0 (x >= 1 gaps) of global alignment.
template <Fam F>
__device__ __forceinline__ double edge_log2(const Consts& k, int x) {
    if constexpr (F == NW) return (double)x * k.gc;
    else return k.oc + (double)(x - 1) * k.ec;
}

__device__ __forceinline__ void element_lengths(const Args& A, int b, int& L1, int& L2) {
    L1 = A.L1max;
    L2 = A.L2max;
    if (A.lengths) {
        L1 = min(max(__builtin_amdgcn_readfirstlane(A.lengths[2 * b]), 0), L1);
        L2 = min(max(__builtin_amdgcn_readfirstlane(A.lengths[2 * b + 1]), 0), L2);
    }
}

// Waits of chunk q (counted in the stripe's own order) on the producer's and the
// consumer's progress words, whose values read during the previous chunk come as
// peeks.
struct Peek {
    int prod, cons;
};
__device__ __forceinline__ void wait_chunk(const Peek& pk, int* prog, int prod, int cons, int q,
                                           int nch, int* st) {
    if (prod >= 0) {
        const int need = min(q + LEAD, nch);
        if (__builtin_amdgcn_readfirstlane(pk.prod) < need) wait_for(prog, prod, need, st);
    }
    if (cons >= 0) {
        const int need = q - 2 - RCH;
        if (__builtin_amdgcn_readfirstlane(pk.cons) < need) wait_for(prog, cons, need, st);
    }
}
__device__ __forceinline__ Peek peek(int* prog, int prod, int cons) {
    Peek p;
    p.prod = prod >= 0 ? prog_peek(prog, prod) : 0;
    p.cons = cons >= 0 ? prog_peek(prog, cons) : 0;
    return p;
}

// ------------------------------------------------------------------ copying waves

// Imports the boundary values of the neighbouring part into `ring`, at most four
// chunks at a time (lane 16 c + n: slot n of chunk c), as they are reported by its
// progress word.  FWD: chunk p covers ring slots 16 p + 1 .. 16 p + 16 (the producer's
// steps 16 p .. 16 p + 15); reverse: the p-th chunk counted down from the last.
template <int N, bool FWD>
__device__ __forceinline__ void import_boundary(Ring<N>* ring, const double* src, size_t plane,
                                                const int* ksrc, const uint64_t* flag,
                                                uint32_t epoch, int* prog, int self, int cons,
                                                int nch, int lane, int* st) {
    int have = 0, cur = 0;
    while (cur < nch) {
        if (have <= cur) have = wait_part(flag, epoch, cur + 1, st);
        const int take = min(min(have - cur, 4), nch - cur);
        const int need = cur + take - 1 - 2 - RCH;
        if (need > 0) wait_for(prog, cons, need, st);
        const int q = cur + (lane >> 4);
        if (q < cur + take) {
            const int ch = FWD ? q : nch - 1 - q;
            const int t = ch * P + (lane & 15);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const double v = __longlong_as_double((long long)load_flag(
                    reinterpret_cast<const uint64_t*>(src + i * plane + t + (FWD ? 1 : 0))));
                const int shift = FWD ? 1 : P - 1;
                ring->v[i][(t + shift) & (RING - 1)] = v;
            }
            if ((lane & 15) == 0) ring->k[ch & (RCH - 1)] = load_status(ksrc + ch);
        }
        cur += take;
        post(prog, self, cur);
    }
}

// Exports ring chunks to the next part as wave `prod` finishes them.
template <int N, bool FWD>
__device__ __forceinline__ void export_boundary(const Ring<N>* ring, double* dst, size_t plane,
                                                int* kdst, uint64_t* flag, uint32_t epoch,
                                                int* prog, int self, int prod, int nch, int lane,
                                                int* st) {
    int cur = 0;
    while (cur < nch) {
        wait_for(prog, prod, cur + 1, st);
        const int have = max(prog_load(prog, prod), cur + 1);
        const int take = min(min(have - cur, 4), nch - cur);
        const int q = cur + (lane >> 4);
        if (q < cur + take) {
            const int ch = FWD ? q : nch - 1 - q;
            const int t = ch * P + (lane & 15);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int shift = FWD ? 1 : P - 1;
                store_sys_f64(dst + i * plane + t + (FWD ? 1 : 0),
                              ring->v[i][(t + shift) & (RING - 1)]);
            }
            if ((lane & 15) == 0) store_sys_i32(kdst + ch, ring->k[ch & (RCH - 1)]);
        }
        cur += take;
        wait_vmcnt<0>();
        if (lane == 0) store_flag(flag, progress_word(epoch, cur));
        // chunks below cur have left the ring: the producer may overwrite them
        post(prog, self, cur - 3);
    }
    wait_vmcnt<0>();
}

// ------------------------------------------------------------------ forward sweep

template <Fam F>
__global__ void __launch_bounds__(MAXW * 64) fwd_kernel(const Args A) {
    using Tr = Traits<F>;
    static_assert(Tr::AFFINE, "linear gaps: fwd2_sweep");
    extern __shared__ __align__(16) char smem[];
    __shared__ int prog[MAXW];
    __shared__ double zred[MAXW];
    __shared__ int kred[MAXW];
    __shared__ float lred[MAXW];
    int b, part;
    split_decode(blockIdx.x, A.G, b, part);
    if (b >= A.B) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int L1, L2;
    element_lengths(A, b, L1, L2);
    const int NS = (L1 > 0 && L2 > 0) ? (L1 + 63) / 64 : 0;
    const int s0 = part * A.SPW;
    const int n = max(0, min(A.SPW, NS - s0));      // stripes of this part
    const int nch = chunks(L2);
    int* st = A.status + b;
    if (threadIdx.x == 0 && A.G == 1) {
        *st = 0;
        A.redo[b] = 0;
    }
    if (threadIdx.x < MAXW) prog[threadIdx.x] = -1;
    __syncthreads();

    const int nring = A.SPW;
    Ring<Tr::NP>* rings = reinterpret_cast<Ring<Tr::NP>*>(smem);
    float* tiles = reinterpret_cast<float*>(rings + nring + 1);
    const int nchmax = chunks(A.L2max);
    const size_t sidx0 = (size_t)b * A.NSmax;
    const size_t brow_plane = (size_t)P * (nchmax + 1);
    const bool from = n > 0 && s0 > 0, to = n > 0 && s0 + n < NS;
    const int W_IN = A.SPW, W_OUT = A.SPW + 1;       // the copying waves

    double zsum = 0.0;      // this wave's share of the partition, scaled by 2^-zk
    int zk = -(1 << 28);
    float low = -FLT_MAX;   // log2 of the largest factor below kMinBits
    if (wave < n) {
        const int s = s0 + wave, i0 = 64 * s;
        const int rows = min(64, L1 - i0);
        const Ring<Tr::NP>* rin = rings + wave;
        Ring<Tr::NP>* rout = rings + wave + 1;
        const int prod = wave > 0 ? wave - 1 : (from ? W_IN : -1);
        const int cons = wave + 1 < n ? wave + 1 : (to ? W_OUT : -1);
        const bool ring_in = prod >= 0;
        const bool below = s + 1 < NS;
        float* tile = tiles + wave * (NT * 64 * P);
        const uint32_t tile_lds = lds_address(tile);
        const float* sbase = A.m + ((size_t)b * A.L1max + i0) * A.L2max;
        const long long room =
            ((long long)(A.B - b) * A.L1max - i0) * (long long)A.L2max;
        const int L1left = A.L1max - i0;
        double* ck = A.mem.ck + (sidx0 + s) * nchmax * 64 * (Tr::NV + 1) + lane * (Tr::NV + 1);
        int* kx = A.mem.kx + (sidx0 + s) * nchmax * 64 + lane;
        double* brow = A.mem.brow + (sidx0 + s) * Tr::NP * brow_plane;
        const bool lane_ok = lane < rows;
        const bool owns_end = s == NS - 1;

        double v[Tr::NV], p[Tr::NP], d = 0.0;
        int K = 0;
#pragma unroll
        for (int i = 0; i < Tr::NV; ++i) v[i] = 0.0;
        if constexpr (F == NWAFF) {                  // column 0: a run of row + 1 gaps
            const double e = edge_log2<F>(A.k, i0 + lane + 1);
            K = (int)floor(e);
            v[1] = exp2(e - (double)K);
        }
        fwd_pass<F>(A.k, v, p);

        // chunk k's scores: tile k % NT, on their way from chunk k - NT on, read into
        // registers during chunk k - 1
        auto load = [&](int k) {
            dma_chunk(tile_lds + (k % NT) * (64 * P * 4), sbase, room, L1left, A.L2max, lane,
                      min(k, nch - 1) * P);
        };
#pragma unroll
        for (int k = 0; k < NT; ++k) load(k);
        // (all of them: the waits below count the loads and stores of three chunks, which the
        // first chunks do not have behind them)
        wait_vmcnt<0>();
        float sN[P];
        read_quads<P, 1>(tile, lane, sN);
        double bw[Tr::NP];       // last row of the previous chunk, on its way to memory
#pragma unroll
        for (int i = 0; i < Tr::NP; ++i) bw[i] = 0.0;
        const bool keep = below && wave + 1 < n;   // (a part's last row: its exporting wave)

        Peek pk = peek(prog, prod, cons);
        int kr_prev = 0;         // scale of lane 0's boundary inputs, previous chunk
        double ring[Tr::NP][P];
        double vend = 0.0;       // global families: the terminal cell
        int kend = 0;
        const int lane_end = rows - 1, t_end = L2 - 1 + lane_end;
        for (int k = 0; k < nch; ++k) {
            wait_chunk(pk, prog, prod, cons, k, nch, st);
            // the previous chunk's last row, for the reverse sweep
            if (keep && k > 0 && lane < P) {
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i)
                    brow[i * brow_plane + (k - 1) * P + lane + 1] = bw[i];
            }

            // boundary inputs of lane 0 and their scale
            int kr = 0;
            if (ring_in) {
                const int base = ((k + 4) & (RCH - 1)) * P;
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i)
#pragma unroll
                    for (int j = 0; j < P; ++j) ring[i][j] = rin->v[i][base + j];
                kr = __builtin_amdgcn_readfirstlane(rin->k[min(k + 4, nch - 1) & (RCH - 1)]);
                // (the first value is the last one of the producer's chunk before, whose
                // scale was the previous chunk's)
                const int ka = k > 0 ? kr_prev
                                     : __builtin_amdgcn_readfirstlane(
                                           rin->k[min(3, nch - 1) & (RCH - 1)]);
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i) ring[i][0] = scale2(ring[i][0], ka - kr);
            } else if (F == NWAFF) {                 // row 0: a run of j gaps
                const double e = edge_log2<F>(A.k, k * P + 1);
                kr = (int)floor(e);
                double x = exp2(e - (double)kr);
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    ring[0][j] = x;
                    ring[Tr::NP - 1][j] = A.k.o * x;
                    x *= A.k.e;
                }
            } else {
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i)
#pragma unroll
                    for (int j = 0; j < P; ++j) ring[i][j] = 0.0;
            }
            double Ed[P];
#pragma unroll
            for (int i = 0; i < P; ++i) Ed[i] = (double)fast_exp2(sN[i] * A.k.c);
            if constexpr (F == AFF) {
                float least = min3_raw(sN[0], sN[1], sN[2]);
#pragma unroll
                for (int i = 3; i < P - 1; i += 2) least = min3_raw(least, sN[i], sN[i + 1]);
                least = min3_raw(least, sN[P - 1], sN[P - 1]);
                if (__builtin_amdgcn_ballot_w64(least * A.k.c < kMinBits) != 0) {
#pragma unroll
                    for (int i = 0; i < P; ++i) {
                        const float x = sN[i] * A.k.c;
                        if (lane_ok && (unsigned)(k * P + i - lane) < (unsigned)L2 && x < kMinBits)
                            low = fmaxf(low, fmaxf(x, -1e30f));
                    }
                }
            }
            // next chunk's scores: its loads were issued three chunks ago, and at least two
            // stores and, in each of the two chunks since, four loads and two stores follow
            wait_vmcnt<2 + 6 * (NT - 2)>();
            read_quads<P, 1>(tile + ((k + 1) % NT) * (64 * P), lane, sN);
            // (tile k % NT was read into registers a chunk ago)
            load(k + NT);

            // the chunk's scale: the exponent of the lane's current value; lanes that have
            // not started take that of the lowest started lane (or the ring's)
            const int ex = exponent(p[0]);
            // (infinities and NaN stay: they are looked for after the last chunk)
            int Kn = K + (ex > -1023 && ex < 1024 ? ex : 0);
            if (Tr::LOCAL) Kn = max(Kn, kMinExp);
            if (Tr::LOCAL) {
                const int started = k * P;           // lanes below have started
                if (started < 64) {
                    const int kb = k == 0 ? kr : __builtin_amdgcn_readlane(Kn, started - 1);
                    if (lane >= started) Kn = kb;
                }
            }
            // lane 0's diagonal input at its first cell: the cell above column 0 (other lanes
            // have it from the lane above)
            if (k == 0) {
                kr_prev = kr;
                if constexpr (F == NWAFF) {
                    const double e = i0 > 0 ? edge_log2<F>(A.k, i0) : 0.0;
                    const int ke = (int)floor(e);
                    d = scale2(exp2(e - (double)ke), ke - kr);
                }
            }
            // (zeros from above the first stripe: any finite factor will do)
            if (!ring_in && F == AFF) kr = __builtin_amdgcn_readlane(Kn, 0);
            const int delta = K - Kn;
#pragma unroll
            for (int i = 0; i < Tr::NV; ++i) v[i] = scale2(v[i], delta);
#pragma unroll
            for (int i = 0; i < Tr::NP; ++i) p[i] = scale2(p[i], delta);
            d = scale2(d, shr1(delta, kr_prev - kr));
            kr_prev = kr;
            K = Kn;
            FwdIn<F> in;
            in.f = scale2(1.0, shr1(Kn, kr) - Kn);
            in.one = Tr::LOCAL ? scale2(1.0, -Kn) : 0.0;

            // checkpoint: the state that enters the chunk
            {
                double* c = ck + (size_t)k * 64 * (Tr::NV + 1);
#pragma unroll
                for (int i = 0; i < Tr::NV; ++i) c[i] = v[i];
                c[Tr::NV] = d;
                kx[(size_t)k * 64] = Kn;
            }

            const int t0 = k * P;
            const bool full = rows == 64 && t0 >= 63 && t0 + P <= L2;
            double hist[Tr::NP][P];
            double zc = 0.0;
            auto steps = [&](auto full_tag) {
                constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    // (read before the last steps, so that it has arrived at the chunk's end)
                    if (j == P - 4) pk = peek(prog, prod, cons);
                    const double E = Ed[j];
                    double u[Tr::NP], w[Tr::NV], t1, t3;
#pragma unroll
                    for (int i = 0; i < Tr::NP; ++i) u[i] = shr1(p[i], ring[i][j]);
#pragma unroll
                    for (int i = 0; i < Tr::NV; ++i) w[i] = v[i];
                    fwd_cell<F>(A.k, in, E, d, u, w, t1, t3);
                    if (FULL) {
#pragma unroll
                        for (int i = 0; i < Tr::NV; ++i) v[i] = w[i];
                        fwd_pass<F>(A.k, v, p);
                        if (Tr::LOCAL) zc += p[0];
                    } else {
                        const int col = t0 + j - lane;
                        const bool ok = lane_ok && col >= 0 && col < L2;
#pragma unroll
                        for (int i = 0; i < Tr::NV; ++i) v[i] = ok ? w[i] : v[i];
                        fwd_pass<F>(A.k, v, p);
                        if (Tr::LOCAL) zc += ok ? p[0] : 0.0;
                        else if (owns_end && lane == lane_end && t0 + j == t_end) {
                            vend = p[0];
                            kend = Kn;
                        }
                    }
                    d = u[0];
#pragma unroll
                    for (int i = 0; i < Tr::NP; ++i) hist[i][j] = p[i];
                }
            };
            if (full) steps(std::true_type{});
            else steps(std::false_type{});

            if (Tr::LOCAL) {
                const int kz = max(zk, Kn);
                zsum = scale2(zsum, max(zk - kz, -4000)) + scale2(zc, Kn - kz);
                zk = kz;
            }
            // the last row to the stripe below and, for the reverse sweep, to memory
            if (lane == 63) {
                const int g0 = (k & (RCH - 1)) * P, g1 = ((k + 1) & (RCH - 1)) * P;
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i) {
#pragma unroll
                    for (int j = 0; j < P - 1; ++j) rout->v[i][g0 + 1 + j] = hist[i][j];
                    rout->v[i][g1] = hist[i][P - 1];
                }
                rout->k[k & (RCH - 1)] = Kn;
            }
            post(prog, wave, k + 1);
#pragma unroll
            for (int i = 0; i < Tr::NP; ++i)
                bw[i] = rout->v[i][(t0 + (lane & (P - 1)) + 1) & (RING - 1)];
        }
        if (keep && lane < P) {
#pragma unroll
            for (int i = 0; i < Tr::NP; ++i)
                brow[i * brow_plane + (nch - 1) * P + lane + 1] = bw[i];
        }
        wait_vmcnt<0>();         // (loads into LDS still under way)
        // values out of range
        if (__builtin_amdgcn_ballot_w64(lane_ok && exponent(p[0]) == 1024) != 0 && lane == 0)
            flag_redo(A.redo + b, REDO_FWD);
        if constexpr (!Tr::LOCAL) {
            if (owns_end) {
                zsum = lane == lane_end ? vend : 0.0;
                zk = __builtin_amdgcn_readlane(kend, lane_end);
            }
        }
    } else if (wave == W_IN && from) {
        import_boundary<Tr::NP, true>(rings, A.mem.brow + (sidx0 + s0 - 1) * Tr::NP * brow_plane,
                                      brow_plane, A.mem.kexp + ((size_t)b * A.G + part - 1) * nchmax,
                                      A.fflag + (size_t)b * A.G + part - 1, A.epoch, prog, W_IN, 0,
                                      nch, lane, st);
    } else if (wave == W_OUT && to) {
        export_boundary<Tr::NP, true>(rings + n, A.mem.brow + (sidx0 + s0 + n - 1) * Tr::NP * brow_plane,
                                      brow_plane, A.mem.kexp + ((size_t)b * A.G + part) * nchmax,
                                      A.fflag + (size_t)b * A.G + part, A.epoch, prog, W_OUT, n - 1,
                                      nch, lane, st);
    }

    // the part's share of the partition
    {
        int km = zk;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) km = max(km, __shfl_xor(km, off, 64));
        zsum = wave_sum(scale2(zsum, max(zk - km, -4000)));
        if (lane == 0) {
            zred[wave] = zsum;
            kred[wave] = km;
        }
        if constexpr (F == AFF) {
            low = wave_reduce(low, [](float a, float b) { return fmaxf(a, b); });
            if (lane == 0) lred[wave] = low;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double z = 0.0;
        int kz = -(1 << 28);
        if (part == 0 && (Tr::LOCAL || NS == 0)) {
            // the empty alignment; global: an element without cells is its boundary,
            // whose value the reverse sweep writes
            z = 1.0;
            kz = 0;
        }
        for (int w = 0; w < n; ++w) {
            const int km = max(kz, kred[w]);
            z = scale2(z, max(kz - km, -4000)) + scale2(zred[w], max(kred[w] - km, -4000));
            kz = km;
        }
        double* zp = A.mem.zpart + ((size_t)b * A.G + part) * 3;
        zp[0] = z;
        zp[1] = (double)kz;
        if constexpr (F == AFF) {
            float least = -FLT_MAX;
            for (int w = 0; w < n; ++w) least = fmaxf(least, lred[w]);
            // (gaps that gain: no bound on what is left out)
            if (least > -FLT_MAX && (A.k.oc > 0.0 || A.k.ec > 0.0)) least = FLT_MAX;
            zp[2] = (double)least;
        }
    }
}

// Marginals on their way out: 32 columns of each of the stripe's 64 rows, column c of
// row r at (c + rot(r)) & 31 (the rotation by 16 on every other pair of rows lets the
// 16-byte reads below use all banks).  A chunk writes columns c - 15 .. c of row r, c = t_hi - r,
// which completes the row's 16-column segment that holds c: each row gets one whole
// segment per chunk, 64-byte aligned in memory wherever the row is.
struct OutTile {
    float v[64 * 32];
    __device__ static int rot(int r) { return (r & 2) << 3; }
};
__device__ __forceinline__ void clear_out(OutTile* o, int lane) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
        reinterpret_cast<f32x4*>(o->v)[64 * i + lane] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
}
// Stores row segments: lane l's q[i] is quarter l % 4 of columns 16 (kf - i) .. + 15 of
// row 16 i + l / 4.
__device__ __forceinline__ void store_quads(const f32x4 (&q)[4], float* obase, float* spare,
                                            int rows_left, int L2max, int lane, int kf) {
    const int r0 = lane >> 2, p4 = 4 * (lane & 3);
    uint32_t off = (uint32_t)(r0 * L2max + 16 * kf + p4) * 4u;
    const uint32_t step = (uint32_t)(16 * L2max - 16) * 4u;
    char* base = reinterpret_cast<char*>(obase);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int col = 16 * (kf - i) + p4;
        // (a quad outside the matrix goes to `spare`, 1 KB that nothing reads again: the
        // number of stores is fixed, so the compiler's waits for the loads issued before
        // them stay exact, and no line is written by more than one wave)
        const bool in = kf >= i && 16 * i + r0 < rows_left;
        char* dst = in && col + 4 <= L2max ? base + off
                                           : reinterpret_cast<char*>(spare + 4 * lane);
        *reinterpret_cast<f32x4*>(dst) = q[i];
        off += step;
    }
    if ((L2max & 3) != 0 && 16 * kf + 16 > (L2max & ~3)) {
        // the last 1 to 3 columns of a row
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = 16 * (kf - i) + p4;
            if (kf >= i && 16 * i + r0 < rows_left && col < L2max && col + 4 > L2max) {
                float* dst = obase + (size_t)(16 * i + r0) * L2max + col;
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (col + e < L2max) dst[e] = q[i][e];
            }
        }
    }
}

// Stores the segments that chunk kf completed: four lanes a row, 16 bytes each.
// rows_left: rows of the matrix from the stripe's first one.
__device__ __forceinline__ void store_segments(const OutTile* o, float* obase, float* spare, int rows_left,
                                               int L2max, int lane, int kf) {
    const int r0 = lane >> 2, p4 = 4 * (lane & 3);
    const float* src = o->v + 32 * r0 + p4;
    const int x0 = ((kf & 1) << 4) ^ OutTile::rot(r0), x1 = x0 ^ 16;
    f32x4 q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        q[i] = *reinterpret_cast<const f32x4*>(src + 512 * i + ((i & 1) ? x1 : x0));
    store_quads(q, obase, spare, rows_left, L2max, lane, kf);
}

// ------------------------------------------------------------------ results

// Value and parameter gradients of element b from the sums r: linear gaps {gaps (global:
// matches), -, sum P s}, affine {opens, extends (global: matches), sum P s}; S = T log Z.
// A global path of M matches has L1 + L2 - 2 M gaps.
template <Fam F>
__device__ inline void finalize(const Args& A, int b, int L1, int L2, const double* r, double S) {
    const bool empty = L1 <= 0 || L2 <= 0;
    double value = S, g0 = r[0], g1 = r[1], path = r[2];
    if constexpr (F == NW) {
        g0 = (double)(L1 + L2) - 2.0 * r[0];
        if (empty) value = g0 * A.gap;
        path += g0 * A.gap;
    } else if constexpr (F == NWAFF) {
        const int len = L1 + L2;
        g0 = empty ? (len > 0 ? 1.0 : 0.0) : r[0] + 1.0;
        g1 = (double)len - 2.0 * r[1] - g0;
        if (empty) value = g0 * A.gap + g1 * A.ext;
        path += g0 * A.gap + g1 * A.ext;
    } else if constexpr (F == SW) {
        path += g0 * A.gap;
    } else {
        path += g0 * A.gap + g1 * A.ext;
    }
    A.value[b] = (float)value;
    if (A.grad0) A.grad0[b] = (float)g0;
    if (A.grad1) A.grad1[b] = (float)g1;
    A.gradT[b] = (float)((value - path) / A.T);
}

// The element's partition, as mantissa in [1, 2) and exponent (zm = 0: out of range).
//
// Local affine gaps: a step from one kind of gap to the other has to match in between, so
// no detour of two gaps bounds what a factor below 2^kMinBits, which is not kept, would
// weigh.  Such a factor E may be left out if
//  * E Z is small: a path through its cell is an alignment before it and one behind it (and
//    gaps, of at most 1 each where they cost), of at most Z each, so its share of Z is at most
//    E Z;
//  * 2^-K, the restart term in the lanes' scale, is within the 64-bit range with room for
//    another factor (K is at most the exponent of Z, and of Z times the rows in the reverse
//    sweep): beside a cell without weight nothing else keeps a row from its neighbour's
//    scale.  What is lost below 2^-1022 of the scale is then nothing beside a restart.
template <Fam F>
__device__ __forceinline__ void element_partition(const Args& A, int b, double& zm, int& zk) {
    zm = 0.0;
    zk = -(1 << 28);
    float low = -FLT_MAX;
    for (int g = 0; g < A.G; ++g) {
        const double* zp = A.mem.zpart + ((size_t)b * A.G + g) * 3;
        const double z = zp[0];
        const int kz = (int)zp[1];
        if constexpr (F == AFF) low = fmaxf(low, (float)zp[2]);
        const int km = max(zk, kz);
        zm = scale2(zm, max(zk - km, -4000)) + scale2(z, max(kz - km, -4000));
        zk = km;
    }
    const int e = exponent(zm);
    if (zm > 0.0 && e < 1024) {
        zm = scale2(zm, -e);
        zk += e;
    } else {
        zm = 0.0;
    }
    if constexpr (F == AFF) {
        if (low > -FLT_MAX && (zk > kMaxMaskedExp || low > kNoShare - (float)zk)) zm = 0.0;
    }
}

// One thread: the part's sums to the results (one part) or to memory.
template <Fam F>
__device__ inline void finish_part(const Args& A, int b, int part, int L1, int L2, const double* r,
                                   double S) {
    for (int i = 0; i < 3; ++i)
        if (exponent(fabs(r[i])) == 1024) flag_redo(A.redo + b, REDO_BWD);
    if (A.G == 1) {
        finalize<F>(A, b, L1, L2, r, S);
    } else {
        double* bp = A.bpart + ((size_t)b * A.G + part) * 4;
        bp[0] = r[0];
        bp[1] = r[1];
        bp[2] = r[2];
        bp[3] = S;
    }
}

template <Fam F>
__device__ inline void poison(const Args& A, int b) {
    const float nan = __builtin_nanf("");
    const size_t n = (size_t)A.L1max * A.L2max;
    float* o = A.out + (size_t)b * n;
    for (size_t i = threadIdx.x; i < n; i += blockDim.x) o[i] = nan;
    if (threadIdx.x == 0) {
        A.value[b] = nan;
        if (A.grad0) A.grad0[b] = nan;
        if (A.grad1) A.grad1[b] = nan;
        A.gradT[b] = nan;
    }
}

// ------------------------------------------------------------------ reverse sweep

template <Fam F>
__global__ void __launch_bounds__((Traits<F>::AFFINE ? 4 : MAXW) * 64) bwd_kernel(const Args A) {
    using Tr = Traits<F>;
    constexpr bool GLOBAL = F == NW || F == NWAFF;
    extern __shared__ __align__(16) char smem[];
    __shared__ int prog[MAXW];
    __shared__ double red[3][MAXW];
    int b, dpart;
    split_decode(blockIdx.x, A.G, b, dpart);
    if (b >= A.B) return;
    const int part = A.G - 1 - dpart;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int L1, L2;
    element_lengths(A, b, L1, L2);
    const int NS = (L1 > 0 && L2 > 0) ? (L1 + 63) / 64 : 0;
    const int s0 = part * A.SPW;
    const int n = max(0, min(A.SPW, NS - s0));
    const int nch = chunks(L2);
    int* st = A.status + b;
    if (threadIdx.x < MAXW) prog[threadIdx.x] = -1;

    // Z of the element
    double zm = 0.0;
    int zk = -(1 << 28);
    element_partition<F>(A, b, zm, zk);
    if (!(zm > 0.0) && threadIdx.x == 0) flag_redo(A.redo + b, REDO_BWD);   // out of range
    const double invZ = 1.0 / zm;
    // S in units of T, from a 64-bit logarithm; every part that reports uses the same
    const double S = A.T * 0.693147180559945309417 * ((double)zk + log2(zm));
    float* obase = A.out + (size_t)b * A.L1max * A.L2max;
    zero_padding(obase, L1, L2, A.L1max, A.L2max, blockDim.x, min(s0 * 64, A.L1max),
                 part == A.G - 1 ? A.L1max : min((s0 + A.SPW) * 64, A.L1max));
    __syncthreads();

    Ring<Tr::NQ>* rings = reinterpret_cast<Ring<Tr::NQ>*>(smem);
    float* tiles = reinterpret_cast<float*>(rings + A.SPW + 1);
    OutTile* outs = reinterpret_cast<OutTile*>(tiles + A.SPW * (64 * P));
    double* rows0 = reinterpret_cast<double*>(outs + A.SPW);
    const int nchmax = chunks(A.L2max);
    const size_t sidx0 = (size_t)b * A.NSmax;
    const size_t brow_plane = (size_t)P * (nchmax + 1);
    const size_t flow_plane = (size_t)P * nchmax;
    const bool to = n > 0 && s0 > 0, from = n > 0 && s0 + n < NS;
    const int W_IN = A.SPW, W_OUT = A.SPW + 1;
    // an element given to the log-domain sweeps needs no reverse sweep here (its parts agree)
    const bool skip = __builtin_amdgcn_readfirstlane(zm > 0.0 ? A.redo[b] & REDO_FWD : 1) != 0;

    double gacc = 0.0, hacc = 0.0, pacc = 0.0;   // open (linear: gap), extend, sum of P s
    if (skip) {
    } else if (wave < n) {
        const int s = s0 + wave, i0 = 64 * s;
        const int rows = min(64, L1 - i0);
        const Ring<Tr::NQ>* rin = rings + wave + 1;
        Ring<Tr::NQ>* rout = rings + wave;
        const int prod = wave + 1 < n ? wave + 1 : (from ? W_IN : -1);
        const int cons = wave > 0 ? wave - 1 : (to ? W_OUT : -1);
        const bool ring_in = prod >= 0;
        const bool above = s > 0;
        float* tile = tiles + wave * (64 * P);
        double* rtile = rows0 + wave * (Tr::NP * P);
        const float* sbase = A.m + ((size_t)b * A.L1max + i0) * A.L2max;
        const long long room = ((long long)(A.B - b) * A.L1max - i0) * (long long)A.L2max;
        const int L1left = A.L1max - i0;
        double* ckb = A.mem.ck + (sidx0 + s) * nchmax * 64 * (Tr::NV + 1);
        const double* ck = ckb + lane * (Tr::NV + 1);
        // where quads outside the matrix go: a checkpoint that has been read
        auto spare = [&](int kf) {
            return reinterpret_cast<float*>(ckb + (size_t)kf * 64 * (Tr::NV + 1));
        };
        const int* kx = A.mem.kx + (sidx0 + s) * nchmax * 64 + lane;
        const double* brow = A.mem.brow + (sidx0 + s - (above ? 1 : 0)) * Tr::NP * brow_plane;
        const int* kup = A.mem.kx + (sidx0 + s - (above ? 1 : 0)) * nchmax * 64 + 63;
        const bool lane_ok = lane < rows;
        const bool owns_end = s == NS - 1;
        const int lane_end = rows - 1, t_end = L2 - 1 + lane_end;
        float* srow = obase + (size_t)i0 * A.L2max;
        OutTile* ot = outs + wave;
        clear_out(ot, lane);
        char* orow = reinterpret_cast<char*>(ot->v + 32 * lane);

        // own state: y = E b (of M, affine) and its previous step's yo; bb = b (bI, affine);
        // bd = bD.  Passed up: w, what the row above takes from this column and the next,
        //   linear gap  y[j+1] + g b[j];  affine  y[j+1] (and bI[j])
        double y = 0.0, bb = 0.0, bd = 0.0, w = 0.0;
        int K = 0;

        // one chunk's inputs, loaded a chunk ahead
        f32x4 sq[P / 4];
        double cv[Tr::NV + 1], rw[Tr::NP];
        int ckx, kk;
        auto load = [&](int kf) {
            stage_chunk(sq, sbase, room, L1left, A.L2max, lane, kf * P);
            const double* c = ck + (size_t)kf * 64 * (Tr::NV + 1);
#pragma unroll
            for (int i = 0; i <= Tr::NV; ++i) cv[i] = c[i];
            ckx = kx[(size_t)kf * 64];
            const int grp = min(kf + 4, nch);
#pragma unroll
            for (int i = 0; i < Tr::NP; ++i) rw[i] = brow[i * brow_plane + grp * P + (lane & 15)];
            kk = kup[(size_t)min(kf + 3 + (lane & 1), nch - 1) * 64];
        };
        load(nch - 1);
        if (!ring_in) {          // nothing below: zero flows
            for (int i = lane; i < Tr::NQ * RING; i += 64) (&rings[wave + 1].v[0][0])[i] = 0.0;
        }
        Peek pk = peek(prog, prod, cons);
        int kr = 0;              // scale of the flows from below
        for (int kf = nch - 1, q = 0; kf >= 0; --kf, ++q) {
            const int t0 = kf * P;
            const bool full = rows == 64 && t0 >= 63 && t0 + P <= L2;
            put_chunk(tile, sq, lane);
            if (lane < P) {
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i) rtile[i * P + lane] = above ? rw[i] : 0.0;
            }
            double v[Tr::NV], p[Tr::NP], d = cv[Tr::NV];
#pragma unroll
            for (int i = 0; i < Tr::NV; ++i) v[i] = cv[i];
            const int Kf = ckx;
            const int ka3 = __builtin_amdgcn_readlane(kk, 0);
            int ka4 = __builtin_amdgcn_readlane(kk, 1);
            // the previous chunk's marginals leave before the next loads are issued: the
            // wait for those loads a chunk later finds both long done
            if (q > 0)
                store_segments(ot, srow, spare(kf + 1), A.L1max - i0, A.L2max, lane, kf + 1);
            load(max(kf - 1, 0));
            __asm__ volatile("" ::: "memory");
            // the lane's scores of steps 4 q0 .. 4 q0 + 3 (read in both passes over the chunk)
            auto scores = [&](int q0) {
                return *reinterpret_cast<const f32x4*>(tile + QuadTile<P>::slot(lane, q0));
            };
            // (without a stripe above: zeros, which rtile holds, or the row-0 gap run)
            double edge = 0.0;
            if (!above) {
                ka4 = 0;
                if (GLOBAL) {
                    const double e = edge_log2<F>(A.k, kf * P + 1);
                    ka4 = (int)floor(e);
                    edge = exp2(e - (double)ka4);
                }
            }
            auto row_above = [&](int q0, double (&r)[Tr::NP][4]) {
                if (GLOBAL && !above) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        r[0][j] = edge;
                        if (F == NWAFF) r[Tr::NP - 1][j] = A.k.o * edge;
                        edge *= F == NW ? A.k.g : A.k.e;
                    }
                    return;
                }
#pragma unroll
                for (int i = 0; i < Tr::NP; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) r[i][j] = rtile[i * P + 4 * q0 + j];
            };

            // the chunk's scale for b, as in the forward: lanes not started take that of the
            // lowest started one (while there is none, the ring's: its first values have to
            // be waited for here), lanes past the element's rows that of the last row
            const int first = max((kf + 1) * P - L2 + 1, 0);    // lowest started lane
            int kra = kr;
            if (first >= rows) {
                wait_chunk(pk, prog, prod, cons, q, nch, st);
                if (ring_in && q == 0)
                    kra = __builtin_amdgcn_readfirstlane(rin->k[(kf - 3) & (RCH - 1)]);
                if (ring_in) kr = __builtin_amdgcn_readfirstlane(rin->k[max(kf - 4, 0) & (RCH - 1)]);
            }
            {
                const int ex = exponent(bb);
                int Kn = K + (ex > -1023 && ex < 1024 ? ex : 0);
                if (first > 0 || rows < 64) {
                    const int kb = first < rows ? __builtin_amdgcn_readlane(Kn, min(first, 63)) : kr;
                    if (lane < first) Kn = kb;
                    const int kl = __builtin_amdgcn_readlane(Kn, rows - 1);
                    if (lane >= rows) Kn = kl;
                }
                const int delta = K - Kn;
                y = scale2(y, delta);
                w = scale2(w, delta);
                bb = scale2(bb, delta);
                if (Tr::AFFINE) bd = scale2(bd, delta);
                K = Kn;
            }
            const double one = Tr::LOCAL ? scale2(1.0, -K) : 0.0;

            // recompute in the scale in which a b is the marginal: 2^-K / Z
            FwdIn<F> in;
            {
                const int sum = Kf + K;
#pragma unroll
                for (int i = 0; i < Tr::NV; ++i) v[i] = scale2(v[i] * invZ, sum - zk);
                const int su = shr1(sum, 0) - zk;
                if (lane > 0) d = scale2(d * invZ, su);
                const int Kb_up = shr1(K, 0);
                const bool top = above || GLOBAL;     // (else zeros come from above)
                in.f = lane > 0 ? scale2(1.0, K - Kb_up)
                                : (top ? scale2(invZ, ka4 + K - zk) : 0.0);
                in.gf = A.k.g * in.f;
                in.one = Tr::LOCAL ? scale2(invZ, K - zk) : 0.0;
                fwd_pass<F>(A.k, v, p);
            }
            double E[P], t1[P], t3[P], vi[Tr::AFFINE ? P : 1], vd[Tr::AFFINE ? P : 1];
            float ps = 0.0f;
            const uint32_t oaddr = (uint32_t)(t0 - lane + OutTile::rot(lane)) * 4u;
            // (boundary values are read four steps at a time, a group ahead: the empty asm
            // statements keep the reads where they are, so that few are live at once)
            auto chunk = [&](auto full_tag) {
                constexpr bool FULL = decltype(full_tag)::value;
                double rq[2][Tr::NP][4];
                f32x4 sq4[2];
                sq4[0] = scores(0);
                row_above(0, rq[0]);
                if (above) {
#pragma unroll
                    for (int i = 0; i < Tr::NP; ++i) rq[0][i][0] = scale2(rq[0][i][0], ka3 - ka4);
                }
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    if (j % 4 == 0 && j + 4 < P) {
                        __asm__ volatile("" ::: "memory");
                        row_above(j / 4 + 1, rq[(j / 4 + 1) & 1]);
                        sq4[(j / 4 + 1) & 1] = scores(j / 4 + 1);
                    }
                    const int col = t0 + j - lane;
                    const bool ok = FULL || (lane_ok && col >= 0 && col < L2);
                    const float x = sq4[(j / 4) & 1][j & 3] * A.k.c;
                    E[j] = (double)fast_exp2(x);
                    double u[Tr::NP], vn[Tr::NV];
#pragma unroll
                    for (int i = 0; i < Tr::NP; ++i) u[i] = shr1(p[i], rq[(j / 4) & 1][i][j & 3]);
#pragma unroll
                    for (int i = 0; i < Tr::NV; ++i) vn[i] = v[i];
                    fwd_cell<F>(A.k, in, E[j], d, u, vn, t1[j], t3[j]);
                    // opens that leave column 0
                    if (F == NWAFF && !FULL) t3[j] = col == 0 ? A.k.o * v[Tr::NV > 1 ? 1 : 0] : 0.0;
#pragma unroll
                    for (int i = 0; i < Tr::NV; ++i) v[i] = ok ? vn[i] : v[i];
                    if constexpr (Tr::AFFINE) {
                        vi[j] = v[1];
                        vd[j] = v[2];
                    }
                    fwd_pass<F>(A.k, v, p);
                    d = u[0];
                }

                // the reverse pass: flows from below, four steps at a time
                if (!(first >= rows)) {
                    wait_chunk(pk, prog, prod, cons, q, nch, st);
                    // (kr is the scale of the producer's chunk kf - 4, the previous chunk's of
                    // its chunk kf - 3, to which the last of the 16 values belongs)
                    if (ring_in)
                        kr = __builtin_amdgcn_readfirstlane(rin->k[max(kf - 4, 0) & (RCH - 1)]);
                }
                double fl[2][Tr::NQ][4];
                auto flows = [&](int q0, double (&r)[Tr::NQ][4]) {
                    const int base = ((kf - 3) & (RCH - 1)) * P + 4 * q0;
#pragma unroll
                    for (int i = 0; i < Tr::NQ; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j) r[i][j] = rin->v[i][base + j];
                };
                flows(P / 4 - 1, fl[(P / 4 - 1) & 1]);
                sq4[(P / 4 - 1) & 1] = scores(P / 4 - 1);
                int krd = kra - kr;
                if (!ring_in) krd = 0;
                if (!ring_in) kr = __builtin_amdgcn_readlane(K, 63);   // (zeros from below)
#pragma unroll
                for (int i = 0; i < Tr::NQ; ++i)
                    fl[(P / 4 - 1) & 1][i][3] = scale2(fl[(P / 4 - 1) & 1][i][3], krd);
                const double fb = scale2(1.0, shl1(K, kr) - K);
                const double ofb = A.k.o * fb, efb = A.k.e * fb;
                double wh[Tr::NQ][4];
#pragma unroll
                for (int j = P - 1; j >= 0; --j) {
                    const int z = (j / 4) & 1, e = j & 3;
                    if (e == 3 && j > 3) {
                        __asm__ volatile("" ::: "memory");
                        flows(j / 4 - 1, fl[(j / 4 - 1) & 1]);
                        sq4[(j / 4 - 1) & 1] = scores(j / 4 - 1);
                    }
                    // (read before the last steps, so that it has arrived at the chunk's end)
                    if (j == 3) pk = peek(prog, prod, cons);
                    const int col = t0 + j - lane;
                    const bool ok = FULL || (lane_ok && col >= 0 && col < L2);
                    const bool end = !FULL && !Tr::LOCAL && owns_end && lane == lane_end &&
                                     t0 + j == t_end;
                    const double wd = shl1(w, fl[z][0][e]);
                    double Pm, yn, gt = 0.0, ht = 0.0;
                    if constexpr (F == SW || F == NW) {
                        double bn = F == SW ? __builtin_fma(A.k.g, bb, one) : A.k.g * bb;
                        if (F == NW && end) bn = scale2(1.0, -K);
                        bn = __builtin_fma(fb, wd, bn);
                        if (!FULL) bn = ok ? bn : 0.0;
                        yn = E[j] * bn;
                        if (!FULL) yn = ok ? yn : 0.0;
                        Pm = t1[j] * yn;
                        if (!FULL) Pm = ok ? Pm : 0.0;
                        // NW: the matches, whose sum gives the gaps
                        if (F == NW) gacc += Pm;
                        else gacc = __builtin_fma(FULL || ok ? t3[j] : 0.0, bn, gacc);
                        w = __builtin_fma(A.k.g, bn, y);
                        bb = bn;
                    } else {
                        const double bi = shl1(bb, fl[z][Tr::NQ - 1][e]);      // bI of (i+1, j)
                        const double w0 = F == AFF ? __builtin_fma(fb, wd, one) : fb * wd;
                        const double wv = end ? scale2(1.0, -K) : w0;
                        const double qi = efb * bi, qd = A.k.e * bd;
                        const double qo = ofb * bi, qr = A.k.o * bd;
                        const double qm = qo + qr;
                        double nI = wv + qi, nD = wv + qd;
                        if (F == NWAFF) {
                            nI += qr;
                            nD += qo;
                        }
                        yn = E[j] * (wv + qm);
                        if (!FULL) yn = ok ? yn : 0.0;
                        Pm = t1[j] * yn;
                        if (!FULL) Pm = ok ? Pm : 0.0;
                        gt = (t1[j] * E[j]) * qm;
                        ht = F == AFF ? __builtin_fma(vi[j], qi, vd[j] * qd) : Pm;
                        if (F == NWAFF) {
                            gt = __builtin_fma(vi[j], qr, __builtin_fma(vd[j], qo, gt));
                            if (!FULL) {
                                gt = __builtin_fma(t3[j], nD, gt);      // from column 0
                                if (!above && lane == 0) {              // from row 0
                                    gt = __builtin_fma(vi[j], nI, gt);
                                    if (col == 0) gt -= Pm;             // starts with a match
                                }
                            }
                        }
                        if (!FULL) {
                            gt = ok ? gt : 0.0;
                            ht = ok ? ht : 0.0;
                            nI = ok ? nI : 0.0;
                            nD = ok ? nD : 0.0;
                        }
                        gacc += gt;
                        hacc += ht;
                        w = y;
                        bb = nI;
                        bd = nD;
                    }
                    y = yn;
                    wh[0][e] = w;
                    if (Tr::NQ > 1) wh[Tr::NQ - 1][e] = bb;
                    const float pf = (float)Pm;
                    *reinterpret_cast<float*>(orow + ((oaddr + 4u * j) & 124u)) = pf;
                    ps = fmaf(pf, FULL || ok ? sq4[z][e] : 0.0f, ps);
                    if (e == 0) {
                        // (sums up to date: their terms are not kept for later)
                        __asm__ volatile("" : "+v"(gacc), "+v"(hacc), "+v"(ps));
                        // the four flows to the stripe above (slot of step t: t + 15)
                        if (lane == 0) {
                            const int g0 = (kf & (RCH - 1)) * P, g1 = ((kf + 1) & (RCH - 1)) * P;
#pragma unroll
                            for (int i = 0; i < Tr::NQ; ++i)
#pragma unroll
                                for (int t = j; t < j + 4; ++t)
                                    rout->v[i][t < 1 ? g0 + P - 1 : g1 + t - 1] = wh[i][t - j];
                        }
                    }
                }
                if (lane == 0) rout->k[kf & (RCH - 1)] = K;
            };
            if (full && !(F == NWAFF && !above)) chunk(std::true_type{});
            else chunk(std::false_type{});
            post(prog, wave, q + 1);
            if (__builtin_amdgcn_ballot_w64(ps != ps) != 0) {
                // -inf scores, whose marginals are 0: the sum again, of finite scores.  (One test
                // a chunk; a clamp of every score would be one instruction a cell.)
                int l = lane;
                __asm__ volatile("" : "+v"(l));   // (rare: nothing of it is kept across chunks)
                const float* marg = ot->v + 32 * l;
                ps = 0.0f;
#pragma unroll 1
                for (int j = P - 1; j >= 0; --j)
                    ps = fmaf(marg[(t0 - l + OutTile::rot(l) + j) & 31],
                              __builtin_amdgcn_fmed3f(tile[QuadTile<P>::slot(l, j / 4) + (j & 3)],
                                                      -FLT_MAX, FLT_MAX),
                              ps);
            }
            pacc += (double)ps;
            __asm__ volatile("" ::: "memory");
        }
        store_segments(ot, srow, spare(0), A.L1max - i0, A.L2max, lane, 0);
    } else if (wave == W_IN && from) {
        import_boundary<Tr::NQ, false>(rings + n, A.mem.flow + ((size_t)b * A.G + part + 1) * Tr::NQ * flow_plane,
                                       flow_plane, A.mem.kflow + ((size_t)b * A.G + part + 1) * nchmax,
                                       A.bflag + (size_t)b * A.G + part + 1, A.epoch, prog, W_IN,
                                       n - 1, nch, lane, st);
    } else if (wave == W_OUT && to) {
        export_boundary<Tr::NQ, false>(rings, A.mem.flow + ((size_t)b * A.G + part) * Tr::NQ * flow_plane,
                                       flow_plane, A.mem.kflow + ((size_t)b * A.G + part) * nchmax,
                                       A.bflag + (size_t)b * A.G + part, A.epoch, prog, W_OUT, 0,
                                       nch, lane, st);
    }

    gacc = wave_sum(gacc);
    hacc = wave_sum(hacc);
    pacc = wave_sum(pacc);
    if (lane == 0) {
        red[0][wave] = gacc;
        red[1][wave] = hacc;
        red[2][wave] = pacc;
    }
    __syncthreads();
    __shared__ int poison_flag;
    if (threadIdx.x == 0) {
        double r[3] = {0.0, 0.0, 0.0};
        for (int w = 0; w < n; ++w)
            for (int i = 0; i < 3; ++i) r[i] += red[i][w];
        finish_part<F>(A, b, part, L1, L2, r, S);
    }
    if (A.G > 1) return;
    // an element whose waits gave up: NaN everywhere
    wait_vmcnt<0>();
    __syncthreads();
    if (threadIdx.x == 0) poison_flag = load_status(st);
    __syncthreads();
    if (poison_flag != 0) poison<F>(A, b);
}

// ------------------------------------------------------------------ two waves a stripe

// Families with one state (linear gaps) run two waves per
// stripe: a sweeping wave that carries the recurrence and nothing else, and a helper on
// the same SIMD that does what does not depend on it (loads, exponentials, the last row
// and, in the reverse sweep, the recomputation and the marginals).  A lone wave issues
// one instruction every 5-6 cycles, so everything taken off the sweeping wave shortens
// the pipeline: its hand-off to the next stripe, five chunks later, is what an
// element's time is made of.
constexpr int MAXW2 = 16;           // waves per workgroup
constexpr int MAXS = 8;             // stripes
constexpr int ROOMY = 4;            // stripes that have a SIMD each
constexpr int SINK = 64 + P;        // doubles that the lanes beside a ring's write into
constexpr int NTF = 4;              // factor tiles of a forward stripe
constexpr int NTB = 4;              // ... of a reverse stripe
constexpr int NBB = 2;              // its b buffers: the sweep runs on while marginals are made
constexpr int BROW = 132;           // floats per step of the b buffer (528 bytes: no bank is
                                    // hit twice when rows of 16 steps are read back)
constexpr int BBUF = P * BROW;      // floats of one b buffer
// progress words (LDS): stripes' chunks swept, tiles ready, b buffers consumed, copying waves,
// marginals made
enum { PW_SWEEP = 0, PW_TILE = 8, PW_USED = 16, PW_IN = 24, PW_OUT = 25, PW_NONE = 26,
       PW_MARG = 27, PW_COUNT = 35 };

// LDS floats of one stripe (without its ring)
constexpr int FWD2_FLOATS = NTF * 64 * P;
constexpr int BWD2_FLOATS = NTB * 64 * P + NBB * (BBUF + 64) + 2 * P;

// Factors E = 2^(c s) of a chunk, in the layout its scores were loaded in.
__device__ __forceinline__ void to_factors(f32x4 (&q)[P / 4], float c) {
#pragma unroll
    for (int i = 0; i < P / 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) q[i][e] = fast_exp2(q[i][e] * c);
}

template <Fam F>
__device__ __forceinline__ void fwd2_sweep(const Args& A, int b, int part) {
    using Tr = Traits<F>;
    static_assert(Tr::NP == 1 && Tr::NV == 1, "one state");
    extern __shared__ __align__(16) char smem[];
    __shared__ int prog[PW_COUNT];
    __shared__ double sink[SINK];
    __shared__ double zred[MAXS];
    __shared__ int kred[MAXS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int L1, L2;
    element_lengths(A, b, L1, L2);
    const int NS = (L1 > 0 && L2 > 0) ? (L1 + 63) / 64 : 0;
    const int s0 = part * A.SPW;
    const int n = max(0, min(A.SPW, NS - s0));      // stripes of this part
    const int nch = chunks(L2);
    int* st = A.status + b;
    if (threadIdx.x == 0 && A.G == 1) {
        *st = 0;
        A.redo[b] = 0;
    }
    if (threadIdx.x < PW_COUNT) prog[threadIdx.x] = threadIdx.x == PW_NONE ? INT_MAX : -1;
    __syncthreads();

    Ring<1>* rings = reinterpret_cast<Ring<1>*>(smem);
    float* tiles = reinterpret_cast<float*>(rings + A.SPW + 1);
    const int nchmax = chunks(A.L2max);
    const size_t sidx0 = (size_t)b * A.NSmax;
    const size_t brow_len = (size_t)P * (nchmax + 1);
    const bool from = n > 0 && s0 > 0, to = n > 0 && s0 + n < NS;

    if (wave < n) {
        // ---- sweeping wave
        const int s = s0 + wave, i0 = 64 * s;
        const int rows = min(64, L1 - i0);
        const Ring<1>* rin = rings + wave;
        Ring<1>* rout = rings + wave + 1;
        const bool ring_in = wave > 0 || from;
        const int prod = wave > 0 ? PW_SWEEP + wave - 1 : (from ? PW_IN : PW_NONE);
        const int cons = wave + 1 < n ? PW_SWEEP + wave + 1 : (to ? PW_OUT : PW_NONE);
        const float* tile = tiles + wave * FWD2_FLOATS;
        double* ck = A.mem.ck + (sidx0 + s) * nchmax * 128;
        int* kx = A.mem.kx + (sidx0 + s) * nchmax * 64;
        const bool lane_ok = lane < rows;
        const unsigned lim = lane_ok ? (unsigned)L2 : 0u;
        const bool owns_end = s == NS - 1;
        const int lane_end = rows - 1, t_end = L2 - 1 + lane_end;

        if (!ring_in) {          // nothing above: zeros
            for (int i = lane; i < RING; i += 64) rings[wave].v[0][i] = 0.0;
        }
        double zsum = 0.0;      // the lane's share of the partition, scaled by 2^-zk
        int zk = -(1 << 28);
        double v = 0.0, d = 0.0;
        int K = 0;
        if constexpr (F == NW) {                    // column 0: a run of row + 1 gaps
            const double e = edge_log2<F>(A.k, i0 + lane + 1);
            K = (int)floor(e);
            v = exp2(e - (double)K);
        }
        int kr_prev = 0;        // scale of lane 0's boundary inputs, previous chunk
        int pp = -1, pc = -1, ph = -1;
        for (int k = 0; k < nch; ++k) {
            if (__builtin_amdgcn_readfirstlane(pp) < min(k + LEAD, nch))
                wait_for(prog, prod, min(k + LEAD, nch), st);
            if (k > 2 + RCH && __builtin_amdgcn_readfirstlane(pc) < k - 2 - RCH)
                wait_for(prog, cons, k - 2 - RCH, st);
            if (__builtin_amdgcn_readfirstlane(ph) < k + 1)
                wait_own(prog, PW_TILE + wave, k + 1, st);
            float E[P];
            read_quads<P, 1>(tile + (k % NTF) * (64 * P), lane, E);
            // boundary inputs of lane 0 and their scale; they are read four steps at a time, a
            // group ahead (the empty asm statements keep the reads where they are)
            int kr = 0, ka = 0;
            if (ring_in) {
                kr = __builtin_amdgcn_readfirstlane(rin->k[min(k + 4, nch - 1) & (RCH - 1)]);
                // (the first value is the last one of the producer's chunk before, whose
                // scale was the previous chunk's)
                ka = k > 0 ? kr_prev
                           : __builtin_amdgcn_readfirstlane(rin->k[min(3, nch - 1) & (RCH - 1)]);
            } else if (F == NW) {                    // row 0: a run of j gaps, put in the ring
                kr = (int)floor(edge_log2<F>(A.k, k * P + 1));
                if (lane < P)
                    rings[wave].v[0][((k + 4) & (RCH - 1)) * P + lane] =
                        exp2(edge_log2<F>(A.k, k * P + 1 + lane) - (double)kr);
                __asm__ volatile("" ::: "memory");
            }
            const double* rsrc = &rin->v[0][((k + 4) & (RCH - 1)) * P];
            auto row_above = [&](int g, double (&r)[4]) {
#pragma unroll
                for (int e = 0; e < 4; ++e) r[e] = rsrc[4 * g + e];
            };
            double rq[2][4];
            row_above(0, rq[0]);
            if (ring_in) rq[0][0] = scale2(rq[0][0], ka - kr);

            // the chunk's scale: the exponent of the lane's current value; lanes that have
            // not started take that of the lowest started lane (or the ring's).  Infinities
            // and NaN stay: they are looked for after the last chunk
            const int ex = exponent(v);
            int Kn = K + (ex > -1023 && ex < 1024 ? ex : 0);
            if (Tr::LOCAL) Kn = max(Kn, kMinExp);
            if (Tr::LOCAL && k < 64 / P) {
                const int kb = k == 0 ? kr : __builtin_amdgcn_readlane(Kn, max(k * P - 1, 0));
                if (lane >= k * P) Kn = kb;
            }
            // lane 0's diagonal input at its first cell: the cell above column 0 (other lanes
            // have it from the lane above)
            if (k == 0) {
                kr_prev = kr;
                if constexpr (F == NW) {
                    const double e = i0 > 0 ? edge_log2<F>(A.k, i0) : 0.0;
                    const int ke = (int)floor(e);
                    d = scale2(exp2(e - (double)ke), ke - kr);
                }
            }
            // (zeros from above the first stripe: any finite factor will do)
            if (!ring_in && Tr::LOCAL) kr = __builtin_amdgcn_readlane(Kn, 0);
            const int delta = K - Kn;
            v = scale2(v, delta);
            d = scale2(d, shr1(delta, kr_prev - kr));
            kr_prev = kr;
            K = Kn;
            FwdIn<F> in;
            in.f = scale2(1.0, shr1(Kn, kr) - Kn);
            in.gf = A.k.g * in.f;
            in.one = Tr::LOCAL ? scale2(1.0, -Kn) : 0.0;
            // checkpoint: the state that enters the chunk
            reinterpret_cast<double2*>(ck)[(unsigned)(k * 64 + lane)] = make_double2(v, d);
            kx[(unsigned)(k * 64 + lane)] = Kn;

            const int t0 = k * P;
            const bool full = rows == 64 && t0 >= 63 && t0 + P <= L2;
            // (lane 63 writes the ring; the others, in the same instructions, a sink)
            double* w0 = lane == 63 ? &rout->v[0][(k & (RCH - 1)) * P] : sink + lane;
            double* w1 = lane == 63 ? &rout->v[0][((k + 1) & (RCH - 1)) * P] : sink + lane;
            double hist[4];
            double zc = 0.0;
            auto steps = [&](auto full_tag) {
                constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    // (read before the last steps, so that it has arrived at the chunk's end)
                    if (j == P - 4) {
                        pp = prog_peek(prog, prod);
                        pc = prog_peek(prog, cons);
                        ph = prog_peek(prog, PW_TILE + wave);
                    }
                    if (j % 4 == 0 && j + 4 < P) {
                        __asm__ volatile("" ::: "memory");
                        row_above(j / 4 + 1, rq[(j / 4 + 1) & 1]);
                    }
                    const double u = shr1(v, rq[(j / 4) & 1][j & 3]);
                    double t1, t3, vn = v;
                    fwd_cell<F>(A.k, in, (double)E[j], d, &u, &vn, t1, t3);
                    if (FULL) {
                        v = vn;
                        if (Tr::LOCAL) zc += v;
                    } else {
                        // (left of the element a lane keeps its boundary value, 0 but for
                        // global alignment; right of it nothing valid reads it)
                        const bool ok = (unsigned)(t0 + j - lane) < lim;
                        v = ok ? vn : (F == NW ? v : 0.0);
                        if (Tr::LOCAL) zc += v;
                        else if (owns_end && t0 + j == t_end && lane == lane_end) {
                            zsum = v;
                            zk = Kn;
                        }
                    }
                    d = u;
                    hist[j & 3] = v;
                    // the last row to the stripe below and to the helper, which stores it
                    if ((j & 3) == 3) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int i = j - 3 + e;
                            if (i < P - 1) w0[1 + i] = hist[e];
                            else w1[0] = hist[e];
                        }
                    }
                }
            };
            if (lane == 63) rout->k[k & (RCH - 1)] = Kn;
            if (full) steps(std::true_type{});
            else steps(std::false_type{});
            post(prog, PW_SWEEP + wave, k + 1);
            if (Tr::LOCAL) {
                const int kz = max(zk, Kn);
                zsum = scale2(zsum, max(zk - kz, -4000)) + scale2(zc, Kn - kz);
                zk = kz;
            }
        }
        // values out of range
        if (__builtin_amdgcn_ballot_w64(lane_ok && exponent(v) == 1024) != 0 && lane == 0)
            flag_redo(A.redo + b, REDO_FWD);
        // the wave's share of the partition
        int km = zk;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) km = max(km, __shfl_xor(km, off, 64));
        zsum = wave_sum(scale2(zsum, max(zk - km, -4000)));
        if (lane == 0) {
            zred[wave] = zsum;
            kred[wave] = km;
        }
    } else if (wave >= A.SPW && wave < A.SPW + n) {
        // ---- helper: loads two chunks ahead, scores to factors, last rows to memory
        const int h = wave - A.SPW;
        const int s = s0 + h, i0 = 64 * s;
        float* tile = tiles + h * FWD2_FLOATS;
        const uint32_t tile_lds = lds_address(tile);
        const float* sbase = A.m + ((size_t)b * A.L1max + i0) * A.L2max;
        const long long room =
            ((long long)(A.B - b) * A.L1max - i0) * (long long)A.L2max;
        const int L1left = A.L1max - i0;
        const Ring<1>* rout = rings + h + 1;
        double* brow = A.mem.brow + (sidx0 + s) * brow_len;
        // (a part's last row: its exporting wave stores it)
        const bool keep = s + 1 < NS && h + 1 < n;
        int stored = 0;
        auto store_rows = [&](int upto) {
            for (; stored < upto; ++stored) {
                const int t = stored * P + (lane & (P - 1)) + 1;
                const double x = rout->v[0][t & (RING - 1)];
                if (keep && lane < P) brow[t] = x;
            }
        };
        for (int k = 0; k < nch + 2; ++k) {
            if (k >= NTF) {
                // tile k % NTF is free once its last chunk has been swept
                wait_own(prog, PW_SWEEP + h, min(k - NTF + 1, nch), st);
                store_rows(min(k - NTF + 1, nch));
            }
            dma_chunk(tile_lds + (k % NTF) * (64 * P * 4), sbase, room, L1left, A.L2max, lane,
                      min(k, nch - 1) * P);
            if (k >= 2) {
                wait_vmcnt<8>();                     // chunk k - 2's loads (two chunks follow)
                float* t = tile + ((k - 2) % NTF) * (64 * P);
                f32x4 q[P / 4];
#pragma unroll
                for (int i = 0; i < P / 4; ++i)
                    q[i] = reinterpret_cast<const f32x4*>(t)[64 * i + lane];
                to_factors(q, A.k.c);
                put_chunk(t, q, lane);
                post(prog, PW_TILE + h, k - 1);
            }
        }
        wait_own(prog, PW_SWEEP + h, nch, st);
        store_rows(nch);
        wait_vmcnt<0>();
    } else if (wave == 2 * A.SPW && from) {
        import_boundary<1, true>(rings, A.mem.brow + (sidx0 + s0 - 1) * brow_len, brow_len,
                                 A.mem.kexp + ((size_t)b * A.G + part - 1) * nchmax,
                                 A.fflag + (size_t)b * A.G + part - 1, A.epoch, prog, PW_IN,
                                 PW_SWEEP, nch, lane, st);
    } else if (wave == 2 * A.SPW + 1 && to) {
        export_boundary<1, true>(rings + n, A.mem.brow + (sidx0 + s0 + n - 1) * brow_len, brow_len,
                                 A.mem.kexp + ((size_t)b * A.G + part) * nchmax,
                                 A.fflag + (size_t)b * A.G + part, A.epoch, prog, PW_OUT,
                                 PW_SWEEP + n - 1, nch, lane, st);
    }

    __syncthreads();
    if (threadIdx.x == 0) {
        double z = 0.0;
        int kz = -(1 << 28);
        if (part == 0 && (Tr::LOCAL || NS == 0)) {   // the empty alignment
            z = 1.0;
            kz = 0;
        }
        for (int w = 0; w < n; ++w) {
            const int km = max(kz, kred[w]);
            z = scale2(z, max(kz - km, -4000)) + scale2(zred[w], max(kred[w] - km, -4000));
            kz = km;
        }
        double* zp = A.mem.zpart + ((size_t)b * A.G + part) * 3;
        zp[0] = z;
        zp[1] = (double)kz;
    }
}

template <Fam F>
__global__ void __launch_bounds__(MAXW2 * 64) fwd2_kernel(const Args A) {
    int b, part;
    split_decode(blockIdx.x, A.G, b, part);
    if (b < A.B) fwd2_sweep<F>(A, b, part);
}

// The end of a chunk of the reverse sweep: its marginals, which lie by step and lane in
// the rows of the b buffer, to memory, and the sum of P log2 E over the lane's cells
// (log2 E = c s, over the whole range of E: there is no marginal where it is 0, and where it is
// infinite the element is out of range).  Row r = 16 i + r0 completes its segment of
// columns 16 (kf - i) .. + 15: column 4 p + e of it was made in step n = 4 p + e + r0 of this
// chunk or, from 16 on, in step n - 16 of the chunk before, whose share is kept in cy.
// The buffer is free once everything has been read.
__device__ __forceinline__ double emit_chunk(float* bq, const float* tq, f32x4 (&cy)[P / 4],
                                             int lane, int kf, float* srow, float* spare,
                                             int rows_left, int L2max, int* prog, int word,
                                             int done) {
    int l = lane;
    __asm__ volatile("" : "+v"(l)::"memory");        // (addresses are not kept across chunks)
    const int r0 = l >> 2, p4 = 4 * (l & 3);
    f32x4 out[P / 4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int n = p4 + e + r0;
        const float* src = bq + (n & 15) * BROW + r0;
#pragma unroll
        for (int i = 0; i < P / 4; ++i) {
            const float x = src[16 * i];
            out[i][e] = n < 16 ? x : cy[i][e];
            cy[i][e] = x;
        }
    }
    float ps = 0.0f;
#pragma unroll
    for (int g = 0; g < P / 4; ++g) {
        const f32x4 E4 = *reinterpret_cast<const f32x4*>(tq + QuadTile<P>::slot(l, g));
#pragma unroll
        for (int e = 0; e < 4; ++e)
            ps = fmaf((bq + (4 * g + e) * BROW)[l],
                      fast_log2(__builtin_amdgcn_fmed3f(E4[e], FLT_MIN, FLT_MAX)), ps);
    }
    __asm__ volatile("" : "+v"(ps)::"memory");
    post(prog, word, done);
    store_quads(out, srow, spare, rows_left, L2max, l, kf);
    return (double)ps;
}

// Two helpers a stripe: a feeding wave makes the factors, two chunks ahead, and writes
// the marginals out, which the other one makes.  (One helper doing both was the
// pipeline's slowest stage: 43 against 36 us at [2, 100, 120], 95 against 85 at
// [48, 300, 411].)
template <Fam F>
__device__ __forceinline__ void bwd2_sweep(const Args& A, int b, int part) {
    using Tr = Traits<F>;
    static_assert(Tr::NP == 1 && Tr::NV == 1 && Tr::NQ == 1, "one state");
    extern __shared__ __align__(16) char smem[];
    __shared__ int prog[PW_COUNT];
    __shared__ double sink[SINK];
    __shared__ double red[2][MAXS];
    __shared__ int poison_flag;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int L1, L2;
    element_lengths(A, b, L1, L2);
    const int NS = (L1 > 0 && L2 > 0) ? (L1 + 63) / 64 : 0;
    const int s0 = part * A.SPW;
    const int n = max(0, min(A.SPW, NS - s0));
    const int nch = chunks(L2);
    int* st = A.status + b;
    if (threadIdx.x < PW_COUNT) prog[threadIdx.x] = threadIdx.x == PW_NONE ? INT_MAX : -1;

    // Z of the element
    double zm = 0.0;
    int zk = -(1 << 28);
    element_partition<F>(A, b, zm, zk);
    if (!(zm > 0.0) && threadIdx.x == 0) flag_redo(A.redo + b, REDO_BWD);
    float* obase = A.out + (size_t)b * A.L1max * A.L2max;
    zero_padding(obase, L1, L2, A.L1max, A.L2max, blockDim.x, min(s0 * 64, A.L1max),
                 part == A.G - 1 ? A.L1max : min((s0 + A.SPW) * 64, A.L1max));
    __syncthreads();

    Ring<1>* rings = reinterpret_cast<Ring<1>*>(smem);
    float* areas = reinterpret_cast<float*>(rings + A.SPW + 1);
    const int area = BWD2_FLOATS;
    const int nchmax = chunks(A.L2max);
    const size_t sidx0 = (size_t)b * A.NSmax;
    const size_t brow_len = (size_t)P * (nchmax + 1);
    const size_t flow_len = (size_t)P * nchmax;
    const bool to = n > 0 && s0 > 0, from = n > 0 && s0 + n < NS;
    // an element given to the log-domain sweeps needs no reverse sweep here (its parts agree)
    const bool skip = __builtin_amdgcn_readfirstlane(zm > 0.0 ? A.redo[b] & REDO_FWD : 1) != 0;

    if (skip) {
    } else if (wave < n) {
        // ---- sweeping wave: b and the flows
        const int s = s0 + wave, i0 = 64 * s;
        const int rows = min(64, L1 - i0);
        const Ring<1>* rin = rings + wave + 1;
        Ring<1>* rout = rings + wave;
        const bool ring_in = wave + 1 < n || from;
        const int prod = wave + 1 < n ? PW_SWEEP + wave + 1 : (from ? PW_IN : PW_NONE);
        const int cons = wave > 0 ? PW_SWEEP + wave - 1 : (to ? PW_OUT : PW_NONE);
        const float* tile = areas + wave * area;
        float* bbuf = areas + wave * area + NTB * 64 * P;
        const bool lane_ok = lane < rows;
        const unsigned lim = lane_ok ? (unsigned)L2 : 0u;
        const bool owns_end = s == NS - 1;
        const int lane_end = rows - 1, t_end = L2 - 1 + lane_end;
        if (!ring_in) {          // nothing below: zero flows
            for (int i = lane; i < RING; i += 64) rings[wave + 1].v[0][i] = 0.0;
        }
        // y = E b of the last cell and b; w: what the row above takes from a column and
        // the next, y[j+1] + g b[j]
        double y = 0.0, bb = 0.0, w = 0.0;
        int K = 0, kr = 0;
        int pp = -1, pc = -1, ph = -1, pu = -1;
        for (int kf = nch - 1, q = 0; kf >= 0; --kf, ++q) {
            if (__builtin_amdgcn_readfirstlane(pp) < min(q + LEAD, nch))
                wait_for(prog, prod, min(q + LEAD, nch), st);
            if (q > 2 + RCH && __builtin_amdgcn_readfirstlane(pc) < q - 2 - RCH)
                wait_for(prog, cons, q - 2 - RCH, st);
            if (__builtin_amdgcn_readfirstlane(ph) < q + 1)
                wait_own(prog, PW_TILE + wave, q + 1, st);
            const int t0 = kf * P;
            const bool full = rows == 64 && t0 >= 63 && t0 + P <= L2;
            float E[P];
            read_quads<P, 1>(tile + (q % NTB) * (64 * P), lane, E);
            const double* fsrc = &rin->v[0][((kf - 3) & (RCH - 1)) * P];
            double fl[2][4];
            auto flows = [&](int g) {
#pragma unroll
                for (int e = 0; e < 4; ++e) fl[g & 1][e] = fsrc[4 * g + e];
            };
            flows(P / 4 - 1);
            int krd = 0;
            if (ring_in) {
                // (the last of the 16 values belongs to the producer's chunk kf - 3, whose
                // scale was the previous chunk's, the others to its chunk kf - 4)
                const int kra = q == 0 ? __builtin_amdgcn_readfirstlane(
                                             rin->k[(kf - 3) & (RCH - 1)])
                                       : kr;
                kr = __builtin_amdgcn_readfirstlane(rin->k[max(kf - 4, 0) & (RCH - 1)]);
                krd = kra - kr;
            }
            // the chunk's scale, as in the forward: lanes not started take that of the lowest
            // started one (or the ring's), lanes past the element's rows that of the last row
            const int first = max((kf + 1) * P - L2 + 1, 0);    // lowest started lane
            const int ex = exponent(bb);
            int Kn = K + (ex > -1023 && ex < 1024 ? ex : 0);
            if (first > 0 || rows < 64) {
                const int kb = first < rows ? __builtin_amdgcn_readlane(Kn, min(first, 63)) : kr;
                if (lane < first) Kn = kb;
                const int kl = __builtin_amdgcn_readlane(Kn, rows - 1);
                if (lane >= rows) Kn = kl;
            }
            {
                const int delta = K - Kn;
                y = scale2(y, delta);
                w = scale2(w, delta);
                bb = scale2(bb, delta);
                K = Kn;
            }
            if (!ring_in) kr = __builtin_amdgcn_readlane(K, 63);   // (zeros from below)
            fl[(P / 4 - 1) & 1][3] = scale2(fl[(P / 4 - 1) & 1][3], krd);
            const double one = Tr::LOCAL ? scale2(1.0, -K) : 0.0;
            const double fb = scale2(1.0, shl1(K, kr) - K);
            // the b buffer must have been used
            const int bi = q % NBB;
            if (__builtin_amdgcn_readfirstlane(pu) < q + 1 - NBB)
                if (q >= NBB) wait_own(prog, PW_USED + wave, q + 1 - NBB, st);
            float* bq = bbuf + bi * (BBUF + 64);
            reinterpret_cast<int*>(bq)[BBUF + lane] = K;
            // (lane 0 writes the ring; the others, in the same instructions, a sink)
            double* w0 = lane == 0 ? &rout->v[0][(kf & (RCH - 1)) * P] : sink + lane;
            double* w1 = lane == 0 ? &rout->v[0][((kf + 1) & (RCH - 1)) * P] : sink + lane;
            double wh[4];
            auto steps = [&](auto full_tag) {
                constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
                for (int j = P - 1; j >= 0; --j) {
                    if (j == 3) {
                        pp = prog_peek(prog, prod);
                        pc = prog_peek(prog, cons);
                        ph = prog_peek(prog, PW_TILE + wave);
                        pu = prog_peek(prog, PW_USED + wave);
                    }
                    if ((j & 3) == 3 && j > 3) {
                        __asm__ volatile("" ::: "memory");
                        flows(j / 4 - 1);
                    }
                    const bool ok = FULL || (unsigned)(t0 + j - lane) < lim;
                    const double wd = shl1(w, fl[(j / 4) & 1][j & 3]);
                    double bn = F == SW ? __builtin_fma(A.k.g, bb, one) : A.k.g * bb;
                    if (!FULL && F == NW && owns_end && t0 + j == t_end && lane == lane_end)
                        bn = scale2(1.0, -K);
                    bn = __builtin_fma(fb, wd, bn);
                    if (!FULL) bn = ok ? bn : 0.0;
                    const double yn = (double)(FULL || ok ? E[j] : 0.0f) * bn;
                    w = __builtin_fma(A.k.g, bn, y);
                    bb = bn;
                    y = yn;
                    wh[j & 3] = w;
                    reinterpret_cast<double*>(bq + j * BROW)[lane] = bn;
                    // flows to the stripe above (slot of step t: t + 15)
                    if ((j & 3) == 0) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (j + e < 1) w0[P - 1] = wh[e];
                            else w1[j + e - 1] = wh[e];
                        }
                    }
                }
            };
            if (lane == 0) rout->k[kf & (RCH - 1)] = K;
            if (full) steps(std::true_type{});
            else steps(std::false_type{});
            post(prog, PW_SWEEP + wave, q + 1);
        }
    } else if (wave >= A.SPW && wave < A.SPW + n) {
        // ---- helper: the forward's values again and the marginals
        const int h = wave - A.SPW;
        const int s = s0 + h;
        const int rows = min(64, L1 - 64 * s);
        const unsigned lim = lane < rows ? (unsigned)L2 : 0u;
        const bool above = s > 0;
        const float* tile = areas + h * area;
        float* bbuf = areas + h * area + NTB * 64 * P;
        double* rtile = reinterpret_cast<double*>(bbuf + NBB * (BBUF + 64));
        const double* ck = A.mem.ck + (sidx0 + s) * nchmax * 128;
        const int* kx = A.mem.kx + (sidx0 + s) * nchmax * 64;
        const double* brow = A.mem.brow + (sidx0 + s - (above ? 1 : 0)) * brow_len;
        const int* kup = A.mem.kx + (sidx0 + s - (above ? 1 : 0)) * nchmax * 64 + 63;
        const double invZ = 1.0 / zm;
        double gacc = 0.0;

        double2 cv;
        double rw;
        int ckx, kk;
        auto load = [&](int kf) {                    // the chunk's checkpoint and row above
            cv = reinterpret_cast<const double2*>(ck)[(unsigned)(kf * 64 + lane)];
            ckx = kx[(unsigned)(kf * 64 + lane)];
            // (no row is longer than the element: what lies behind it in memory may be anything)
            const double x = brow[(unsigned)(min(kf + 4, nch) * P + (lane & 15))];
            rw = kf * P + (lane & 15) < L2 ? x : 0.0;
            kk = kup[(unsigned)(min(kf + 3 + (lane & 1), nch - 1) * 64)];
        };
        load(nch - 1);
        for (int kf = nch - 1, q = 0; kf >= 0; --kf, ++q) {
            const int t0 = kf * P;
            const bool full = rows == 64 && t0 >= 63 && t0 + P <= L2;
            const float* tq = tile + (q % NTB) * (64 * P);
            const int Kf = ckx;
            const int ka3 = __builtin_amdgcn_readlane(kk, 0);
            int ka4 = __builtin_amdgcn_readlane(kk, 1);
            double v = cv.x, d = cv.y;
            if (!above) {
                // zeros, or (global) the row-0 gap run
                ka4 = F == NW ? (int)floor(edge_log2<F>(A.k, kf * P + 1)) : 0;
                rw = F == NW ? exp2(edge_log2<F>(A.k, kf * P + 1 + (lane & 15)) - (double)ka4) : 0.0;
            }
            if (lane < P) rtile[lane] = rw;
            load(max(kf - 1, 0));

            // once the chunk has been swept: the forward's values again, in the scale in
            // which a b is the marginal (2^-K / Z, K the exponent of the lane's b)
            wait_own(prog, PW_SWEEP + h, q + 1, st);
            float* bq = bbuf + (q % NBB) * (BBUF + 64);
            FwdIn<F> in;
            {
                const int K = reinterpret_cast<const int*>(bq)[BBUF + lane];
                const int sum = Kf + K;
                v = scale2(v * invZ, sum - zk);
                const int su = shr1(sum, 0) - zk;
                if (lane > 0) d = scale2(d * invZ, su);
                const int K_up = shr1(K, 0);         // (not inside the select: every lane active)
                in.f = lane > 0 ? scale2(1.0, K - K_up) : scale2(invZ, ka4 + K - zk);
                if (Tr::LOCAL && !above && lane == 0) in.f = 0.0;
                in.gf = A.k.g * in.f;
                in.one = Tr::LOCAL ? scale2(invZ, K - zk) : 0.0;
            }
            auto marginals = [&](auto full_tag) {
                constexpr bool FULL = decltype(full_tag)::value;
                f32x4 E4[2];
                double r4[2][4], b4[2][4];
                auto read = [&](int g, int z) {
                    E4[z] = *reinterpret_cast<const f32x4*>(tq + QuadTile<P>::slot(lane, g));
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        b4[z][e] = reinterpret_cast<const double*>(bq + (4 * g + e) * BROW)[lane];
#pragma unroll
                    for (int e = 0; e < 4; ++e) r4[z][e] = rtile[4 * g + e];
                };
                read(0, 0);
                r4[0][0] = scale2(r4[0][0], above ? ka3 - ka4 : 0);
                // (eight steps a turn, in a loop that is kept rolled: registers)
#pragma unroll 1
                for (int gg = 0; gg < P / 4; gg += 2) {
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) {
                        const int z = jj / 4, e = jj & 3, j = 4 * gg + jj;
                        if (jj == 0) read(gg + 1, 1);
                        if (jj == 4) {
                            __asm__ volatile("" : "+v"(gacc)::"memory");
                            read(min(gg + 2, P / 4 - 1), 0);
                        }
                        const bool ok = FULL || (unsigned)(t0 + j - lane) < lim;
                        const double u = shr1(v, r4[z][e]);
                        double t1, t3, vn = v;
                        fwd_cell<F>(A.k, in, (double)E4[z][e], d, &u, &vn, t1, t3);
                        // (outside the element b is 0 and everything it is multiplied with finite)
                        v = ok ? vn : (F == NW ? v : 0.0);
                        d = u;
                        const double bs = b4[z][e];
                        const double Pm = (v - t3) * bs;
                        if (F == SW) gacc = __builtin_fma(t3, bs, gacc);
                        if (F == NW) gacc += Pm;
                        (bq + j * BROW)[lane] = (float)Pm;
                    }
                    __asm__ volatile("" : "+v"(gacc)::"memory");
                }
                __asm__ volatile("" ::: "memory");
            };
            if (full) marginals(std::true_type{});
            else marginals(std::false_type{});
            post(prog, PW_MARG + h, q + 1);
        }
        gacc = wave_sum(gacc);
        if (lane == 0) red[0][h] = gacc;
    } else if (wave >= 2 * A.SPW && wave < 2 * A.SPW + n) {
        // ---- feeding wave: scores two chunks ahead and their factors; the marginals out
        const int h = wave - 2 * A.SPW;
        const int i0 = 64 * (s0 + h);
        float* tile = areas + h * area;
        float* bbuf = areas + h * area + NTB * 64 * P;
        const uint32_t tile_lds = lds_address(tile);
        const float* sbase = A.m + ((size_t)b * A.L1max + i0) * A.L2max;
        const long long room = ((long long)(A.B - b) * A.L1max - i0) * (long long)A.L2max;
        double* ck = A.mem.ck + (sidx0 + s0 + h) * nchmax * 128;
        float* srow = obase + (size_t)i0 * A.L2max;
        double pacc = 0.0;
        f32x4 cy[P / 4];
#pragma unroll
        for (int i = 0; i < P / 4; ++i) cy[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        for (int it = 0; it < nch + NTB; ++it) {
            if (it >= 2 && it < nch + 2) {
                const int q = it - 2;
                wait_vmcnt<4>();                     // chunk q's loads (chunk q + 1's follow)
                float* t = tile + (q % NTB) * (64 * P);
                f32x4 f[P / 4];
#pragma unroll
                for (int i = 0; i < P / 4; ++i)
                    f[i] = reinterpret_cast<const f32x4*>(t)[64 * i + lane];
                to_factors(f, A.k.c);
                put_chunk(t, f, lane);
                post(prog, PW_TILE + h, q + 1);
            }
            if (it >= NTB) {
                // chunk it - NTB out: tile it % NTB is free after it
                const int q = it - NTB, kf = nch - 1 - q;
                wait_own(prog, PW_MARG + h, q + 1, st);
                pacc += emit_chunk(bbuf + (q % NBB) * (BBUF + 64),
                                   tile + (q % NTB) * (64 * P), cy, lane, kf, srow,
                                   reinterpret_cast<float*>(ck + (size_t)kf * 128), A.L1max - i0,
                                   A.L2max, prog, PW_USED + h, q + 1);
            }
            if (it < nch + 1)
                dma_chunk(tile_lds + (it % NTB) * (64 * P * 4), sbase, room, A.L1max - i0, A.L2max,
                          lane, max(nch - 1 - it, 0) * P);
        }
        wait_vmcnt<0>();
        pacc = wave_sum(pacc * (1.0 / (double)A.k.c));
        if (lane == 0) red[1][h] = pacc;
    } else if (wave == 3 * A.SPW && from) {
        import_boundary<1, false>(rings + n, A.mem.flow + ((size_t)b * A.G + part + 1) * flow_len,
                                  flow_len, A.mem.kflow + ((size_t)b * A.G + part + 1) * nchmax,
                                  A.bflag + (size_t)b * A.G + part + 1, A.epoch, prog, PW_IN,
                                  PW_SWEEP + n - 1, nch, lane, st);
    } else if (wave == 3 * A.SPW + 1 && to) {
        export_boundary<1, false>(rings, A.mem.flow + ((size_t)b * A.G + part) * flow_len, flow_len,
                                  A.mem.kflow + ((size_t)b * A.G + part) * nchmax,
                                  A.bflag + (size_t)b * A.G + part, A.epoch, prog, PW_OUT, PW_SWEEP,
                                  nch, lane, st);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r[3] = {0.0, 0.0, 0.0};
        if (!skip)
            for (int w = 0; w < n; ++w) {
                r[0] += red[0][w];
                r[2] += red[1][w];
            }
        element_partition<F>(A, b, zm, zk);
        finish_part<F>(A, b, part, L1, L2, r,
                       A.T * 0.693147180559945309417 * ((double)zk + log2(zm)));
    }
    if (A.G > 1) return;
    // an element whose waits gave up: NaN everywhere
    wait_vmcnt<0>();
    __syncthreads();
    if (threadIdx.x == 0) poison_flag = load_status(st);
    __syncthreads();
    if (poison_flag != 0) poison<F>(A, b);
}

template <Fam F>
__global__ void __launch_bounds__(3 * ROOMY * 64 + 128) bwd2_kernel(const Args A) {
    int b, dpart;
    split_decode(blockIdx.x, A.G, b, dpart);
    if (b < A.B) bwd2_sweep<F>(A, b, A.G - 1 - dpart);
}

// Both sweeps of elements of one part, in one launch: 46 us at [2, 100, 120], against 19 + 32
// and the gap between two launches.
template <Fam F>
__global__ void __launch_bounds__(3 * ROOMY * 64) both_kernel(const Args A) {
    int b, part;
    split_decode(blockIdx.x, 1, b, part);
    if (b >= A.B) return;
    fwd2_sweep<F>(A, b, 0);
    __threadfence_block();
    __syncthreads();
    bwd2_sweep<F>(A, b, 0);
}

// The end of a split element that stays here: sums its parts, or its poison pass.  Called by the
// kernel that redoes elements out of range, which every call launches: a launch less (NW [96,
// 301, 277], forward and backward: 186 -> 184 us).
template <Fam F>
__device__ inline void finish_element(const Args& A, int b) {
    if (A.G == 1) return;
    if (__builtin_amdgcn_readfirstlane(A.status[b]) != 0) {
        poison<F>(A, b);
        return;
    }
    if (threadIdx.x != 0) return;
    int L1, L2;
    element_lengths(A, b, L1, L2);
    double r[3] = {0.0, 0.0, 0.0};
    const double* bp = A.bpart + (size_t)b * A.G * 4;
    for (int g = 0; g < A.G; ++g)
        for (int i = 0; i < 3; ++i) r[i] += bp[4 * g + i];
    finalize<F>(A, b, L1, L2, r, bp[3]);
}

static __global__ void reset_kernel(int* __restrict__ status, int* __restrict__ redo,
                             uint64_t* __restrict__ fflag, uint64_t* __restrict__ bflag, int B,
                             int flags) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < B) status[i] = redo[i] = 0;
    if (i < flags) {
        store_flag(fflag + i, 0);
        store_flag(bflag + i, 0);
    }
}

// ------------------------------------------------------------------ launches

// Parts of an element.  Parts of four stripes (a wave per SIMD) where the whole grid is
// resident at once; else up to eight stripes in one workgroup, or parts of six and two
// copying waves if those are resident.  SPW = 0: none of these; parts that run one after
// another lose to the log-domain sweeps' resident parts of eight (SW [128, 1024, 512],
// forward and backward: 806 against 621 us).  D2P_AMD_SPLIT=<n> asks for n parts.
// Affine gaps: the reverse sweep keeps three states of a chunk and needs more registers
// than two waves on a SIMD leave each other (the spilling form took 700 us at [32, 500,
// 450], against 524 for the log-domain sweep), so a workgroup has four waves: an element
// of up to four stripes, or parts of two and the copying waves, where all of them are
// resident at once.
template <Fam F>
inline Split choose_parts(int B, int ns) {
    Split sp{1, ns > 0 ? ns : 1};
    int G = 0;
    if (const char* e = getenv("D2P_AMD_SPLIT")) G = atoi(e);
    if constexpr (Traits<F>::AFFINE) {
        G = G < ns ? G : ns;
        if (G <= 1 && ns <= 4) return sp;
        G = G > (ns + 1) / 2 ? G : (ns + 1) / 2;
        sp.SPW = (ns + G - 1) / G;
        sp.G = (ns + sp.SPW - 1) / sp.SPW;
        if (split_grid(B, sp.G) > device_cus()) sp.SPW = 0;
        return sp;
    }
    if (G <= 0) {
        const int g4 = (ns + 3) / 4;
        G = ns > 4 && split_grid(B, g4) <= device_cus() ? g4 : 1;
    }
    G = G < ns ? G : ns;
    if (G <= 1 && ns <= MAXW) return sp;
    const int g6 = (ns + MAXS_SPLIT - 1) / MAXS_SPLIT;
    G = G > g6 ? G : g6;
    sp.SPW = (ns + G - 1) / G;
    sp.G = (ns + sp.SPW - 1) / sp.SPW;
    if (split_grid(B, sp.G) > device_cus()) sp.SPW = 0;
    return sp;
}

inline Consts consts(double T, double gap_or_open, double ext) {
    Consts k;
    const double c = 1.4426950408889634074 / T;
    k.c = (float)c;
    k.gc = k.oc = gap_or_open * c;
    k.ec = ext * c;
    k.g = k.o = exp2(k.gc);
    k.e = exp2(k.ec);
    return k;
}

// Whether the sweeps take a call.
//  * Gaps small enough that a value lost below a neighbour's range weighs nothing, and
//    a temperature at which scores of usual size stay in range.
//  * Elements of at most kMaxLength (rows and columns together, at a temperature of 1 or
//    more).  The results are some 200 times nearer to the exact ones than 32-bit
//    log-domain sweeps are; but this library promises its marginals within 1e-4 of the
//    reference's, whose own 32-bit rounding (alpha on a grid of ulp(alpha), over T) reaches
//    1e-4 of the exact marginals at 1024 x 1024 and T = 1, 3e-4 at 2048 x 2048, and grows
//    with 1/T.  Longer elements keep the log-domain sweeps, which round as it does.
constexpr double kMinTemperature = 0.2, kMaxLength = 2048.0;
inline bool takes(int L1, int L2, double T, double g0, double g1) {
    const double c = 1.4426950408889634074 / T;
    return T >= kMinTemperature && fabs(g0 * c) <= kMaxGapBits && fabs(g1 * c) <= kMaxGapBits &&
           (double)L1 + (double)L2 <= kMaxLength * (T < 1.0 ? T : 1.0);
}

template <Fam F>
int run(Args& A, void* table, size_t table_bytes, bool* done, hipStream_t st, const char* fname,
        const char* bname) {
    using Tr = Traits<F>;
    *done = false;
    const int ns = (A.L1max + 63) / 64;
    const Split sp = choose_parts<F>(A.B, ns);
    A.NSmax = ns;
    A.G = sp.G;
    A.SPW = sp.SPW;
    A.mem = carve<F>(table, A.B, A.L1max, A.L2max, sp.G);
    if (ns == 0 || A.L2max == 0 || sp.SPW == 0 || A.mem.bytes > table_bytes) return D2P_OK;
    A.epoch = next_epoch();
    const int copying = sp.G > 1 ? 2 : 0;
    if (sp.G > 1)
        // (every word: the sweeps that redo an element may have other parts)
        D2P_LAUNCH("split_reset", reset_kernel, dim3((A.B * ns + 255) / 256), dim3(256), 0, st,
                   A.status, A.redo, A.fflag, A.bflag, A.B, A.B * ns);
    const dim3 grid(split_grid(A.B, sp.G));
    void (*fwd)(const Args) = nullptr;
    void (*bwd)(const Args) = bwd_kernel<F>;
    void (*both)(const Args) = nullptr;
    int fw = sp.SPW, bw = sp.SPW;
    size_t fl = (sp.SPW + 1) * sizeof(Ring<Tr::NP>) + (size_t)sp.SPW * NT * 64 * P * 4;
    size_t bl = (sp.SPW + 1) * sizeof(Ring<Tr::NQ>) +
                (size_t)sp.SPW * (64 * P * 4 + sizeof(OutTile)) + (size_t)sp.SPW * Tr::NP * P * 8;
    if constexpr (Tr::AFFINE) {
        fwd = fwd_kernel<F>;
    } else {
        // more waves a stripe: the forward always; the reverse sweep where every part has a
        // CU to itself and its stripes a SIMD each.  Two stripes a SIMD are bound by the
        // instructions they issue, of which the one-wave form has fewer (231 against 259 us
        // at [256, 512, 512])
        fwd = fwd2_kernel<F>;
        fw = 2 * sp.SPW;
        fl = (sp.SPW + 1) * sizeof(Ring<1>) + (size_t)sp.SPW * FWD2_FLOATS * 4;
        if (sp.SPW <= ROOMY && grid.x <= (unsigned)device_cus()) {
            bwd = bwd2_kernel<F>;
            if (sp.G == 1) both = both_kernel<F>;
            bw = 3 * sp.SPW;
            bl = (sp.SPW + 1) * sizeof(Ring<1>) + (size_t)sp.SPW * BWD2_FLOATS * 4;
        }
    }
    auto launch = [&](const char* name, void (*k)(const Args), int waves, size_t lds) {
        if (lds > 64 * 1024)
            D2P_HIP(hipFuncSetAttribute((const void*)k,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        D2P_LAUNCH(name, k, grid, dim3(waves * 64), lds, st, A);
        return (int)D2P_OK;
    };
    if (both != nullptr) {
        D2P_TRY(launch(bname, both, bw, fl > bl ? fl : bl));
    } else {
        D2P_TRY(launch(fname, fwd, fw + copying, fl));
        D2P_TRY(launch(bname, bwd, bw + copying, bl));
    }
    D2P_HIP(hipGetLastError());
    *done = true;
    return D2P_OK;
}

}  // namespace sc
}  // namespace d2p_amd
