// Internal interface and device code of the apply kernels (shared by
// apply.hip and kpm.hip).
//
// Two row kernels, both one wavefront per block row at a time:
//
// * row_loop (fused steps with per-column dots, and batched steps of one
//   column): the 64 lanes are split
//   into Kp = min(64, pow2ceil(K)) vector columns x NG = 64/Kp lane groups; a
//   group holds rpp row slots x P block partitions (P > 1 when the block row
//   has fewer scalar rows than groups, merged at the end with xor shuffles),
//   and each lane keeps RB row accumulators (register blocking) so that one X
//   element feeds up to RB rows.  The row's block metadata comes from ONE
//   lane-parallel load of 64 slots (meta: x offset, width, panel column), so
//   the inner loop issues only the value and X loads -- no dependent index
//   chains.  Accumulation is in FP64 registers for every storage precision.
//
// * row_loop_spmv (K == 1, blocks up to 8 x 8): lanes are (row a, partition
//   p); the values of each run of 64/RPP consecutive blocks (contiguous in
//   memory) are first streamed into a wave-private LDS tile with 16-byte
//   coalesced loads, each lane loads one x entry of the run into the tile's x
//   strip, then every lane forms its block-row dot product from LDS.  The next
//   run's loads are issued before the current run is computed.
//
// The other products run in quads.hpp (uniform 4 x 4 blocks) and tiles.hpp,
// the batched steps in lanes.hpp.
#pragma once

#include <initializer_list>
#include <type_traits>
#include <utility>

#include "common.hpp"

namespace vbh {

// T: vector (and accumulation input) type; V: matrix value type, T or its
// FP32 partner (precision 2: FP32 values against FP64 vectors).
template <typename T, typename V = T>
struct ApplyArgs {
    DevPattern p;
    const V* vals;
    int K;
    const T* X;
    int64_t ldx;
    T* Y;
    int64_t ldy;
    // fused epilogue: Y = alpha*AX + beta*X_own + gamma*Z; dots vs W (or Y) and X_own
    double alpha, beta, gamma;
    const T* Z;
    int64_t ldz;
    const T* W;
    int64_t ldw;
    double* partials;  // [G][2*max(dot_cols,1)] per-work-group FP64 partial dots, or null
    int dot_cols;      // K: one partial per column; 1 (or 0, no dots): summed over the columns
    int row_list;      // batched lane family: 1 = rows come from p.small_rows (the class rows run apart)
    int parts;         // lane family: partitions of each row's slots (1, 2, 4, 8)
    const int* split;  // G+1 row chunk boundaries
    int G;
};

// The adjoint plan of a matrix (see vbh_matrix): incoming blocks of every block
// column.
struct AdjointPlan {
    const int* t_ptr;
    const int64_t* t_voff;
    const int2* t_rows;
};

// What a lane loads in place of a block or of X rows that its row does not have:
// zeros on both sides of the product, since a zero matrix entry would still turn
// an infinity or NaN of X into NaN.  The choice is between numbers, and
// what comes out a global address: a choice of pointers becomes a flat load.
static __device__ const double kZeros[32] = {};
template <typename T>
__device__ __forceinline__ const T* or_zeros(bool there, const T* p) {
    using Global = const char __attribute__((address_space(1)))*;
    return (const T*)(Global)(there ? uint64_t(p) : uint64_t(kZeros));
}

// Register accumulator of a storage type: FP64 for every storage precision,
// so an FP32 recursion rounds once per step (at the store), not per term.
template <typename T>
struct Wide {
    using type = double;
};
template <>
struct Wide<c64> {
    using type = c128;
};
template <>
struct Wide<c128> {
    using type = c128;
};
__device__ inline double widen(double x) { return x; }
__device__ inline double widen(float x) { return double(x); }
__device__ inline c128 widen(c128 x) { return x; }
__device__ inline c128 widen(c64 x) { return c128{double(x.re), double(x.im)}; }
template <typename T>
__device__ inline T narrow_to(typename Wide<T>::type x) {
    if constexpr (std::is_same_v<T, float>) return float(x);
    else if constexpr (std::is_same_v<T, c64>) return c64{float(x.re), float(x.im)};
    else return x;
}

__device__ inline int lane_read(int v, int lane_idx) { return __builtin_amdgcn_readlane(v, lane_idx); }
// A 64-bit value the wave holds in every lane, as a scalar.
__device__ inline int64_t uniform64(int64_t v) {
    const uint64_t u = uint64_t(v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(u)), hi = __builtin_amdgcn_readfirstlane(uint32_t(u >> 32));
    return int64_t((uint64_t(hi) << 32) | lo);
}

// Series accumulation for Chebyshev sums sum_n c_n t_n built term by term:
// acc[row * ld + column] += (re + i im) * y for every stored (rounded) y of a
// fused step.  A kernel parameter of its own, not an ApplyArgs field: a larger
// argument struct raises the register use of every row kernel.
template <typename T>
struct SeriesAcc {
    T* acc;
    int64_t ld;
    double re, im;
};

// Fused epilogue for one output element (row yr, column v); ACC: also the
// series accumulation sa, or with TERM its counterpart Y += (re + i im) sa.acc.
template <typename T, bool FUSED, bool ACC = false, bool TERM = false>
__device__ inline void emit(const ApplyArgs<T>& g, int64_t yr, int64_t xr, int v, typename Wide<T>::type acc,
                            double& d1, double& d2, const SeriesAcc<T>* sa = nullptr) {
    using A = typename Wide<T>::type;
    A y = acc;
    if constexpr (ACC && TERM) y = widen(narrow_to<T>(y));  // the product as a vector of its own type
    if constexpr (FUSED) {
        const A xo = widen(g.X[xr * g.ldx + v]);
        y = rscale(g.alpha, y);
        if (g.beta != 0.0) y = y + rscale(g.beta, xo);
        if (g.gamma != 0.0) y = y + rscale(g.gamma, widen(g.Z[yr * g.ldz + v]));
        if constexpr (ACC && TERM)
            y = Sc<A>::fma(Sc<A>::make(sa->re, sa->im), widen(sa->acc[yr * sa->ld + v]), y);
        // dots of the stored (rounded) value: the state the recursion carries on
        const A ys = widen(narrow_to<T>(y));
        d1 += redot(g.W ? widen(g.W[yr * g.ldw + v]) : ys, ys);
        d2 += redot(xo, ys);
    }
    g.Y[yr * g.ldy + v] = narrow_to<T>(y);
    if constexpr (ACC && !TERM) {
        T* ap = sa->acc + yr * sa->ld + v;
        const A c = Sc<A>::make(sa->re, sa->im);
        *ap = narrow_to<T>(Sc<A>::fma(c, widen(narrow_to<T>(y)), widen(*ap)));
    }
}

// SpMM row loop (see the file comment).  BS > 0: uniform BS x BS blocks.
template <typename T, int BS, int RB>
__device__ inline void row_loop(const ApplyArgs<T>& g, int r0, int r1, int lane, int wave, double& d1, double& d2) {
    using A = typename Wide<T>::type;
    const DevPattern& p = g.p;
    const int K = g.K;
    const int Kp = K >= 64 ? 64 : pow2ceil(K);
    const int lgK = __builtin_ctz(Kp);
    const int NG = 64 >> lgK;
    const int v_l = lane & (Kp - 1);
    const int g_l = lane >> lgK;
    for (int i = r0 + wave; i < r1; i += kWaves) {
        const int r = BS > 0 ? BS : p.rbs[i];
        const int kb = p.row_ptr[i], ke = p.row_ptr[i + 1];
        const int rp = pow2ceil(r);
        const int rpp = rp < NG ? rp : NG;
        const int P = NG / rpp;
        const int a_l = g_l & (rpp - 1);
        const int p_l = g_l >> __builtin_ctz(rpp);
        const int64_t y0 = BS > 0 ? int64_t(i) * BS : p.roff[i];
        const int64_t x0 = BS > 0 ? int64_t(i) * BS : p.coff[i];
        const int64_t vrow = BS > 0 ? int64_t(kb) * (BS * BS) : p.voff[kb];
        for (int a0 = 0; a0 < r; a0 += rpp * RB) {
            for (int v0 = 0; v0 < K; v0 += Kp) {
                const int v = v0 + v_l;
                const bool vok = v < K;
                A acc[RB];
#pragma unroll
                for (int q = 0; q < RB; ++q) acc[q] = Sc<A>::zero();
                for (int t0 = kb; t0 < ke; t0 += 64) {
                    const int nb = ke - t0 < 64 ? ke - t0 : 64;
                    int mx = 0, mw = 0;
                    if (lane < nb) {
                        if constexpr (BS > 0) {
                            mx = p.col_ind[t0 + lane] * BS;
                            mw = ((t0 + lane - kb) * BS) << 8 | BS;
                        } else {
                            const int2 mm = p.meta[t0 + lane];
                            mx = mm.x;
                            mw = mm.y;
                        }
                    }
#pragma unroll 2
                    for (int ub = 0; ub < nb; ub += P) {
                        const int u = ub + p_l;
                        int xo, w;
                        if (P == 1) {
                            xo = lane_read(mx, ub);
                            w = lane_read(mw, ub);
                        } else {
                            xo = __shfl(mx, u, 64);
                            w = __shfl(mw, u, 64);
                        }
                        if (!vok || u >= nb) continue;
                        const int c = BS > 0 ? BS : (w & 255);
                        const T* ab = g.vals + vrow + int64_t(r) * (w >> 8);
                        const T* xb = g.X + int64_t(xo) * g.ldx + v;
                        if constexpr (BS > 0) {
                            T xv[BS];
#pragma unroll
                            for (int b = 0; b < BS; ++b) xv[b] = xb[int64_t(b) * g.ldx];
#pragma unroll
                            for (int q = 0; q < RB; ++q) {
                                const int a = a0 + a_l + q * rpp;
                                if (a < r) {
                                    T av[BS];
                                    const T* ar = ab + a * BS;
                                    if constexpr ((BS * sizeof(T)) % 16 == 0) {
                                        const T* al = static_cast<const T*>(__builtin_assume_aligned(ar, 16));
#pragma unroll
                                        for (int b = 0; b < BS; ++b) av[b] = al[b];
                                    } else {
#pragma unroll
                                        for (int b = 0; b < BS; ++b) av[b] = ar[b];
                                    }
#pragma unroll
                                    for (int b = 0; b < BS; ++b) acc[q] = Sc<A>::fma(widen(av[b]), widen(xv[b]), acc[q]);
                                }
                            }
                        } else {
                            for (int b = 0; b < c; ++b) {
                                const A xv = widen(xb[int64_t(b) * g.ldx]);
#pragma unroll
                                for (int q = 0; q < RB; ++q) {
                                    const int a = a0 + a_l + q * rpp;
                                    if (a < r) acc[q] = Sc<A>::fma(widen(ab[a * c + b]), xv, acc[q]);
                                }
                            }
                        }
                    }
                }
#pragma unroll
                for (int q = 0; q < RB; ++q)
                    for (int s = Kp * rpp; s < 64; s <<= 1) acc[q] = acc[q] + shfl_xor(acc[q], s);
                if (vok && p_l == 0) {
#pragma unroll
                    for (int q = 0; q < RB; ++q) {
                        const int a = a0 + a_l + q * rpp;
                        if (a < r) emit<T, true>(g, y0 + a, x0 + a, v, acc[q], d1, d2);
                    }
                }
            }
        }
    }
}

// LDS tile of the SpMV per wave: a run's values (at most 64*rpp plus two
// partial 16-byte words), then the run's 64 x entries (kSpmvX onwards), then
// a zero element (kSpmvZero) that the columns past a block's width read.
constexpr int kSpmvTile(int rpp) { return 64 * rpp + 16 + 64 + 2; }
constexpr int kSpmvX(int rpp) { return 64 * rpp + 16; }
constexpr int kSpmvZero(int rpp) { return 64 * rpp + 16 + 64; }

// 16-byte vector of a storage type, for the coalesced LDS staging copies.
template <typename T>
struct Vec16 {
    static constexpr int n = 16 / sizeof(T);
    T v[16 / sizeof(T)];
};

// 16 raw bytes as a native vector type: staging words kept in registers
// across loop iterations stay registers (arrays of structs would not).
typedef int vbh_w4 __attribute__((ext_vector_type(4)));

// Words of one staged run of the LDS SpMV per lane.
template <typename T, int RPP>
constexpr int spmv_words() {
    return (kSpmvX(RPP) / Vec16<T>::n + 63) / 64;
}

// Issues the loads of one staged run into registers: its 16-byte value words
// and one x entry per lane -- entry b of the run's block j/RPP for lane j, so
// the run's x segments are read once, not once per row -- with clamped
// (unconditional, in-bounds) indices: a guarded load compiles to a branch with
// its own wait.
template <typename T, int RPP>
__device__ __forceinline__ void spmv_issue(const ApplyArgs<T>& g, int64_t vrow, int r, int nb, int ub, int mx, int mw,
                                           int lane, vbh_w4 (&stage)[spmv_words<T, RPP>()], T& xone, int& lead,
                                           int& nvec, int& pc_first, int& w, bool& act) {
    constexpr int CH = 64 / RPP;
    constexpr int EV = Vec16<T>::n;
    const int a_l = lane & (RPP - 1);
    const int p_l = lane / RPP;
    const int ulast = (ub + CH < nb ? ub + CH : nb) - 1;
    pc_first = lane_read(mw, ub) >> 8;
    const int wl = lane_read(mw, ulast);
    const int pc_end = (wl >> 8) + (wl & 255);
    const int64_t s0 = vrow + int64_t(r) * pc_first;  // first value of the run
    const int64_t sa = s0 & ~int64_t(EV - 1);         // 16-byte aligned start
    lead = int(s0 - sa);
    nvec = (lead + r * (pc_end - pc_first) + EV - 1) / EV;
    const vbh_w4* src = reinterpret_cast<const vbh_w4*>(g.vals + sa);
    const int u = ub + p_l;
    const int xo = __shfl(mx, u, 64);  // lanes past the row's slots hold x offset 0, width 0
    w = __shfl(mw, u, 64);
    act = u <= ulast && a_l < r;
#pragma unroll
    for (int q = 0; q < spmv_words<T, RPP>(); ++q) {
        // words past the run are skipped on a wave-uniform condition (a scalar
        // branch: no per-lane wait); inside the run the index is clamped
        if (q == 0 || q * 64 < nvec) {
            const int e = q * 64 + lane;
            // non-temporal: the value stream is read once, and evict-first
            // lines leave the L2 to the x entries, which are gathered again
            stage[q] = __builtin_nontemporal_load(src + (e < nvec ? e : nvec - 1));
        }
    }
    // lane = p*RPP + b loads x[xo_p + b] (clamped into the block's width;
    // complex types: zero past it)
    const int c = w & 255;
    const int cm = c > 0 ? c - 1 : 0;
    xone = g.X[int64_t(xo + (a_l < cm ? a_l : cm)) * g.ldx];
    if constexpr (Sc<T>::is_complex) xone = pick(a_l < c, xone, Sc<T>::zero());
}

// SpMV row loop for blocks up to RPP x RPP (RPP in {1, 2, 4, 8}); lds is this
// wave's 16-byte aligned tile of kSpmvTile(RPP) elements: a run of 64/RPP
// blocks holds at most 64*RPP values, plus up to two partial 16-byte words.
// Software-pipelined within each 64-slot chunk of a row: run n+1's loads are
// in flight while run n is computed from the tile.
template <typename T, int RPP, bool FUSED, bool ACC = false>
__device__ inline void row_loop_spmv(const ApplyArgs<T>& g, int r0, int r1, int lane, int wave, double& d1,
                                     double& d2, T* lds, const SeriesAcc<T>* sa = nullptr) {
    using A = typename Wide<T>::type;
    constexpr int CH = 64 / RPP;  // blocks per staged run = partitions
    const DevPattern& p = g.p;
    const int a_l = lane & (RPP - 1);
    if (lane == 0) lds[kSpmvZero(RPP)] = Sc<T>::zero();  // visible after the first run's wave barrier
    for (int i = r0 + wave; i < r1; i += kWaves) {
        const int r = p.rbs[i];
        const int kb = p.row_ptr[i], ke = p.row_ptr[i + 1];
        const int64_t vrow = p.voff[kb];
        A acc = Sc<A>::zero();
        for (int t0 = kb; t0 < ke; t0 += 64) {
            const int nb = ke - t0 < 64 ? ke - t0 : 64;
            int mx = 0, mw = 0;
            {
                const int2 mm = p.meta[t0 + (lane < nb ? lane : nb - 1)];
                mx = lane < nb ? mm.x : 0;
                mw = lane < nb ? mm.y : 0;
            }
            constexpr int NV = spmv_words<T, RPP>();
            vbh_w4 stage[NV];
            T xone;
            int lead = 0, nvec = 1, pc_first = 0, w = 0;
            bool act = false;
            spmv_issue<T, RPP>(g, vrow, r, nb, 0, mx, mw, lane, stage, xone, lead, nvec, pc_first, w, act);
            for (int ub = 0; ub < nb; ub += CH) {
                // this run's words to the tile (lanes past the run rewrite word
                // nvec-1 with the value it already holds), its x to xc
                {
                    vbh_w4* dstw = reinterpret_cast<vbh_w4*>(lds);
#pragma unroll
                    for (int q = 0; q < NV; ++q) {
                        if (q == 0 || q * 64 < nvec) {
                            const int e = q * 64 + lane;
                            dstw[e < nvec ? e : nvec - 1] = stage[q];
                        }
                    }
                }
                lds[kSpmvX(RPP) + lane] = xone;
                const int lead_c = lead, pc_first_c = pc_first, w_c = w;
                const bool act_c = act;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#ifndef VBH_SPMV_NOPIPE
                if (ub + CH < nb)  // overlaps the FMAs below
                    spmv_issue<T, RPP>(g, vrow, r, nb, ub + CH, mx, mw, lane, stage, xone, lead, nvec, pc_first, w,
                                       act);
#endif
                if (act_c) {
                    const int c = w_c & 255;
                    const T* ab = lds + lead_c + r * ((w_c >> 8) - pc_first_c) + a_l * c;
                    const T* xs = lds + kSpmvX(RPP) + (lane & ~(RPP - 1));  // this block's x entries
                    if constexpr (Sc<T>::is_complex) {
                        // columns b >= c of a narrower block multiply the zero
                        // element by a zero x entry: exact, without a select
                        // on the four words of the accumulator (propagation
                        // forward 68.9 -> 59.3 ms; for real types the select
                        // measured faster: 0.36 against 0.378 ms on the
                        // 1.54 GB SpMV)
                        const T* zp = lds + kSpmvZero(RPP);
#pragma unroll
                        for (int b = 0; b < RPP; ++b)
                            acc = Sc<A>::fma(widen(*(b < c ? ab + b : zp)), widen(xs[b]), acc);
                    } else {
                        const int cm = c > 0 ? c - 1 : 0;
#pragma unroll
                        for (int b = 0; b < RPP; ++b) {
                            const A t = Sc<A>::fma(widen(ab[b < cm ? b : cm]), widen(xs[b]), acc);
                            acc = pick(b < c, t, acc);
                        }
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#ifdef VBH_SPMV_NOPIPE
                if (ub + CH < nb)
                    spmv_issue<T, RPP>(g, vrow, r, nb, ub + CH, mx, mw, lane, stage, xone, lead, nvec, pc_first, w,
                                       act);
#endif
            }
        }
#pragma unroll
        for (int s = RPP; s < 64; s <<= 1) acc = acc + shfl_xor(acc, s);
        if (lane < r)
            emit<T, FUSED, ACC>(g, int64_t(p.roff[i]) + lane, int64_t(p.coff[i]) + lane, 0, acc, d1, d2, sa);
    }
}

// Per-column sums of the lane partials d1, d2 of a whole work-group, written
// to out[0..K) and out[K..2K) by wave 0 (K <= 64).  Every thread must call it.
__device__ inline void write_partials(int K, int lane, int wave, double d1, double d2, double* out) {
    __shared__ double red[kWaves][2][64];
    const int Kp = K >= 64 ? 64 : pow2ceil(K);
    for (int s = Kp; s < 64; s <<= 1) {
        d1 += __shfl_xor(d1, s, 64);
        d2 += __shfl_xor(d2, s, 64);
    }
    red[wave][0][lane] = d1;
    red[wave][1][lane] = d2;
    __syncthreads();
    if (wave == 0 && lane < K) {
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            s1 += red[w][0][lane];
            s2 += red[w][1][lane];
        }
        out[lane] = s1;
        out[K + lane] = s2;
    }
}

// The same for column-summed dots: out[0], out[1].  The first exchange of the wave
// halves folds the two sums into one register (d1 in lanes 0 .. 31, d2 in 32 .. 63),
// the rest stays in the vector ALUs.  Six stages of two 64-bit shuffles each through
// the LDS crossbar before: 64 moments on 288 block rows of 4 x 4 217 us, now 194;
// 200 on graphene 200 x 200, 10 FP32 columns, 2311 and 2218.
__device__ __forceinline__ void write_dots(int lane, int wave, double d1, double d2, double* out) {
    __shared__ double red[kWaves][2];
    auto halves = [](double x, double y, auto swap) {
        const uint64_t u = uint64_t(__double_as_longlong(x)), w = uint64_t(__double_as_longlong(y));
        const auto lo = swap(uint32_t(u), uint32_t(w)), hi = swap(uint32_t(u >> 32), uint32_t(w >> 32));
        return __longlong_as_double(int64_t(uint64_t(hi[0]) << 32 | lo[0])) +
               __longlong_as_double(int64_t(uint64_t(hi[1]) << 32 | lo[1]));
    };
    auto dpp = [](double x, auto ctrl) {
        const uint64_t u = uint64_t(__double_as_longlong(x));
        const uint32_t lo = __builtin_amdgcn_mov_dpp(int(u), decltype(ctrl)::value, 0xf, 0xf, false);
        const uint32_t hi = __builtin_amdgcn_mov_dpp(int(u >> 32), decltype(ctrl)::value, 0xf, 0xf, false);
        return __longlong_as_double(int64_t(uint64_t(hi) << 32 | lo));
    };
    double d = halves(d1, d2, [](uint32_t x, uint32_t y) { return __builtin_amdgcn_permlane32_swap(x, y, false, false); });
    d = halves(d, d, [](uint32_t x, uint32_t y) { return __builtin_amdgcn_permlane16_swap(x, y, false, false); });
    d += dpp(d, std::integral_constant<int, 0x128>{});  // row_ror:8
    d += dpp(d, std::integral_constant<int, 0x124>{});  // row_ror:4, the sums repeat every 8 lanes
    d += dpp(d, std::integral_constant<int, 0x4e>{});   // quad_perm [2, 3, 0, 1]
    d += dpp(d, std::integral_constant<int, 0xb1>{});   // quad_perm [1, 0, 3, 2]
    if ((lane & 31) == 0) red[wave][lane >> 5] = d;
    __syncthreads();
    if (wave == 0 && lane < 2) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) s += red[w][lane];
        out[lane] = s;
    }
}

// Row-loop configuration chosen per launch: which kernel family and its
// compile-time parameters.
struct RowConfig {
    int spmv_rpp;  // > 0: LDS SpMV family with RPP = this
    int bs;        // SpMM family: uniform block size (4) or 0
    int rb;        // SpMM family: row accumulators per lane (1, 2, 4, 8)
};
RowConfig row_config(int K, int max_block, int uniform_bs);

// Lane-per-row family (lanes.hpp): S lanes per scalar row, KT columns each.
struct LaneShape {
    int S, KT;   // S == 0: family not applicable
    int P = 1;   // partitions of each row's slots (lane_parts)
    int rw = 0;  // > 0: the row-wave kernel instead, rw scalar rows per work-group
    int brw = 0;  // 1: the matrix-core class rows on the block-row wave kernel (vector ALUs)
    int rows = 0;  // batched steps: kRows*, every row on that kernel, 0: the families above
};
// Batched steps on the kernels of single matrices: tiles.hpp, quads.hpp or
// smalls.hpp (block size kRowsSmall - 1 + size).
constexpr int kRowsTiles = 1, kRowsQuads = 2, kRowsSmall = 3;
// Columns per lane of the row-wave kernel (16 bytes of a row), or 0 when it
// does not serve (T, K): real types, K a multiple of it with K / it a power
// of two up to 64.
template <typename T>
inline int rowwave_cpl(int K) {
    if constexpr (Sc<T>::is_complex) {
        return 0;
    } else {
        const int cpl = int(16 / sizeof(T));
        if (K < cpl || K % cpl) return 0;
        const int lq = K / cpl;
        return (lq & (lq - 1)) == 0 && lq <= 64 ? cpl : 0;
    }
}
// Columns per lane of the block-row wave kernel (K = 16 * it: 1, 2 or 4), or
// 0 when it does not serve (T, K): real types only.
template <typename T>
inline int brw_cpl(int K) {
    if constexpr (Sc<T>::is_complex) {
        return 0;
    } else {
        return (K == 16 || K == 32 || K == 64) ? K / 16 : 0;
    }
}
// Instantiated shapes: real K <= 16 one lane per row (KT in 4, 8, 10, 12, 16),
// up to 64 with 2 or 4 lanes of 16 columns; complex KT = 8 with 1..8 lanes.
// K == 1 runs here only for mixed value/vector types (the SpMV families are
// single-type).
inline LaneShape lane_shape(bool complex, int K, bool mixed = false) {
    if (K == 1 && mixed) K = 2;
    if (K < 2 || K > 64) return {0, 0};
    if (complex) {
        if (K <= 4) return {1, 4};
        if (K <= 8) return {1, 8};
        return {K <= 16 ? 2 : K <= 32 ? 4 : 8, 8};
    }
    if (K <= 16) return {1, K <= 4 ? 4 : K <= 8 ? 8 : K <= 10 ? 10 : K <= 12 ? 12 : 16};
    return {K <= 32 ? 2 : 4, 16};
}
// Scalar rows handled by one work-group of the lane family.
inline int lane_rows_per_group(int S, int P = 1) { return kWaves * (64 / (S * P)); }
// Partitions of each row's slots: small launches split rows over more lanes,
// so every lane's dependent chain of block loads gets shorter and the chip
// fills.  Target: 4 waves on each of 1024 SIMDs for 4-byte vectors, 8 for
// wider ones (measured on the 200x200 graphene KPM step: FP32 is fastest at
// P = 1, FP64 at P = 2).
inline int lane_parts(int64_t rows, int S, int elem_bytes) {
    const int64_t target = int64_t(256) * 4 * (elem_bytes <= 4 ? 4 : 8) * 64;
    const int pmax = 64 / S < 8 ? 64 / S : 8;
    int P = 1;
#ifdef VBH_FORCE_PARTS
    while (P * 2 <= pmax && P < VBH_FORCE_PARTS) P *= 2;
    return P;
#endif
    while (P * 2 <= pmax && rows * S * P < target) P *= 2;
    return P;
}
// Widest vector (elements of T, at most 16 bytes, dividing KT and K, so no
// vector straddles column K) that every operand (base pointer, leading
// dimension) admits; null operands are skipped.
template <typename T>
int lane_vector(int KT, int K, std::initializer_list<std::pair<const void*, int64_t>> operands) {
    int vn = sizeof(T) >= 16 ? 1 : int(16 / sizeof(T));
    for (; vn > 1; vn >>= 1) {
        bool ok = KT % vn == 0 && K % vn == 0;
        for (const auto& o : operands)
            if (o.first && (reinterpret_cast<uintptr_t>(o.first) % (vn * sizeof(T)) != 0 || o.second % vn != 0))
                ok = false;
        if (ok) break;
    }
    return vn;
}

template <typename T, typename V>
constexpr bool is_mixed() {
    return !std::is_same_v<T, V>;
}
template <typename T, typename V>
inline LaneShape lane_shape_of(int K) {
    return lane_shape(Sc<T>::is_complex, K, is_mixed<T, V>());
}
// Uniform 4x4 blocks (quads.hpp): S waves per four block rows, each with NG
// columns per lane (4 NG per wave).
template <typename T>
constexpr int kQuadMaxGroups = sizeof(T) >= 16 ? 2 : 4;
struct QuadShape {
    int S, NG;
};
template <typename T>
inline QuadShape quad_shape(int K) {
    const int S = (K + 4 * kQuadMaxGroups<T> - 1) / (4 * kQuadMaxGroups<T>);
    return {S, (K + 4 * S - 1) / (4 * S)};
}
template <typename T, typename V>
inline bool uses_quads(const vbh_matrix* m, const ApplyArgs<T, V>& a) {
    return m->uniform_bs == 4 && a.dot_cols <= 1 && (is_mixed<T, V>() ? a.K <= 64 : a.K > 1);
}
// Few waves with long sums: where a launch of uniform 4x4 blocks has fewer units
// than the chip has SIMDs and rows of more than one pass of 16 slots, a whole work-
// group takes a unit and its waves share the row's slots.  us without / with, 16 FP64
// columns: 128 block rows of 128 blocks 12.3 / 5.1 (a lane per scalar row, its slots
// in parts, took 10.6), 1000 of 1000 blocks every 97th row 73 / 25 (40); one column,
// complex, 128 rows of 128 17.0 / 10.8.  From 1024 units on it loses 10 %.
constexpr int kSplitUnits = 1024;
// What the rules below ask of a matrix, or of a batch.
struct RowStats {
    int64_t out_rows = 0, nnz = 0, n_rows = 0;  // block rows (adjoint: columns), values, scalar rows
    int max_block = 0, longest_row = 0;
    RowStats() = default;
    RowStats(const vbh_matrix* m, int64_t out)
        : out_rows(out), nnz(m->nnz), n_rows(m->n_rows), max_block(m->max_block), longest_row(m->longest_row) {}
    void add(const vbh_matrix* m) {
        out_rows += m->nbr;
        nnz += m->nnz;
        n_rows += m->n_rows;
        max_block = std::max(max_block, m->max_block);
        longest_row = std::max(longest_row, m->longest_row);
    }
};
inline int padded_groups(int64_t g) { return int(((g < 8 ? 8 : g) + 7) & ~int64_t(7)); }
struct QuadGrid {
    int S, NG;
    bool split;
    int G;
};
template <typename T>
inline QuadGrid quad_grid(const RowStats& r, int K) {
    const QuadShape q = quad_shape<T>(K);
    const int64_t units = (r.out_rows + 3) / 4 * q.S;
    const bool split = units < kSplitUnits && r.longest_row > 16;
    return {q.S, q.NG, split, padded_groups(split ? units : (units + kWaves - 1) / kWaves)};
}
// One column of uniform 4x4 blocks (quad_spmv.hpp): a wave per four block rows.
template <typename T, typename V>
inline bool uses_quad_spmv(const vbh_matrix* m, const ApplyArgs<T, V>& a) {
    return !is_mixed<T, V>() && m->uniform_bs == 4 && a.K == 1 && a.dot_cols <= 1;
}
struct QuadSpmvGrid {
    bool split;
    int G;
};
inline QuadSpmvGrid quad_spmv_grid(const vbh_matrix* m, int out_rows) {
    const int units = (out_rows + 3) / 4;
    const bool split = units < kSplitUnits && m->longest_row > 16;
    return {split, padded_groups(split ? units : (units + kWaves - 1) / kWaves)};
}
// One column of uniform blocks up to 3: from this many block rows on smalls.hpp
// is used; below, where a launch is bounded by its chain of loads, the LDS
// SpMV's chain is the shorter one (FP64 series step, size 2, us with the LDS SpMV
// / smalls.hpp: 288 block rows 4.1 / 5.1, 1,472 4.6 / 5.3, 16,200 10.2 / 5.2).
constexpr int kManyRows = 8192;
// Uniform blocks of size 1 to 3 (smalls.hpp): lanes of NC columns, L of them per
// block row, S column slices, the slots of a row over P partitions of the wave.
struct SmallShape {
    int NC, L, S, P, rows, G;  // rows: block rows per wave; G: work-groups
};
template <typename T>
inline SmallShape small_shape(int64_t nnzb, int64_t out_rows, int K) {
    SmallShape sh{};
    sh.NC = K >= 4 && 4 * sizeof(T) <= 16 ? 4 : K >= 2 && 2 * sizeof(T) <= 16 ? 2 : 1;
    const int lanes = (K + sh.NC - 1) / sh.NC;
    sh.S = (lanes + 15) / 16;
    sh.L = (lanes + sh.S - 1) / sh.S;
    int64_t units = 0;
    // two waves per SIMD; a partition keeps at least three slots (graphene 65 x
    // 71, size 2, 2 FP64 columns, 64 moments: 246 us, without partitions 316;
    // twice the waves cost 150 x 150 up to 27 %), and there are as many as the lanes
    // allow (128 block rows of 128 blocks of size 2, one complex column, adjoint, up to
    // 16 / 64 partitions: 6.5 / 4.6 us)
    for (sh.P = 1;; sh.P *= 2) {
        sh.rows = 64 / sh.P / sh.L;
        units = (out_rows + sh.rows - 1) / sh.rows * sh.S;
        if (units >= 2048 || sh.P * 2 * sh.L > 64 || nnzb < 3 * sh.P * out_rows) break;
    }
    const int64_t g = (units + kWaves - 1) / kWaves;
    sh.G = int(((g < 8 ? 8 : g) + 7) & ~int64_t(7));
    return sh;
}
// Size 3 only with short rows: from about 16 blocks a row the variable-block
// kernel's shared loads win (20,000 rows of 61 blocks, 4 FP64 columns: 26.6 us
// here, 19.1 there; 13,824 rows of 7: 9.0 here, 10.8 there).
inline bool small_blocks(const vbh_matrix* m) {
    return m->uniform_bs >= 1 && (m->uniform_bs <= 2 || (m->uniform_bs == 3 && m->nnzb <= int64_t(16) * m->nbr));
}
template <typename T, typename V>
inline bool uses_smalls(const vbh_matrix* m, const ApplyArgs<T, V>& a) {
    if (is_mixed<T, V>() && a.K > 64) return false;
    return small_blocks(m) && a.dot_cols <= 1 && (a.K > 1 || is_mixed<T, V>() || m->nbr >= kManyRows);
}
// Column slices of a K-column product on variable blocks: S waves per output
// block row, 4 NG columns each; up to 24 columns in one slice, beyond that
// slices of 16 (more columns a wave read A less often but hold its X operands,
// 4 NG sizeof(T) bytes a lane, in registers: 64 FP64 columns on blocks of 4-8,
// slices of 16 / 32: 53 / 65 us, on blocks of 1, 4, 9, 13: 83 / 85 us).
struct TileShape {
    int S, NG;
};
inline TileShape tile_shape(bool complex, int K) {
    if (!complex && K > 16 && K <= 24) return {1, 6};
    const int S = (K + 15) / 16;
    return {S, (K + 4 * S - 1) / (4 * S)};
}

// Units of a product on variable blocks: output block rows x slices x parts.  A
// part takes every parts-th 16 rows of the blocks, so that few, wide block rows fill
// the chip: up to 8192 units, eight waves a SIMD.  A work-group shares a unit's
// blocks between its waves while there are few units with long sums (steps: the
// instructions of an average row).  us, one wave per block row and slice / now / a
// lane per scalar row before: 12 block rows of 6 blocks of 255, 2 FP64 columns 579 /
// 17 / 39, 16 columns 1007 / 27 / 105; 100 of 10 of 64, 16 columns 99 / 21 / 61; 32 of 32 of
// 16, 16 columns 20 / 7 / 19.  With fewer steps or more units sharing loses (1000 rows
// of 40 blocks of 3, 8 columns 6.2 / 7.6).
constexpr int kPartUnits = 8192, kShareUnits = 512;
struct TileGrid {
    int S, NG, parts;
    bool split;
    int G;
};
template <typename T>
inline TileGrid tile_grid(const RowStats& r, int K) {
    const TileShape q = tile_shape(Sc<T>::is_complex, K);
    int64_t units = r.out_rows * q.S;
    int parts = 1;
    if (r.max_block > 16 && units > 0)
        parts = int(std::max<int64_t>(1, std::min<int64_t>((r.max_block + 15) / 16, kPartUnits / units)));
    units *= parts;
    // 16, 8 or 4 chunks of four columns an instruction
    const int64_t chunks = r.max_block <= 4 ? 16 : r.max_block <= 8 ? 8 : 4;
    const int64_t steps = r.n_rows > 0 ? r.nnz / r.n_rows / (4 * chunks) : 0;
    const bool split = steps >= 2 && units < std::min<int64_t>(kShareUnits, 128 * steps);
    return {q.S, q.NG, parts, split, padded_groups(split ? units : (units + kWaves - 1) / kWaves)};
}
// One column of blocks up to 8 on the variable-block kernel: sizes that differ,
// rows of eight blocks or more, values that fit the 256 MB memory-side cache.  The
// LDS SpMV stages a row's blocks run by run and reaches more of the HBM rate; us
// there / here: 500 rows of 60 blocks of 4-8 10.1 / 6.2, 1728 of 27 9.4 / 6.9, 20,000
// of 40 (230 MB) 55 / 46, complex (460 MB) 98 / 106, FP64 of 724 MB 148 / 177; uniform
// 5, ten blocks a row, 16,200 rows of FP32 18.3 / 24.6; seven blocks a row 8.4 / 7.6.
template <typename V>
inline bool one_column_tiles(const vbh_matrix* m) {
    return m->uniform_bs == 0 && m->nnzb >= int64_t(8) * m->nbr &&
           m->nnz <= int64_t(size_t(256) << 20) / int64_t(sizeof(V));
}
// Whether the variable-block kernel (tiles.hpp) runs these arguments: every K
// except the single-type SpMV of blocks up to 8 outside that rule, column-summed
// dots.
template <typename T, typename V>
inline bool uses_tiles(const vbh_matrix* m, const ApplyArgs<T, V>& a) {
    if (is_mixed<T, V>() && a.K > 64) return false;
    return a.dot_cols <= 1 && !uses_quads(m, a) && !uses_smalls(m, a) && (a.K > 1 || is_mixed<T, V>() || m->max_block > 8 || one_column_tiles<V>(m));
}
// Batched steps: block rows of a class run one per wave (the FP64 matrix cores,
// or the block-row wave kernel), the other rows on the lane family.
constexpr int kMfmaRowsPerGroup = kWaves * kMfmaRowsPerWave;  // block rows per work-group
// Work-groups (= partial slots) a launch_rows call with these arguments uses.
template <typename T, typename V>
inline int apply_groups(const vbh_matrix* m, const ApplyArgs<T, V>& a) {
    if (uses_quads(m, a)) return quad_grid<T>(RowStats(m, m->nbr), a.K).G;
    if (uses_quad_spmv(m, a)) return quad_spmv_grid(m, m->nbr).G;
    if (uses_smalls(m, a)) return small_shape<T>(m->nnzb, m->nbr, a.K).G;
    if (uses_tiles(m, a)) return tile_grid<T>(RowStats(m, m->nbr), a.K).G;
    return m->G;
}

template <typename T, bool FUSED, typename V = T>
void launch_rows(const vbh_matrix* m, const ApplyArgs<T, V>& a, hipStream_t s);
// Uniform 4x4 blocks; sa: also the series accumulation (no dots).
template <typename T, typename V>
void launch_quads(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>* sa, hipStream_t s);
// One column of uniform 4x4 blocks, forward (sa as above) and adjoint (term as
// below).
template <typename T>
void launch_quad_spmv(const vbh_matrix* m, const ApplyArgs<T>& a, bool fused, const SeriesAcc<T>* sa, hipStream_t s);
template <typename T>
void launch_quad_spmv_adjoint(const vbh_matrix* m, const ApplyArgs<T>& a, const AdjointPlan& ap, const SeriesAcc<T>* term,
                              hipStream_t s);
// Uniform blocks of size 1 to 3, forward and adjoint (sa and term likewise).
template <typename T, typename V>
void launch_smalls(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>* sa, hipStream_t s);
template <typename T>
void launch_smalls_adjoint(const vbh_matrix* m, const ApplyArgs<T>& a, const AdjointPlan& ap, const SeriesAcc<T>* term,
                           hipStream_t s);
// Variable blocks; sa as above.
template <typename T, typename V>
void launch_tiles(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>* sa, hipStream_t s);
// Adjoint products Y = alpha A^H X + beta X + gamma Z (+ (re + i im) term->acc).
template <typename T>
void launch_tiles_adjoint(const vbh_matrix* m, const ApplyArgs<T, T>& a, const AdjointPlan& ap, const SeriesAcc<T>* term,
                          hipStream_t s);
// One matrix of a batched KPM launch.
template <typename T, typename V = T>
struct BatchItem {
    DevPattern p;
    const V* vals;
    T* buf[3];     // recursion vectors t_{n-1}, t_n, t_{n+1} rotate through these
    const T* v0;   // mode 1: the start vectors (W of the dot)
    const int* split;
    int64_t n_rows;
    int64_t lane_rows;  // rows of the lane launch: n_rows, or the small rows (row_list)
    int row_list;       // 1: the lane launch takes p.small_rows, the matrix-core launch p.big_brows
    int G;              // this matrix's lane (or row-loop) work-groups
    int g_base;         // its first work-group in the lane launch
    int g_base2;        // its first work-group in the matrix-core launch
    // block-row wave kernel (class rows on the vector ALUs): the column-major
    // FP32 values and the X row of every stored scalar column of each block
    // row (entries eoff[i] .. eoff[i+1])
    const float* vt;
    const int64_t* eoff;
    const int* ecol;
};
template <typename T, typename V>
void launch_batched_lanes(const BatchItem<T, V>* items, int nitems, int Gtot, int K, int ld, LaneShape sh, int step,
                          double alpha, double beta, double gamma0, double gamma, int mode, double* partials,
                          hipStream_t s);
template <typename T, typename V>
void launch_batched_rowwave(const BatchItem<T, V>* items, int nitems, int Gtot, int K, int ld, int rw, int step,
                            double alpha, double beta, double gamma0, double gamma, int mode, double* partials,
                            hipStream_t s);
template <typename T, typename V>
void launch_batched_brw(const BatchItem<T, V>* items, int nitems, int Gtot, int K, int ld, int step, double alpha,
                        double beta, double gamma0, double gamma, int mode, double* partials, hipStream_t s);
template <typename T, typename V>
void launch_batched_mfma(const BatchItem<T, V>* items, int nitems, int Gtot, int K, int ld, int step, double alpha,
                         double beta, double gamma0, double gamma, int mode, double* partials, hipStream_t s);
// Batched steps with every row on the kernel of single matrices: units of `per`
// block rows, `slices` and `parts` a unit's row, on a wave or (split) a work-group
// each; small: the shape of kRowsSmall.
struct RowsShape {
    int per = 1, slices = 1, parts = 1;
    bool split = false;
    SmallShape small{};
};
// A step with every row on the kernel `rows`.
template <typename T, typename V>
void launch_batched_rows(const BatchItem<T, V>* items, int nitems, int Gtot, int K, int ld, int rows,
                         const RowsShape& shape, int step, double alpha, double beta, double gamma0, double gamma,
                         int mode, double* partials, hipStream_t s);
template <typename T, typename V = T>
ApplyArgs<T, V> make_args(const vbh_matrix* m, const V* vals, int K, const T* X, int64_t ldx, T* Y, int64_t ldy);
template <typename T>
const T* compute_values(vbh_matrix* m, hipStream_t s);
// One fused step with the series accumulation sa in the same launch.  Returns
// false (nothing launched) where no kernel serves the arguments: with dots, which
// the caller launches and accumulates separately, and for more than 64 mixed
// columns, which launch_rows refuses.
template <typename T, typename V>
bool launch_series(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>& sa, hipStream_t s);

template <typename T, typename V = T>
void apply_plain(vbh_matrix* m, const V* vals, int K, const void* X, int64_t ldx, void* Y, int64_t ldy, hipStream_t s);
// A fused adjoint step: Y = alpha A^H X + beta X - Z + (re + i im) term.acc (Z
// null: absent).
template <typename T>
struct AdjointStep {
    double alpha, beta;
    const T* Z;
    int64_t ldz;
    SeriesAcc<T> term;
};
template <typename T>
void apply_adjoint(vbh_matrix* m, const T* vals, int K, const void* X, int64_t ldx, void* Y, int64_t ldy,
                   hipStream_t s, const AdjointStep<T>* step = nullptr);
// Y (=, for n == 0, or +=) c_n t over N rows of K columns.
template <typename T>
void cheb_accum(int64_t N, int K, const T* t, int64_t ldt, T* Y, int64_t ldy, const double* coef, int n, hipStream_t s);
void reduce_partials(const double* partials, int G, int E, double* out, bool accumulate, hipStream_t s);

// dtype/precision dispatch: calls f(T*, V*) with typed null pointers of the
// vector type T and the matrix value type V.  precision 0: native (FP64 /
// complex128) throughout; 1: FP32 / complex64 throughout; 2: FP32 values
// against native vectors (the value stream halves, vectors keep full
// precision).
template <typename F>
void dispatch_compute(const vbh_matrix* m, int precision, F&& f) {
    VBH_REQUIRE(precision >= 0 && precision <= 2,
                "precision must be 0 (native), 1 (FP32) or 2 (FP32 values, native vectors)");
    if (m->dtype == VBH_F64) {
        if (precision == 0) f((double*)nullptr, (double*)nullptr);
        else if (precision == 1) f((float*)nullptr, (float*)nullptr);
        else f((double*)nullptr, (float*)nullptr);
    } else {
        if (precision == 0) f((c128*)nullptr, (c128*)nullptr);
        else if (precision == 1) f((c64*)nullptr, (c64*)nullptr);
        else f((c128*)nullptr, (c64*)nullptr);
    }
}

}  // namespace vbh
