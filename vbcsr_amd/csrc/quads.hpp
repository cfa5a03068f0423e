// SpMM of uniform 4 x 4 blocks on the FP64 matrix cores (real and complex,
// every storage precision), included by the per-type lanes_*.hip units.
//
// One wavefront owns four consecutive block rows (few of them with long rows: one
// work-group, quad_grid).  v_mfma_f64_4x4x4f64 is
// four independent 4 x 4 x 4 products (lane = i + 4 b + 16 k; A operand: row i,
// step k; B operand: step k, column i; result: row k, column i, of product b),
// and product b belongs to block row 4 w + b.  Lane (i, b, k) loads row i of
// block 4 u + k of its block row -- one 16-byte run in FP32 -- and NG
// consecutive columns of that block's four X rows; instruction m then
// contracts column m of four neighbouring blocks at once.  So every load is
// 8 to 32 bytes a lane (a load instruction costs the address unit a cycle per
// four lanes whatever their width), there is no cross-lane exchange, no
// reduction, and no padding inside a block.
//
// Complex values are two real products per component on the same operands:
// re += Are Xre - Aim Xim, im += Are Xim + Aim Xre.
//
// The columns go to S slices of 4 NG columns, one wave each.  Lane i of a slice
// starting at v0 takes columns c0 .. c0 + NG - 1 with c0 = min(v0 + NG i, K -
// NG): near column K neighbouring lanes overlap instead of reading past the
// row, compute the same sums, and only the first owner stores them and counts
// them in a dot product.
//
// What bounds it: the matrix (streamed once) and the X rows through the L1s.
// Before, a lane held one scalar row and every X element reached it by two
// DPP moves and a conversion, about 120 vector instructions per block and
// lane of a 10-column FP32 step.  Measured before / now, us per launch: the
// fused 10-column KPM step on graphene 200 x 200 FP32 28.0 / 25.2, FP64 42.2 /
// 33.6, FP32 values with FP64 vectors 39.5 / 29.3; 60 x 60 (launches of a few
// us) 17.0 / 5.6, 18.1 / 5.9, 18.8 / 5.7; 4 complex64 columns on 60 x 60
// 15.3 / 4.2; 64 columns FP64 on 200 x 200 331 / 159.  Other layouts of the
// same instruction were slower: one slot per instruction with a dword of A
// per lane (FP32 36 us), and one block row per instruction with 16 columns
// (FP32 48 us, FP64 66 us a step).
#pragma once

#include "apply.hpp"

namespace vbh {

// Value of lane (l & ~3) + B of v's quad (DPP quad permutation, any 4/8/16-byte type).
template <int B, typename V>
__device__ __forceinline__ V quad_bcast(V v) {
    static_assert(sizeof(V) % 4 == 0, "32-bit granular types only");
    constexpr int ctrl = B * 0x55;  // quad_perm [B, B, B, B]
    union {
        V v;
        int w[sizeof(V) / 4];
    } in{v}, out;
#pragma unroll
    for (int i = 0; i < int(sizeof(V) / 4); ++i) out.w[i] = __builtin_amdgcn_mov_dpp(in.w[i], ctrl, 0xf, 0xf, false);
    return out.v;
}

// Lane u's v of the quad, u a compile-time constant after unrolling.
__device__ __forceinline__ int quad_pick(int v, int u) {
    switch (u) {
        case 0: return quad_bcast<0>(v);
        case 1: return quad_bcast<1>(v);
        case 2: return quad_bcast<2>(v);
        default: return quad_bcast<3>(v);
    }
}

// N consecutive elements with the alignment of the underlying real type (the
// loads and stores below become the widest the target has).
template <typename T, int N>
struct __attribute__((packed, aligned(sizeof(typename Sc<T>::real)))) RowRun {
    T v[N];
};

// FP64 sums of one lane: NG columns of one row of Y.
template <typename T, int NG>
struct QuadAcc {
    double re[NG];
    double im[Sc<T>::is_complex ? NG : 1];
};

// acc += the products of one contraction step: a, one element of a block, with
// NG columns x of the X row it meets.
template <typename T, typename V, int NG>
__device__ __forceinline__ void quad_mfma(const V& a, const RowRun<T, NG>& x, QuadAcc<T, NG>& acc) {
    if constexpr (Sc<T>::is_complex) {
        const double ar = double(a.re), ai = double(a.im);
#pragma unroll
        for (int t = 0; t < NG; ++t) {
            const double xr = double(x.v[t].re), xi = double(x.v[t].im);
            acc.re[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, xr, acc.re[t], 0, 0, 0);
            acc.im[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, xi, acc.im[t], 0, 0, 0);
            acc.re[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(-ai, xi, acc.re[t], 0, 0, 0);
            acc.im[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(ai, xr, acc.im[t], 0, 0, 0);
        }
    } else {
        const double ad = double(a);
#pragma unroll
        for (int t = 0; t < NG; ++t)
            acc.re[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(ad, double(x.v[t]), acc.re[t], 0, 0, 0);
    }
}

// a += b.
template <typename T, int NG>
__device__ __forceinline__ void quad_sum(QuadAcc<T, NG>& a, const QuadAcc<T, NG>& b) {
#pragma unroll
    for (int t = 0; t < NG; ++t) {
        a.re[t] += b.re[t];
        if constexpr (Sc<T>::is_complex) a.im[t] += b.im[t];
    }
}

// Fused epilogue of NG columns c0.. of row yr of Y (row xr of X for the X_own
// terms); the first `skip` columns belong to another lane.  ACC: also the series
// accumulation sa, or with TERM its counterpart Y += (re + i im) sa.acc.
template <typename T, typename V, int NG, bool DOT, bool ACC, bool TERM = false>
__device__ __forceinline__ void quad_emit(const ApplyArgs<T, V>& g, int64_t yr, int64_t xr, int c0, int skip,
                                          const QuadAcc<T, NG>& acc, double& d1, double& d2, const SeriesAcc<T>& sa) {
    using A = typename Wide<T>::type;
    using Run = RowRun<T, NG>;
    Run xo{}, zo{}, wo{}, so{}, out;
    const bool need_x = DOT || g.beta != 0.0, need_z = g.gamma != 0.0, need_w = DOT && g.W != nullptr;
    if (need_x) xo = *reinterpret_cast<const Run*>(g.X + xr * g.ldx + c0);
    if (need_z) zo = *reinterpret_cast<const Run*>(g.Z + yr * g.ldz + c0);
    if (need_w) wo = *reinterpret_cast<const Run*>(g.W + yr * g.ldw + c0);
    if constexpr (ACC) so = *reinterpret_cast<const Run*>(sa.acc + yr * sa.ld + c0);
#pragma unroll
    for (int t = 0; t < NG; ++t) {
        A y;
        if constexpr (Sc<T>::is_complex) y = A{acc.re[t], acc.im[t]};
        else y = acc.re[t];
        if constexpr (ACC && TERM) y = widen(narrow_to<T>(y));  // the product as a vector of its own type
        y = rscale(g.alpha, y);
        if (g.beta != 0.0) y = y + rscale(g.beta, widen(xo.v[t]));
        if (need_z) y = y + rscale(g.gamma, widen(zo.v[t]));
        if constexpr (ACC && TERM) y = Sc<A>::fma(Sc<A>::make(sa.re, sa.im), widen(so.v[t]), y);
        out.v[t] = narrow_to<T>(y);
        // dots and series of the stored (rounded) value: the state the
        // recursion carries on; a term is added in FP64 and rounded once
        const A ys = widen(out.v[t]);
        if constexpr (DOT) {
            const double t1 = redot(need_w ? widen(wo.v[t]) : ys, ys);
            const double t2 = redot(widen(xo.v[t]), ys);
            d1 += t >= skip ? t1 : 0.0;
            d2 += t >= skip ? t2 : 0.0;
        }
        if constexpr (ACC && !TERM)
            so.v[t] = narrow_to<T>(Sc<A>::fma(Sc<A>::make(sa.re, sa.im), ys, widen(so.v[t])));
    }
    T* yp = g.Y + yr * g.ldy + c0;
    if (skip == 0) {
        *reinterpret_cast<Run*>(yp) = out;
        if constexpr (ACC && !TERM) *reinterpret_cast<Run*>(sa.acc + yr * sa.ld + c0) = so;
    } else {
#pragma unroll
        for (int t = 0; t < NG; ++t)
            if (t >= skip) {
                yp[t] = out.v[t];
                if constexpr (ACC && !TERM) sa.acc[yr * sa.ld + c0 + t] = so.v[t];
            }
    }
}

// Groups of four slots in flight per lane (a block row of V, and NG columns of
// four X rows of T each).  More waves serve better than more loads a wave: one
// group except for the narrowest operands (graphene 200 x 200, U = 1 / 2 / 3:
// 10 FP32 columns 19.9 / 24.8 / 21.7 us, 10 FP64 columns 29.1 / 35.7 / 30.7 us;
// 60 x 60, 4 FP32 columns 3.8 / 3.9 / 3.4 us).  Several units per wave with the
// next unit's bounds and columns in flight, or the epilogue's operands loaded
// ahead of the slot loop, cost registers and were 3-10 % slower.
template <typename T, typename V, int NG>
constexpr int quad_batch() {
    return NG == 1 && sizeof(V) + sizeof(T) <= 16 ? 3 : 1;
}

// Sums of a lane to and from LDS, 64 values apart.
template <typename T, int NG>
__device__ __forceinline__ void sums_store(double* at, const QuadAcc<T, NG>& a) {
#pragma unroll
    for (int t = 0; t < NG; ++t) {
        at[64 * t] = a.re[t];
        if constexpr (Sc<T>::is_complex) at[64 * (NG + t)] = a.im[t];
    }
}
template <typename T, int NG>
__device__ __forceinline__ void sums_add(const double* at, QuadAcc<T, NG>& a) {
#pragma unroll
    for (int t = 0; t < NG; ++t) {
        a.re[t] += at[64 * t];
        if constexpr (Sc<T>::is_complex) a.im[t] += at[64 * (NG + t)];
    }
}

// The work of one wave: block rows 4 (unit / slices) to + 3, slice unit % slices.
// SPLIT: of one work-group, whose waves take every kWaves-th pass of 16 slots and
// are summed in the order of the waves, in `sums` (kWaves - 1 areas).
template <typename T, typename V, int NG, bool DOT, bool ACC, bool SPLIT = false>
__device__ __forceinline__ void quad_wave(const ApplyArgs<T, V>& g, int slices, const SeriesAcc<T>& sa, int unit,
                                          int lane, double& d1, double& d2, int wave = 0, double* sums = nullptr) {
    constexpr int U = quad_batch<T, V, NG>();
    const DevPattern& p = g.p;
    const int rows4 = unit / slices;
    const int li = lane & 3, lb = (lane >> 2) & 3, lk = lane >> 4;
    if (rows4 * 4 < p.nbr) {
        const int row = rows4 * 4 + lb;
        const bool live = row < p.nbr;
        const int kb = live ? p.row_ptr[row] : 0;
        const int cnt = live ? p.row_ptr[row + 1] - kb : 0;
        // longest of the four rows (wave-uniform)
        int nmax = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int c = __builtin_amdgcn_readlane(cnt, 4 * b);
            nmax = c > nmax ? c : nmax;
        }
        const int cb = (unit - rows4 * slices) * 4 * NG + NG * li;
        const int c0 = cb < g.K - NG ? cb : g.K - NG;
        const int skip = cb - c0 < NG ? cb - c0 : NG;
        const int last = cnt > 0 ? cnt - 1 : 0;
        const int kb0 = cnt > 0 ? kb : 0;  // rows without blocks read the column of slot 0
        const RowRun<V, 4>* va = reinterpret_cast<const RowRun<V, 4>*>(g.vals) + int64_t(kb0) * 4 + li;
        const T* xc = g.X + c0;
        QuadAcc<T, NG> acc[2] = {};  // even and odd contraction steps
        for (int j0 = SPLIT ? 16 * wave : 0; j0 < nmax; j0 += SPLIT ? 16 * kWaves : 16) {
            // this lane's slots of the pass are j0 + 4 u + k; lane i of a quad
            // reads the column index of u = i
            const int sc = j0 + 4 * li + lk;
            const int colv = p.col_ind[kb0 + (sc < last ? sc : last)];
#pragma unroll
            for (int u0 = 0; u0 < 4; u0 += U) {
                if (j0 + 4 * u0 >= nmax) break;
                RowRun<V, 4> av[U];
                RowRun<T, NG> xv[U][4];
                // every load of the batch is unconditional and in bounds: slots
                // past a row's last read zeros
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (u0 + u >= 4) continue;
                    const int s = j0 + 4 * (u0 + u) + lk;
                    const int col = quad_pick(colv, u0 + u);
                    av[u] = *or_zeros(s < cnt, va + int64_t(s) * 4);
                    const T* xr = or_zeros(s < cnt, xc + int64_t(col) * 4 * g.ldx);
                    const int64_t ld = s < cnt ? g.ldx : 0;
#pragma unroll
                    for (int m = 0; m < 4; ++m) xv[u][m] = *reinterpret_cast<const RowRun<T, NG>*>(xr + m * ld);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (u0 + u >= 4) continue;
#pragma unroll
                    for (int m = 0; m < 4; ++m) quad_mfma<T, V, NG>(av[u].v[m], xv[u][m], acc[m & 1]);
                }
            }
        }
        quad_sum<T, NG>(acc[0], acc[1]);
        if constexpr (SPLIT) {
            constexpr int area = 64 * NG * (Sc<T>::is_complex ? 2 : 1);
            if (wave > 0) sums_store<T, NG>(sums + (wave - 1) * area + lane, acc[0]);
            __syncthreads();
            if (wave > 0) return;
#pragma unroll
            for (int w = 0; w < kWaves - 1; ++w) sums_add<T, NG>(sums + w * area + lane, acc[0]);
        }
        if (live) {
            const int64_t yr = int64_t(row) * 4 + lk;
            quad_emit<T, V, NG, DOT, ACC>(g, yr, yr, c0, skip, acc[0], d1, d2, sa);
        }
    }
}

template <typename T, typename V, int NG, bool DOT, bool ACC, bool SPLIT>
__global__ __launch_bounds__(kThreads) void k_apply_quads(ApplyArgs<T, V> g, int slices, SeriesAcc<T> sa) {
    __shared__ double sums[SPLIT ? (kWaves - 1) * 64 * NG * (Sc<T>::is_complex ? 2 : 1) : 1];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(g.G);
    const int unit = SPLIT ? chunk : chunk * kWaves + __builtin_amdgcn_readfirstlane(wave);
    double d1 = 0.0, d2 = 0.0;
    quad_wave<T, V, NG, DOT, ACC, SPLIT>(g, slices, sa, unit, lane, d1, d2, __builtin_amdgcn_readfirstlane(wave), sums);
    if constexpr (DOT) write_dots(lane, wave, d1, d2, g.partials + int64_t(chunk) * 2);
}

template <typename T, typename V, bool DOT, bool ACC>
static void launch_quads_as(const ApplyArgs<T, V>& a, const QuadGrid& q, const SeriesAcc<T>& sa, hipStream_t s) {
    const dim3 grid(a.G), block(kThreads);
    auto go = [&](auto NG_) {
        constexpr int NG = decltype(NG_)::value;
        if constexpr (NG <= kQuadMaxGroups<T>) {
            if (q.split) hipLaunchKernelGGL((k_apply_quads<T, V, NG, DOT, ACC, true>), grid, block, 0, s, a, q.S, sa);
            else hipLaunchKernelGGL((k_apply_quads<T, V, NG, DOT, ACC, false>), grid, block, 0, s, a, q.S, sa);
        } else {
            throw Error(VBH_ERR_ARG, "internal: no 4 x 4 block kernel for this shape");
        }
    };
    switch (q.NG) {
        case 1: go(std::integral_constant<int, 1>{}); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        default: go(std::integral_constant<int, 4>{}); break;
    }
    VBH_CHECK_HIP(hipGetLastError());
}

template <typename T, typename V>
void launch_quads(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>* sa, hipStream_t s) {
    const QuadGrid q = quad_grid<T>(RowStats(m, m->nbr), a.K);
    ApplyArgs<T, V> b = a;
    b.G = q.G;
    if (a.partials) launch_quads_as<T, V, true, false>(b, q, SeriesAcc<T>{}, s);
    else if (sa) launch_quads_as<T, V, false, true>(b, q, *sa, s);
    else launch_quads_as<T, V, false, false>(b, q, SeriesAcc<T>{}, s);
}

#define VBH_QUADS_INSTANTIATE(T, V) \
    template void launch_quads<T, V>(const vbh_matrix*, const ApplyArgs<T, V>&, const SeriesAcc<T>*, hipStream_t);

}  // namespace vbh
