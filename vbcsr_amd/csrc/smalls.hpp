// Products and adjoints of uniform blocks of size 1, 2 or 3, any number of
// columns, real and complex, every storage precision, included by the per-type
// lanes_*.hip units.
//
// A lane owns one block row (adjoint: block column) and NC columns, 16 bytes of
// a row of X where K allows it; neighbouring lanes hold the row's other
// columns, the next lanes the next block rows, and with P > 1 the 64 / P lanes
// are repeated P times over partitions of the rows' slots.  A lane loads whole
// blocks (the lanes of a row ask for the same lines) and the BS runs of X they
// meet, and multiplies on the vector ALUs in FP64: blocks this small fill a
// quarter to a half of a 4 x 4 x 4 matrix instruction, and a wave per block row
// spends more on the row than on its products.  A row's last lane overlaps its
// neighbour instead of reading past column K (see quads.hpp).
//
// What bounds it: the launch and the chain of bounds, column and X loads of a
// row, then the address unit (2 to 5 loads a lane and slot).
// Measured in us, a lane per scalar row / a wave per block row (tiles.hpp) /
// here: 64 moments on graphene 150 x 150, size 2, 12 FP32 columns 603 / 1524 /
// 415, 8 FP64 columns 827 / 1538 / 420; 65 x 71, 8 columns, FP32 values with
// FP64 vectors 362 / 412 / 278; 20,000 rows of 61 blocks of size 2, 8 FP64
// columns 20.7 / 18.4 / 15.3, adjoint 49.6 / 25.9 / 22.4; of size 1, one column
// 11.0 (staged through LDS) / 6.8 here.
#pragma once

#include "quads.hpp"

namespace vbh {

// Slots in flight per lane.
constexpr int kSmallBatch = 4;

template <typename T, typename V, int NC>
__device__ __forceinline__ void small_fma(const V& a, const RowRun<T, NC>& x, QuadAcc<T, NC>& acc) {
    if constexpr (Sc<T>::is_complex) {
        const double ar = double(a.re), ai = double(a.im);
#pragma unroll
        for (int t = 0; t < NC; ++t) {
            const double xr = double(x.v[t].re), xi = double(x.v[t].im);
            acc.re[t] = __builtin_fma(-ai, xi, __builtin_fma(ar, xr, acc.re[t]));
            acc.im[t] = __builtin_fma(ai, xr, __builtin_fma(ar, xi, acc.im[t]));
        }
    } else {
#pragma unroll
        for (int t = 0; t < NC; ++t) acc.re[t] = __builtin_fma(double(a), double(x.v[t]), acc.re[t]);
    }
}

// The work of one wave: sh.rows block rows from sh.rows (unit / sh.S), slice
// unit % sh.S.
template <typename T, typename V, int BS, int NC, bool ADJ, bool DOT, bool ACC>
__device__ __forceinline__ void small_wave(const ApplyArgs<T, V>& g, const AdjointPlan& ap, const SmallShape& sh,
                                           const SeriesAcc<T>& sa, int unit, int lane, double& d1, double& d2) {
    constexpr int U = kSmallBatch;
    const DevPattern& p = g.p;
    const int group = unit / sh.S, slice = unit - group * sh.S;
    const int per = 64 / sh.P;
    const int part = lane / per, in = lane - part * per;
    const int rl = in / sh.L;
    const int row = group * sh.rows + rl;
    const int cb = NC * (slice * sh.L + in - rl * sh.L);
    const bool live = rl < sh.rows && row < (ADJ ? p.nbc : p.nbr) && cb < g.K;
    QuadAcc<T, NC> acc[BS] = {};
    const int c0 = cb < g.K - NC ? cb : g.K - NC;
    if (live) {
        const int* ptr = ADJ ? ap.t_ptr : p.row_ptr;
        const int kb = ptr[row], ke = ptr[row + 1];
        const T* xc = g.X + c0;
        for (int s0 = kb + part; s0 < ke; s0 += U * sh.P) {
            // slots past a row's last read zeros; those that no row of the wave
            // has are skipped
            int64_t xo[U];
            RowRun<V, BS * BS> av[U];
            RowRun<T, NC> xv[U][BS];
            bool any[U];
#pragma unroll
            for (int u = 0; u < U; ++u) any[u] = u == 0 || __ballot(s0 + u * sh.P < ke) != 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (!any[u]) continue;
                const bool on = s0 + u * sh.P < ke;
                const int s = on ? s0 + u * sh.P : ke - 1;
                if constexpr (ADJ) xo[u] = ap.t_rows[s].x;
                else xo[u] = int64_t(p.col_ind[s]) * BS;
                const int64_t at = ADJ ? ap.t_voff[s] : int64_t(s) * (BS * BS);
                av[u] = *reinterpret_cast<const RowRun<V, BS * BS>*>(or_zeros(on, g.vals + at));
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (!any[u]) continue;
                const bool on = s0 + u * sh.P < ke;
                const T* xr = or_zeros(on, xc + xo[u] * g.ldx);
                const int64_t ld = on ? g.ldx : 0;
#pragma unroll
                for (int m = 0; m < BS; ++m) xv[u][m] = *reinterpret_cast<const RowRun<T, NC>*>(xr + m * ld);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (!any[u]) continue;
#pragma unroll
                for (int m = 0; m < BS; ++m)
#pragma unroll
                    for (int a = 0; a < BS; ++a)
                        small_fma<T, V, NC>(ADJ ? Sc<V>::conj(av[u].v[m * BS + a]) : av[u].v[a * BS + m], xv[u][m],
                                            acc[a]);
            }
        }
    }
    for (int d = per; d < 64; d <<= 1) {
#pragma unroll
        for (int a = 0; a < BS; ++a)
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                acc[a].re[t] += __shfl_xor(acc[a].re[t], d, 64);
                if constexpr (Sc<T>::is_complex) acc[a].im[t] += __shfl_xor(acc[a].im[t], d, 64);
            }
    }
    if (live && part == 0) {
#pragma unroll
        for (int a = 0; a < BS; ++a) {
            const int64_t yr = int64_t(row) * BS + a;
            quad_emit<T, V, NC, DOT, ACC, ADJ>(g, yr, yr, c0, cb - c0, acc[a], d1, d2, sa);
        }
    }
}

template <typename T, typename V, int BS, int NC, bool ADJ, bool DOT, bool ACC>
__global__ __launch_bounds__(kThreads) void k_apply_smalls(ApplyArgs<T, V> g, AdjointPlan ap, SmallShape sh,
                                                           SeriesAcc<T> sa) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(g.G);
    const int unit = chunk * kWaves + __builtin_amdgcn_readfirstlane(wave);
    double d1 = 0.0, d2 = 0.0;
    small_wave<T, V, BS, NC, ADJ, DOT, ACC>(g, ap, sh, sa, unit, lane, d1, d2);
    if constexpr (DOT) write_dots(lane, wave, d1, d2, g.partials + int64_t(chunk) * 2);
}

template <typename T, typename V, bool ADJ, bool DOT, bool ACC>
static void launch_smalls_as(int bs, const ApplyArgs<T, V>& a, const AdjointPlan& ap, const SmallShape& sh,
                             const SeriesAcc<T>& sa, hipStream_t s) {
    const dim3 grid(a.G), block(kThreads);
    auto go = [&](auto BS_, auto NC_) {
        constexpr int BS = decltype(BS_)::value, NC = decltype(NC_)::value;
        if constexpr (NC * sizeof(T) <= 16)
            hipLaunchKernelGGL((k_apply_smalls<T, V, BS, NC, ADJ, DOT, ACC>), grid, block, 0, s, a, ap, sh, sa);
        else
            throw Error(VBH_ERR_ARG, "internal: no small block kernel for this shape");
    };
    auto sized = [&](auto NC_) {
        switch (bs) {
            case 1: go(std::integral_constant<int, 1>{}, NC_); break;
            case 2: go(std::integral_constant<int, 2>{}, NC_); break;
            default: go(std::integral_constant<int, 3>{}, NC_); break;
        }
    };
    switch (sh.NC) {
        case 1: sized(std::integral_constant<int, 1>{}); break;
        case 2: sized(std::integral_constant<int, 2>{}); break;
        default: sized(std::integral_constant<int, 4>{}); break;
    }
    VBH_CHECK_HIP(hipGetLastError());
}

template <typename T, typename V>
void launch_smalls(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>* sa, hipStream_t s) {
    const SmallShape sh = small_shape<T>(m->nnzb, m->nbr, a.K);
    ApplyArgs<T, V> b = a;
    b.G = sh.G;
    const int bs = m->uniform_bs;
    if (a.partials) launch_smalls_as<T, V, false, true, false>(bs, b, AdjointPlan{}, sh, SeriesAcc<T>{}, s);
    else if (sa) launch_smalls_as<T, V, false, false, true>(bs, b, AdjointPlan{}, sh, *sa, s);
    else launch_smalls_as<T, V, false, false, false>(bs, b, AdjointPlan{}, sh, SeriesAcc<T>{}, s);
}
template <typename T>
void launch_smalls_adjoint(const vbh_matrix* m, const ApplyArgs<T>& a, const AdjointPlan& ap, const SeriesAcc<T>* term,
                           hipStream_t s) {
    const SmallShape sh = small_shape<T>(m->nnzb, m->nbc, a.K);
    ApplyArgs<T> b = a;
    b.G = sh.G;
    if (term) launch_smalls_as<T, T, true, false, true>(m->uniform_bs, b, ap, sh, *term, s);
    else launch_smalls_as<T, T, true, false, false>(m->uniform_bs, b, ap, sh, SeriesAcc<T>{}, s);
}

#define VBH_SMALLS_INSTANTIATE(T, V) \
    template void launch_smalls<T, V>(const vbh_matrix*, const ApplyArgs<T, V>&, const SeriesAcc<T>*, hipStream_t);
#define VBH_SMALLS_ADJOINT_INSTANTIATE(T)                                                                  \
    template void launch_smalls_adjoint<T>(const vbh_matrix*, const ApplyArgs<T>&, const AdjointPlan&, const SeriesAcc<T>*, \
                                           hipStream_t);

}  // namespace vbh
