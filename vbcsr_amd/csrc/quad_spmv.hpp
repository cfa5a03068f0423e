// SpMV (K = 1) of uniform 4 x 4 blocks and its adjoint, real and complex,
// included by the per-type lanes_*.hip units.
//
// A wavefront owns four consecutive block rows (adjoint: block columns), one
// per 16 lanes: lane i + 4 k of the 16 takes row i of the slots 4 u + k.  It
// loads a whole block row (16 bytes in FP32, 64 in complex128) and entry i of
// the block's x, so one load instruction of the wave covers four consecutive
// blocks of four block rows.  Forward: the quad broadcasts its four x entries
// to each other, and the row sums merge over k by two rotations of the 16
// lanes; adjoint: a lane adds its row times its x entry to four column sums,
// which merge over the 16 lanes with lane i keeping column i.
//
// What bounds it: the value stream; a row of ten blocks costs the row bounds,
// the column indices, and three batches of loads.  Measured before / now in us,
// forward (values staged through LDS) and adjoint (one block entry a lane, a
// serial chain over the incoming blocks), honeycomb lattice: 100 x 100 cells
// complex128 (51 MB) 16.3, 16.4 / 10.7, 10.4, FP64 9.9, 12.6 / 4.5, 5.4; 200 x
// 200 FP64 42.3, 39.1 / 17.6, 18.9, FP32 35.1, 34.4 / 12.6, 13.6; 400 x 400 FP64
// (409 MB) 158, 206 / 85, 92 (4.8 TB/s).  With four x entries loaded a lane
// instead of broadcast the forward took 20.8 us (200 x 200) and 108 us.
#pragma once

#include "tiles.hpp"

namespace vbh {

template <int N>
__device__ __forceinline__ double row_rot(double v) {
    return row_rotate<N>(v);
}
template <int N>
__device__ __forceinline__ c128 row_rot(c128 v) {
    return c128{row_rotate<N>(v.re), row_rotate<N>(v.im)};
}
// v of lane (l ^ M) of the quad, M = 1 or 2.
template <int M>
__device__ __forceinline__ double quad_xor(double v) {
    constexpr int ctrl = M == 1 ? 0xb1 : 0x4e;  // quad_perm [1, 0, 3, 2] / [2, 3, 0, 1]
    union {
        double d;
        int w[2];
    } in{v}, out;
    out.w[0] = __builtin_amdgcn_mov_dpp(in.w[0], ctrl, 0xf, 0xf, false);
    out.w[1] = __builtin_amdgcn_mov_dpp(in.w[1], ctrl, 0xf, 0xf, false);
    return out.d;
}
template <int M>
__device__ __forceinline__ c128 quad_xor(c128 v) {
    return c128{quad_xor<M>(v.re), quad_xor<M>(v.im)};
}

// Slots of each lane in flight: two batches for the narrow types.
template <typename T>
constexpr int kQuadSpmvBatch = sizeof(T) <= 8 ? 2 : 1;

// SPLIT: a work-group per four block rows, its waves on every kWaves-th pass of 16
// slots, summed in their order.
template <typename T, bool ADJ, bool FUSED, bool ACC, bool SPLIT>
__global__ __launch_bounds__(kThreads) void k_quad_spmv(ApplyArgs<T> g, AdjointPlan ap, SeriesAcc<T> sa) {
    using A = typename Wide<T>::type;
    constexpr int U = kQuadSpmvBatch<T>;
    const DevPattern& p = g.p;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(g.G);
    const int rows4 = SPLIT ? chunk : chunk * kWaves + __builtin_amdgcn_readfirstlane(wave);
    const int nrows = ADJ ? p.nbc : p.nbr;
    const int li = lane & 3, lk = (lane >> 2) & 3, lb = lane >> 4;
    double d1 = 0.0, d2 = 0.0;
    if (rows4 * 4 < nrows) {
        const int row = rows4 * 4 + lb;
        const bool live = row < nrows;
        const int* ptr = ADJ ? ap.t_ptr : p.row_ptr;
        const int kb = live ? ptr[row] : 0;
        const int cnt = live ? ptr[row + 1] - kb : 0;
        int nmax = 0;  // longest of the four rows (wave-uniform)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int c = __builtin_amdgcn_readlane(cnt, 16 * b);
            nmax = c > nmax ? c : nmax;
        }
        const int last = cnt > 0 ? cnt - 1 : 0;
        const int kb0 = cnt > 0 ? kb : 0;  // rows without blocks read the column of slot 0
        constexpr int NA = ADJ ? 4 : 1;
        A acc[NA];
#pragma unroll
        for (int t = 0; t < NA; ++t) acc[t] = Sc<A>::zero();
        for (int j0 = SPLIT ? 16 * __builtin_amdgcn_readfirstlane(wave) : 0; j0 < nmax; j0 += SPLIT ? 16 * kWaves : 16) {
            // lane i of a quad looks after slot j0 + 4 i + k: the first x row of
            // its block, and in the adjoint the block's place in the values
            const int sl = j0 + 4 * li + lk, slc = kb0 + (sl < last ? sl : last);
            int xv;
            int vlo = 0, vhi = 0;
            if constexpr (ADJ) {
                xv = ap.t_rows[slc].x;
                const int64_t vo = ap.t_voff[slc];
                vlo = int(uint32_t(uint64_t(vo)));
                vhi = int(uint32_t(uint64_t(vo) >> 32));
            } else {
                xv = p.col_ind[slc] * 4;
            }
#pragma unroll
            for (int u0 = 0; u0 < 4; u0 += U) {
                if (j0 + 4 * u0 >= nmax) break;
                RowRun<T, 4> av[U];
                T x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int s = j0 + 4 * (u0 + u) + lk;
                    const bool on = s < cnt;  // else zeros
                    const int xr = quad_pick(xv, u0 + u);
                    int64_t at;
                    if constexpr (ADJ)
                        at = int64_t((uint64_t(uint32_t(quad_pick(vhi, u0 + u))) << 32) |
                                     uint32_t(quad_pick(vlo, u0 + u)));
                    else
                        at = int64_t(kb0 + s) * 16;
                    av[u] = *reinterpret_cast<const RowRun<T, 4>*>(or_zeros(on, g.vals + at + 4 * li));
                    x[u] = *or_zeros(on, g.X + int64_t(xr + li) * g.ldx);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const T* a = av[u].v;
                    if constexpr (ADJ) {
                        const A xw = widen(x[u]);
#pragma unroll
                        for (int b = 0; b < 4; ++b) acc[b] = Sc<A>::fma(widen(Sc<T>::conj(a[b])), xw, acc[b]);
                    } else {
                        acc[0] = Sc<A>::fma(widen(a[0]), widen(quad_bcast<0>(x[u])), acc[0]);
                        acc[0] = Sc<A>::fma(widen(a[1]), widen(quad_bcast<1>(x[u])), acc[0]);
                        acc[0] = Sc<A>::fma(widen(a[2]), widen(quad_bcast<2>(x[u])), acc[0]);
                        acc[0] = Sc<A>::fma(widen(a[3]), widen(quad_bcast<3>(x[u])), acc[0]);
                    }
                }
            }
        }
        A y;
        if constexpr (ADJ) {
            // column i to lane i of the quad: exchange halves, then neighbours
            const bool hi = li & 2, odd = li & 1;
            const A k0 = pick(hi, acc[2], acc[0]), k1 = pick(hi, acc[3], acc[1]);
            const A s0 = pick(hi, acc[0], acc[2]), s1 = pick(hi, acc[1], acc[3]);
            const A m0 = k0 + quad_xor<2>(s0), m1 = k1 + quad_xor<2>(s1);
            y = pick(odd, m1, m0) + quad_xor<1>(pick(odd, m0, m1));
        } else {
            y = acc[0];
        }
        y = y + row_rot<2>(y);
        y = y + row_rot<1>(y);
        if constexpr (SPLIT) {
            __shared__ A sums[kWaves - 1][64];
            if (wave > 0) sums[wave - 1][lane] = y;
            __syncthreads();
            if (wave == 0)
#pragma unroll
                for (int w = 0; w < kWaves - 1; ++w) y = y + sums[w][lane];
        }
        if (live && lk == 0 && (!SPLIT || wave == 0)) {
            const int64_t yr = int64_t(row) * 4 + li;
            emit<T, FUSED, ACC, ADJ>(g, yr, yr, 0, y, d1, d2, &sa);
        }
    }
    if constexpr (FUSED && !ADJ && !ACC) {
        if (g.partials != nullptr) write_dots(lane, wave, d1, d2, g.partials + int64_t(chunk) * 2);
    }
}

template <typename T, bool ADJ, bool FUSED, bool ACC>
static void launch_quad_spmv_as(const vbh_matrix* m, const ApplyArgs<T>& a, const AdjointPlan& ap, const SeriesAcc<T>& sa,
                                hipStream_t s) {
    const QuadSpmvGrid q = quad_spmv_grid(m, ADJ ? m->nbc : m->nbr);
    ApplyArgs<T> b = a;
    b.G = q.G;
    const dim3 grid(q.G), block(kThreads);
    if (q.split) hipLaunchKernelGGL((k_quad_spmv<T, ADJ, FUSED, ACC, true>), grid, block, 0, s, b, ap, sa);
    else hipLaunchKernelGGL((k_quad_spmv<T, ADJ, FUSED, ACC, false>), grid, block, 0, s, b, ap, sa);
    VBH_CHECK_HIP(hipGetLastError());
}
template <typename T>
void launch_quad_spmv(const vbh_matrix* m, const ApplyArgs<T>& a, bool fused, const SeriesAcc<T>* sa, hipStream_t s) {
    if (sa) launch_quad_spmv_as<T, false, true, true>(m, a, AdjointPlan{}, *sa, s);
    else if (fused) launch_quad_spmv_as<T, false, true, false>(m, a, AdjointPlan{}, SeriesAcc<T>{}, s);
    else launch_quad_spmv_as<T, false, false, false>(m, a, AdjointPlan{}, SeriesAcc<T>{}, s);
}
template <typename T>
void launch_quad_spmv_adjoint(const vbh_matrix* m, const ApplyArgs<T>& a, const AdjointPlan& ap, const SeriesAcc<T>* term,
                              hipStream_t s) {
    if (term) launch_quad_spmv_as<T, true, true, true>(m, a, ap, *term, s);
    else launch_quad_spmv_as<T, true, false, false>(m, a, ap, SeriesAcc<T>{}, s);
}

#define VBH_QUAD_SPMV_INSTANTIATE(T)                                                                                     \
    template void launch_quad_spmv<T>(const vbh_matrix*, const ApplyArgs<T>&, bool, const SeriesAcc<T>*, hipStream_t);   \
    template void launch_quad_spmv_adjoint<T>(const vbh_matrix*, const ApplyArgs<T>&, const AdjointPlan&, const SeriesAcc<T>*, \
                                              hipStream_t);

}  // namespace vbh
