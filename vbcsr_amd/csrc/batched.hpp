// Steps of the batched recursion on the kernels of single matrices (tiles.hpp,
// quads.hpp, smalls.hpp): a work-group finds its matrix by binary search over the
// items' first groups and does that matrix's share there; groups past the last
// matrix's rows write zero partials.  Whether waves share a row, and the parts of
// wide blocks, follow the rules of single matrices on the sums over the batch (32
// moments of 12 block rows of 6 blocks of 255, 2 FP64 columns 9.0 ms without, 0.37 with;
// 0.69 on a lane per scalar row).  Included by the per-type lanes_*.hip units.
//
// Measured, us per step of 8000 block rows on a 20^3 grid of 19 blocks a row, the
// families of lanes.hpp as tuned / here: blocks of 1, 4, 9, 13, FP64, 8 columns
// 54.7 / 26.4, 17 columns 90 / 45; blocks of 4-8, 2 columns 22.5 / 17.6; uniform 4,
// FP32, 17 columns 139 / 11.3; uniform 3, FP64, 17 columns 88 / 18.3.  With 32 or
// 64 real columns on FP32 values of variable blocks the block-row wave kernel of
// lanes.hpp is the faster one (blocks of 1, 4, 9, 13, 32 columns: 55 here, 35).
#pragma once

#include "lanes.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {

template <typename T, typename V, int NG, bool SPLIT>
__global__ __launch_bounds__(kThreads) void k_batched_tiles(const BatchItem<T, V>* __restrict__ items, int nitems,
                                                            int Gtot, int K, int ld, int step, double alpha,
                                                            double beta, double gamma0, double gamma, int mode,
                                                            double* __restrict__ partials, int slices, int parts) {
    __shared__ TileArea areas[kWaves];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int gg = xcd_chunk(Gtot);
    const int lo = batch_item<T, V, false>(items, nitems, gg);
    const ApplyArgs<T, V> a = batch_args(items, lo, K, ld, step, alpha, beta, gamma0, gamma, mode);
    const int group = gg - items[lo].g_base, unit = SPLIT ? group : group * kWaves + __builtin_amdgcn_readfirstlane(wave);
    double d1 = 0.0, d2 = 0.0;
    tile_wave<T, V, NG, false, true, false, SPLIT>(a, AdjointPlan{}, slices, parts, SeriesAcc<T>{}, areas, wave, unit,
                                                   lane, d1, d2);
    write_dots(lane, wave, d1, d2, partials + int64_t(gg) * 2);
}

template <typename T, typename V, int NG, bool SPLIT>
__global__ __launch_bounds__(kThreads) void k_batched_quads(const BatchItem<T, V>* __restrict__ items, int nitems,
                                                            int Gtot, int K, int ld, int step, double alpha,
                                                            double beta, double gamma0, double gamma, int mode,
                                                            double* __restrict__ partials, int slices) {
    __shared__ double sums[SPLIT ? (kWaves - 1) * 64 * NG * (Sc<T>::is_complex ? 2 : 1) : 1];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gg = xcd_chunk(Gtot);
    const int lo = batch_item<T, V, false>(items, nitems, gg);
    const ApplyArgs<T, V> a = batch_args(items, lo, K, ld, step, alpha, beta, gamma0, gamma, mode);
    const int group = gg - items[lo].g_base, unit = SPLIT ? group : group * kWaves + wave;
    double d1 = 0.0, d2 = 0.0;
    quad_wave<T, V, NG, true, false, SPLIT>(a, slices, SeriesAcc<T>{}, unit, lane, d1, d2, wave, sums);
    write_dots(lane, wave, d1, d2, partials + int64_t(gg) * 2);
}

template <typename T, typename V, int BS, int NC>
__global__ __launch_bounds__(kThreads) void k_batched_smalls(const BatchItem<T, V>* __restrict__ items, int nitems,
                                                             int Gtot, int K, int ld, int step, double alpha,
                                                             double beta, double gamma0, double gamma, int mode,
                                                             double* __restrict__ partials, SmallShape sh) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int gg = xcd_chunk(Gtot);
    const int lo = batch_item<T, V, false>(items, nitems, gg);
    const ApplyArgs<T, V> a = batch_args(items, lo, K, ld, step, alpha, beta, gamma0, gamma, mode);
    const int unit = (gg - items[lo].g_base) * kWaves + __builtin_amdgcn_readfirstlane(wave);
    double d1 = 0.0, d2 = 0.0;
    small_wave<T, V, BS, NC, false, true, false>(a, AdjointPlan{}, sh, SeriesAcc<T>{}, unit, lane, d1, d2);
    write_dots(lane, wave, d1, d2, partials + int64_t(gg) * 2);
}

template <typename T, typename V>
void launch_batched_rows(const BatchItem<T, V>* items, int nitems, int Gtot, int K, int ld, int rows,
                         const RowsShape& shape, int step, double alpha, double beta, double gamma0, double gamma,
                         int mode, double* partials, hipStream_t s) {
    auto go = [&](auto kernel, auto... sizes) {
        hipLaunchKernelGGL(kernel, dim3(Gtot), dim3(kThreads), 0, s, items, nitems, Gtot, K, ld, step, alpha, beta, gamma0,
                           gamma, mode, partials, sizes...);
    };
    auto tiles = [&](auto NG_) {
        constexpr int NG = decltype(NG_)::value;
        if (shape.split) go(k_batched_tiles<T, V, NG, true>, shape.slices, shape.parts);
        else go(k_batched_tiles<T, V, NG, false>, shape.slices, shape.parts);
    };
    auto quads = [&](auto NG_) {
        constexpr int NG = decltype(NG_)::value;
        if (shape.split) go(k_batched_quads<T, V, NG, true>, shape.slices);
        else go(k_batched_quads<T, V, NG, false>, shape.slices);
    };
    if (rows == kRowsTiles) {
        switch (tile_shape(Sc<T>::is_complex, K).NG) {
            case 1: tiles(std::integral_constant<int, 1>{}); break;
            case 2: tiles(std::integral_constant<int, 2>{}); break;
            case 3: tiles(std::integral_constant<int, 3>{}); break;
            case 4: tiles(std::integral_constant<int, 4>{}); break;
            default:
                if constexpr (!Sc<T>::is_complex) tiles(std::integral_constant<int, 6>{});
                else throw Error(VBH_ERR_ARG, "internal: no variable-block kernel for this shape");
        }
    } else if (rows == kRowsQuads) {
        const int NG = quad_shape<T>(K).NG;
        switch (NG) {
            case 1: quads(std::integral_constant<int, 1>{}); break;
            case 2: quads(std::integral_constant<int, 2>{}); break;
            default:
                if constexpr (kQuadMaxGroups<T> == 4) {
                    if (NG == 3) quads(std::integral_constant<int, 3>{});
                    else quads(std::integral_constant<int, 4>{});
                } else {
                    throw Error(VBH_ERR_ARG, "internal: no 4 x 4 block kernel for this shape");
                }
        }
    } else {
        const SmallShape& small = shape.small;
        auto sized = [&](auto NC_) {
            constexpr int NC = decltype(NC_)::value;
            if constexpr (NC * sizeof(T) <= 16) {
                switch (rows - kRowsSmall) {
                    case 0: go(k_batched_smalls<T, V, 1, NC>, small); break;
                    case 1: go(k_batched_smalls<T, V, 2, NC>, small); break;
                    default: go(k_batched_smalls<T, V, 3, NC>, small); break;
                }
            } else {
                throw Error(VBH_ERR_ARG, "internal: no small block kernel for this shape");
            }
        };
        switch (small.NC) {
            case 1: sized(std::integral_constant<int, 1>{}); break;
            case 2: sized(std::integral_constant<int, 2>{}); break;
            default: sized(std::integral_constant<int, 4>{}); break;
        }
    }
    VBH_CHECK_HIP(hipGetLastError());
}

#define VBH_BATCHED_INSTANTIATE(T, V)                                                                             \
    template void launch_batched_rows<T, V>(const BatchItem<T, V>*, int, int, int, int, int, const RowsShape&, int, \
                                            double, double, double, double, int, double*, hipStream_t);

}  // namespace vbh
