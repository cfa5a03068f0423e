// Products of variable blocks with K columns, forward and adjoint, real and
// complex, on the FP64 matrix cores (included by the per-type lanes_*.hip
// units).
//
// One wavefront owns one block row of the output (forward: a block row of A;
// adjoint: a block column) and one slice of the columns; with few block rows the
// 16-row steps of wide blocks go to several waves, and the waves of a work-group
// share a row's blocks and add up through LDS (tile_grid).  The row's blocks are
// cut along the contraction into chunks of at most four consecutive scalar
// columns (adjoint: rows) of one block; the chunks of up to kTileList at a
// time go to a per-wave LDS list (X row, value offset, width).  A lane's A
// operand is the four values of one output row in one chunk, its X operand NG
// or NT consecutive columns of the chunk's four X rows, and instruction m
// contracts element m of several chunks at once: chunks of different blocks
// share an instruction, so a row of narrow blocks wastes only what a chunk's
// last elements leave empty.  Three shapes by the rows r of the output block:
//
//   r <= 4:  v_mfma_f64_4x4x4f64, its four products on different chunks
//            (16 chunks an instruction, merged by two rotations at the end);
//   r <= 8:  the same instruction, two products for the two row quads, two
//            for different chunks (8 chunks);
//   else:    16 rows at a time, four chunks an instruction (blocks over 16 rows
//            in several passes): the same instruction with four row quads for
//            slices of up to 12 columns, v_mfma_f64_16x16x4f64 for wider ones.
//
// Value loads past a chunk's width stay inside the block row (kVecPad elements
// follow the last), those past the list repeat its last chunk, and both enter as
// zeros against X rows of zeros (or_zeros); columns past K overlap earlier
// ones, as in quads.hpp.
// Accumulation is FP64 for every storage type.
//
// What bounds it: the values and the X rows gathered through the L1s, and with
// more than 16 columns the matrix cores.  Measured before / now in us, forward
// and adjoint, 4.5 M FP64 values in blocks of 4-8 (36 MB, 7 us at the copy
// rate): 6 columns 36, 100 / 13, 16; 16 columns 37, 204 / 17, 20; 96 columns 835,
// 1422 / 78, 85; the same in complex128: 6 columns 58, 125 / 22, 26; 64 columns
// 295, 929 / 130, 130.  7.1 M values in blocks of 1, 4, 9, 13: 1 column 41, 48 /
// 20, 24; 16 columns 66, 328 / 31, 32; 96 columns 1768, 2147 / 120, 124.  Before:
// one scalar row a lane, or one 16-row tile a block with a dword of X a lane;
// the adjoint and more than 64 columns one X element a lane at a time.
#pragma once

#include "quads.hpp"

namespace vbh {

constexpr int kTileList = 256;  // chunks in a wave's list (a block of 255 has 64)

struct TileChunk {
    int xrow;       // first X row
    int shape;      // width | block width << 8
    int64_t value;  // offset of its first value
};

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return v;
}
// v of the lane 4 N places on in the 16-lane row (rotating).
template <int N>
__device__ __forceinline__ double row_rotate(double v) {
    union {
        double d;
        int w[2];
    } in{v}, out;
    out.w[0] = __builtin_amdgcn_mov_dpp(in.w[0], 0x120 + 4 * N, 0xf, 0xf, false);
    out.w[1] = __builtin_amdgcn_mov_dpp(in.w[1], 0x120 + 4 * N, 0xf, 0xf, false);
    return out.d;
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Chunk e of a list of nch; past its end the last one, with no columns.
__device__ __forceinline__ TileChunk tile_chunk(const TileChunk* list, int e, int nch) {
    TileChunk ch = list[e < nch ? e : nch - 1];
    if (e >= nch) ch.shape &= ~255;
    return ch;
}

// The four A values of output row `row` in a chunk (zero from its width on).
template <typename V, bool ADJ>
__device__ __forceinline__ void tile_values(const V* __restrict__ vals, const TileChunk& ch, int row, V (&a)[4]) {
    const int w = ch.shape & 255, c = ch.shape >> 8;
    if constexpr (ADJ) {
        const V* p = vals + ch.value + row;
        const int wl = w > 0 ? w - 1 : 0;
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = p[(m < wl ? m : wl) * c];
    } else {
        const RowRun<V, 4> run = *reinterpret_cast<const RowRun<V, 4>*>(vals + ch.value + row * c);
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = run.v[m];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        a[m] = pick(m < w, a[m], Sc<V>::zero());
        if constexpr (ADJ) a[m] = Sc<V>::conj(a[m]);
    }
}
// N columns of the X rows a chunk meets, zeros from its width on: by address, or
// with one column of at most 8 bytes after the load (blocks of 4-8, by address /
// after the load: 500 block rows of 60 blocks, one FP64 column 6.6 / 6.3 us, ten
// FP32 columns adjoint 8.9 / 9.8; 4000 of 40, 64 FP32 columns adjoint 44 / 51).
template <typename T, int N>
__device__ __forceinline__ void tile_columns(const T* __restrict__ xc, int64_t ldx, const TileChunk& ch,
                                             RowRun<T, N> (&x)[4]) {
    const int w = ch.shape & 255;
    const T* x0 = xc + int64_t(ch.xrow) * ldx;
    if constexpr (N == 1 && sizeof(T) <= 8) {
        const int wl = w > 0 ? w - 1 : 0;
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m].v[0] = pick(m < w, x0[(m < wl ? m : wl) * ldx], Sc<T>::zero());
    } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = *reinterpret_cast<const RowRun<T, N>*>(or_zeros(m < w, x0 + m * ldx));
    }
}

// acc += one 16 x 16 x 4 step with N columns per lane.
template <typename T, int N>
struct TileAcc16 {
    vbh_d4 re[N];
    vbh_d4 im[Sc<T>::is_complex ? N : 1];
};
template <typename T, typename V, int N>
__device__ __forceinline__ void tile_mfma16(const V& a, const RowRun<T, N>& x, TileAcc16<T, N>& acc) {
    if constexpr (Sc<T>::is_complex) {
        const double ar = double(a.re), ai = double(a.im);
#pragma unroll
        for (int t = 0; t < N; ++t) {
            const double xr = double(x.v[t].re), xi = double(x.v[t].im);
            acc.re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, xr, acc.re[t], 0, 0, 0);
            acc.im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, xi, acc.im[t], 0, 0, 0);
            acc.re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, xi, acc.re[t], 0, 0, 0);
            acc.im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, xr, acc.im[t], 0, 0, 0);
        }
    } else {
        const double ad = double(a);
#pragma unroll
        for (int t = 0; t < N; ++t)
            acc.re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ad, double(x.v[t]), acc.re[t], 0, 0, 0);
    }
}

// The blocks of one output block row: slots [kb, ke), forward from meta (row
// values from vrow, r rows), adjoint from the plan (width c of the block
// column).
struct TileRow {
    int kb, ke, size;
    int64_t vrow, out;
};

// Runs steps(nch) for every list of the row's chunks in `list`.
template <bool ADJ, typename F>
__device__ __forceinline__ void tile_lists(const DevPattern& p, const AdjointPlan& ap, const TileRow& row, int lane,
                                           TileChunk* list, F&& steps) {
    for (int t0 = row.kb; t0 < row.ke; t0 += 64) {
        const int nb = row.ke - t0 < 64 ? row.ke - t0 : 64;
        const int slot = t0 + (lane < nb ? lane : nb - 1);
        int x0, width, stride;
        int64_t v0;
        if constexpr (ADJ) {
            const int2 rr = ap.t_rows[slot];
            x0 = rr.x;
            width = rr.y;
            stride = row.size;
            v0 = ap.t_voff[slot];
        } else {
            const int2 mm = p.meta[slot];
            x0 = mm.x;
            width = mm.y & 255;
            stride = width;
            v0 = row.vrow + int64_t(row.size) * (mm.y >> 8);
        }
        const int mine = lane < nb ? (width + 3) >> 2 : 0;
        const int upto = wave_scan(mine);
        int done = 0;
        for (int u0 = 0; u0 < nb;) {
            const bool fits = lane >= u0 && lane < nb && upto - done <= kTileList;
            const int u1 = u0 + __popcll(__ballot(fits));
            if (fits) {
                const int at = upto - mine - done;
                for (int t = 0; t < mine; ++t) {
                    const int w = width - 4 * t < 4 ? width - 4 * t : 4;
                    list[at + t] = TileChunk{x0 + 4 * t, w | stride << 8, v0 + int64_t(ADJ ? stride : 1) * (4 * t)};
                }
            }
            const int upto1 = __builtin_amdgcn_readlane(upto, u1 - 1);
            wave_lds_sync();
            steps(upto1 - done);
            wave_lds_sync();
            done = upto1;
            u0 = u1;
        }
    }
}

// The sum over the chunk partitions of an instruction with nq row quads.
__device__ __forceinline__ void tile_merge(double& v, int nq) {
    const double a = v + row_rotate<2>(v);
    v = nq < 4 ? a : v;
    const double b = v + row_rotate<1>(v);
    v = nq < 2 ? b : v;
}
// Narrow slices keep the 4 x 4 x 4 instruction for 16 rows (four row quads):
// 64 NG cycles for four chunks against 256 of the 16 x 16 x 4 one.
template <int NG>
constexpr bool kTileQuads16 = NG <= 3;

// LDS of one wave: its chunk list, and between two lists the sums it hands over.
union TileArea {
    TileChunk list[kTileList];
    double sums[kTileList * 2];
};
template <typename T, int N>
__device__ __forceinline__ void sums_store(double* at, const TileAcc16<T, N>& a) {
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            at[64 * (4 * t + e)] = a.re[t][e];
            if constexpr (Sc<T>::is_complex) at[64 * (4 * (N + t) + e)] = a.im[t][e];
        }
}
template <typename T, int N>
__device__ __forceinline__ void sums_add(const double* at, TileAcc16<T, N>& a) {
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a.re[t][e] += at[64 * (4 * t + e)];
            if constexpr (Sc<T>::is_complex) a.im[t][e] += at[64 * (4 * (N + t) + e)];
        }
}
// acc of wave 0 += those of the work-group's other waves, in their order.
template <int VALUES, typename A>
__device__ __forceinline__ void waves_sum(TileArea* areas, int wave, int lane, A& acc) {
    static_assert(64 * VALUES * sizeof(double) <= sizeof(TileArea), "a lane's values fit the areas");
    if (wave > 0) sums_store(areas[wave].sums + lane, acc);
    __syncthreads();
    if (wave == 0)
#pragma unroll
        for (int w = 1; w < kWaves; ++w) sums_add(areas[w].sums + lane, acc);
    __syncthreads();
}

// The work of one wave: output block row unit / (slices x parts), its 16-row
// steps part, part + parts, .., and slice unit % slices.  SPLIT: of one
// work-group, whose waves share the row's blocks.
template <typename T, typename V, int NG, bool ADJ, bool DOT, bool ACC, bool SPLIT = false>
__device__ __forceinline__ void tile_wave(const ApplyArgs<T, V>& g, const AdjointPlan& ap, int slices, int parts,
                                          const SeriesAcc<T>& sa, TileArea* areas, int wave, int unit, int lane,
                                          double& d1, double& d2) {
    constexpr int E = Sc<T>::is_complex ? 2 : 1;
    const DevPattern& p = g.p;
    TileChunk* list = areas[wave].list;
    int ob = unit / slices;  // output block row
    const int v0 = (unit - ob * slices) * 4 * NG;
    int first_row = 0;
    if (parts > 1) {
        const int row_part = ob;
        ob = row_part / parts;
        first_row = 16 * (row_part - ob * parts);
    }
    const int row_step = 16 * parts;
    if (ob < (ADJ ? p.nbc : p.nbr)) {
        TileRow row;
        if constexpr (ADJ) {
            row = TileRow{ap.t_ptr[ob], ap.t_ptr[ob + 1], p.cbs[ob], 0, p.coff[ob]};
        } else {
            row = TileRow{p.row_ptr[ob], p.row_ptr[ob + 1], p.rbs[ob], 0, p.roff[ob]};
            row.vrow = p.voff[row.kb];
        }
        row.kb = __builtin_amdgcn_readfirstlane(row.kb);
        row.ke = __builtin_amdgcn_readfirstlane(row.ke);
        row.size = __builtin_amdgcn_readfirstlane(row.size);
        if constexpr (SPLIT) {
            const int kb = row.kb, len = row.ke - kb;
            row.kb = kb + int(int64_t(len) * wave / kWaves);
            row.ke = kb + int(int64_t(len) * (wave + 1) / kWaves);
        }
        const int64_t xown = ADJ ? row.out : ob < p.nbc ? int64_t(p.coff[ob]) : 0;
        const int li = lane & 3, lb = (lane >> 2) & 3, lk = lane >> 4;
        if (kTileQuads16<NG> || row.size <= 8) {
            const int nq = row.size <= 4 ? 1 : row.size <= 8 ? 2 : 4;  // row quads an instruction
            const int cb = v0 + NG * li;
            const int c0 = cb < g.K - NG ? cb : g.K - NG;
            const int skip = cb - c0 < NG ? cb - c0 : NG;
            const int quad = lb & (nq - 1);
            const int first = (nq == 1 ? lb : nq == 2 ? lb >> 1 : 0) * 4 + lk, per = 16 / nq;
            const T* xc = g.X + c0;
            for (int r0 = first_row; r0 < row.size; r0 += row_step) {
                const int ar = r0 + 4 * quad + li < row.size ? r0 + 4 * quad + li : row.size - 1;
                QuadAcc<T, NG> acc[2] = {};
                tile_lists<ADJ>(p, ap, row, lane, list, [&](int nch) {
                    // steps in flight
                    constexpr int U = NG * sizeof(T) <= 16 ? 2 : 1;
                    for (int e0 = 0; e0 < nch; e0 += U * per) {
                        V a[U][4];
                        RowRun<T, NG> x[U][4];
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const int e = e0 + u * per + first;
                            const TileChunk ch = tile_chunk(list, e, nch);
                            tile_values<V, ADJ>(g.vals, ch, ar, a[u]);
                            tile_columns<T, NG>(xc, g.ldx, ch, x[u]);
                        }
#pragma unroll
                        for (int u = 0; u < U; ++u)
#pragma unroll
                            for (int m = 0; m < 4; ++m) quad_mfma<T, V, NG>(a[u][m], x[u][m], acc[m & 1]);
                    }
                });
                quad_sum<T, NG>(acc[0], acc[1]);
#pragma unroll
                for (int t = 0; t < NG; ++t) {
                    tile_merge(acc[0].re[t], nq);
                    if constexpr (Sc<T>::is_complex) tile_merge(acc[0].im[t], nq);
                }
                if constexpr (SPLIT) {
                    waves_sum<NG * E>(areas, wave, lane, acc[0]);
                    if (wave > 0) continue;
                }
                const int yrow = r0 + 4 * quad + lk;
                if (lb < nq && yrow < row.size)
                    quad_emit<T, V, NG, DOT, ACC, ADJ>(g, row.out + yrow, xown + yrow, c0, skip, acc[0], d1, d2, sa);
            }
        } else if constexpr (!kTileQuads16<NG>) {
            constexpr int NT = (NG + 3) / 4;
            const int l16 = lane & 15;
            const int lc = NT * l16 < 4 * NG ? l16 : 0;  // lanes past a narrow slice repeat its first columns
            const int cb = v0 + NT * lc;
            const int c0 = cb < g.K - NT ? cb : g.K - NT;
            const int skip = lc != l16 ? NT : cb - c0 < NT ? cb - c0 : NT;
            const T* xc = g.X + c0;
            for (int r0 = first_row; r0 < row.size; r0 += row_step) {
                const int ar = r0 + l16 < row.size ? r0 + l16 : row.size - 1;
                TileAcc16<T, NT> acc = {};
                tile_lists<ADJ>(p, ap, row, lane, list, [&](int nch) {
                    for (int e0 = 0; e0 < nch; e0 += 8) {
                        V a[2][4];
                        RowRun<T, NT> x[2][4];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const int e = e0 + 4 * u + lk;
                            const TileChunk ch = tile_chunk(list, e, nch);
                            tile_values<V, ADJ>(g.vals, ch, ar, a[u]);
                            tile_columns<T, NT>(xc, g.ldx, ch, x[u]);
                        }
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            if (e0 + 4 * u >= nch) break;
#pragma unroll
                            for (int m = 0; m < 4; ++m) tile_mfma16<T, V, NT>(a[u][m], x[u][m], acc);
                        }
                    }
                });
                if constexpr (SPLIT) {
                    waves_sum<4 * NT * E>(areas, wave, lane, acc);
                    if (wave > 0) continue;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int yrow = r0 + 4 * e + lk;
                    QuadAcc<T, NT> s;
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        s.re[t] = acc.re[t][e];
                        if constexpr (Sc<T>::is_complex) s.im[t] = acc.im[t][e];
                    }
                    if (yrow < row.size)
                        quad_emit<T, V, NT, DOT, ACC, ADJ>(g, row.out + yrow, xown + yrow, c0, skip, s, d1, d2, sa);
                }
            }
        }
    }
}

template <typename T, typename V, int NG, bool ADJ, bool DOT, bool ACC, bool SPLIT>
__global__ __launch_bounds__(kThreads) void k_apply_tiles(ApplyArgs<T, V> g, AdjointPlan ap, int slices, int parts,
                                                          SeriesAcc<T> sa) {
    __shared__ TileArea areas[kWaves];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int chunk = xcd_chunk(g.G);
    const int unit = SPLIT ? chunk : chunk * kWaves + wave;
    double d1 = 0.0, d2 = 0.0;
    tile_wave<T, V, NG, ADJ, DOT, ACC, SPLIT>(g, ap, slices, parts, sa, areas, wave, unit, lane, d1, d2);
    if constexpr (DOT) write_dots(lane, wave, d1, d2, g.partials + int64_t(chunk) * 2);
}

template <typename T, typename V, bool ADJ, bool DOT, bool ACC>
static void launch_tiles_as(const ApplyArgs<T, V>& a, const AdjointPlan& ap, const TileGrid& q, const SeriesAcc<T>& sa,
                            hipStream_t s) {
    ApplyArgs<T, V> b = a;
    b.G = q.G;
    const dim3 grid(q.G), block(kThreads);
    auto go = [&](auto NG_) {
        constexpr int NG = decltype(NG_)::value;
        if (q.split)
            hipLaunchKernelGGL((k_apply_tiles<T, V, NG, ADJ, DOT, ACC, true>), grid, block, 0, s, b, ap, q.S, q.parts, sa);
        else
            hipLaunchKernelGGL((k_apply_tiles<T, V, NG, ADJ, DOT, ACC, false>), grid, block, 0, s, b, ap, q.S, q.parts, sa);
    };
    switch (q.NG) {
        case 1: go(std::integral_constant<int, 1>{}); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        default:
            if constexpr (!Sc<T>::is_complex) go(std::integral_constant<int, 6>{});
            else throw Error(VBH_ERR_ARG, "internal: no variable-block kernel for this shape");
    }
    VBH_CHECK_HIP(hipGetLastError());
}

template <typename T, typename V>
void launch_tiles(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>* sa, hipStream_t s) {
    const TileGrid q = tile_grid<T>(RowStats(m, m->nbr), a.K);
    if (a.partials) launch_tiles_as<T, V, false, true, false>(a, AdjointPlan{}, q, SeriesAcc<T>{}, s);
    else if (sa) launch_tiles_as<T, V, false, false, true>(a, AdjointPlan{}, q, *sa, s);
    else launch_tiles_as<T, V, false, false, false>(a, AdjointPlan{}, q, SeriesAcc<T>{}, s);
}
template <typename T>
void launch_tiles_adjoint(const vbh_matrix* m, const ApplyArgs<T, T>& a, const AdjointPlan& ap, const SeriesAcc<T>* term,
                          hipStream_t s) {
    const TileGrid q = tile_grid<T>(RowStats(m, m->nbc), a.K);
    if (term) launch_tiles_as<T, T, true, false, true>(a, ap, q, *term, s);
    else launch_tiles_as<T, T, true, false, false>(a, ap, q, SeriesAcc<T>{}, s);
}

#define VBH_TILES_INSTANTIATE(T, V) \
    template void launch_tiles<T, V>(const vbh_matrix*, const ApplyArgs<T, V>&, const SeriesAcc<T>*, hipStream_t);
#define VBH_TILES_ADJOINT_INSTANTIATE(T) \
    template void launch_tiles_adjoint<T>(const vbh_matrix*, const ApplyArgs<T, T>&, const AdjointPlan&, const SeriesAcc<T>*, \
                                          hipStream_t);

}  // namespace vbh
