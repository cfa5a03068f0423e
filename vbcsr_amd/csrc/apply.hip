// Block SpMV / SpMM and their adjoints on gfx950.
//
// Dispatch (launch_rows, apply_adjoint): uniform blocks of size 1 to 3 run in
// smalls.hpp, uniform 4 x 4 blocks with several columns in quads.hpp, one column
// of them and its adjoint in quad_spmv.hpp, other blocks, wide columns and every
// other adjoint in tiles.hpp, calls with per-column dots in the row loop below.
// One column of blocks up to 8 x 8 runs in the LDS SpMV below (row_loop_spmv)
// where neither smalls.hpp (from kManyRows block rows on) nor tiles.hpp (differing
// sizes in long rows within the memory-side cache: one_column_tiles) takes it.
// Every Y element is written exactly once -- no atomics, no Y zero pass.
// Work-groups are remapped so that each XCD streams one contiguous run of
// rows and keeps the X rows it gathers in its own L2.
//
// The optional fused epilogue computes Y = alpha*AX + beta*X_own + gamma*Z and
// FP64 partial dot products of Y with W (or Y) and with X_own, one partial per
// work-group, written (not accumulated) into the partials array.
#include "apply.hpp"

namespace vbh {

template <typename T, int BS, int RB>
__global__ __launch_bounds__(kThreads) void k_apply_rows(ApplyArgs<T> g) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(g.G);
    double d1 = 0.0, d2 = 0.0;
    row_loop<T, BS, RB>(g, g.split[chunk], g.split[chunk + 1], lane, wave, d1, d2);
    if (g.partials != nullptr) {
        const int E = g.dot_cols > 1 ? g.K : 1;
        write_partials(E, lane, wave, d1, d2, g.partials + int64_t(chunk) * 2 * E);
    }
}

template <typename T, int RPP, bool FUSED>
__global__ __launch_bounds__(kThreads) void k_apply_spmv(ApplyArgs<T> g) {
    __shared__ __attribute__((aligned(16))) T tile[kWaves][kSpmvTile(RPP)];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(g.G);
    double d1 = 0.0, d2 = 0.0;
    row_loop_spmv<T, RPP, FUSED>(g, g.split[chunk], g.split[chunk + 1], lane, wave, d1, d2, tile[wave]);
    if constexpr (FUSED) {
        if (g.partials != nullptr) write_dots(lane, wave, d1, d2, g.partials + int64_t(chunk) * 2);
    }
}

// The fused SpMV step with the series accumulation (no dots).
template <typename T, int RPP>
__global__ __launch_bounds__(kThreads) void k_apply_spmv_series(ApplyArgs<T> g, SeriesAcc<T> sa) {
    __shared__ __attribute__((aligned(16))) T tile[kWaves][kSpmvTile(RPP)];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(g.G);
    double d1 = 0.0, d2 = 0.0;
    row_loop_spmv<T, RPP, true, true>(g, g.split[chunk], g.split[chunk + 1], lane, wave, d1, d2, tile[wave], &sa);
}

RowConfig row_config(int K, int max_block, int uniform_bs) {
    RowConfig c{0, 0, 1};
    if (K == 1 && max_block <= 8) {
        c.spmv_rpp = pow2ceil(max_block);
        return c;
    }
    c.bs = uniform_bs == 4 ? 4 : 0;
    const int Kp = K >= 64 ? 64 : pow2ceil(K);
    const int NG = 64 / Kp;
    const int need = (max_block + NG - 1) / NG;
    c.rb = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : 8;
    return c;
}

// Sum per-work-group partials: out[e] (+)= sum_g partials[g][e], e < E.
__global__ void k_reduce_partials(const double* __restrict__ partials, int G, int E, double* __restrict__ out,
                                  int accumulate) {
    const int e = blockIdx.x;
    double s = 0.0;
    for (int gg = threadIdx.x; gg < G; gg += blockDim.x) s += partials[int64_t(gg) * E + e];
    __shared__ double red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int m = 128; m >= 1; m >>= 1) {
        if (threadIdx.x < m) red[threadIdx.x] += red[threadIdx.x + m];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[e] = accumulate ? out[e] + red[0] : red[0];
}

template <typename T, int BS>
static void launch_spmm_family(int rb, const ApplyArgs<T>& a, hipStream_t s) {
    const dim3 grid(a.G), block(kThreads);
    switch (rb) {
        case 1: hipLaunchKernelGGL((k_apply_rows<T, BS, 1>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((k_apply_rows<T, BS, 2>), grid, block, 0, s, a); break;
        case 4: hipLaunchKernelGGL((k_apply_rows<T, BS, 4>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((k_apply_rows<T, BS, 8>), grid, block, 0, s, a); break;
    }
}

template <typename T, bool FUSED>
static void launch_single(const vbh_matrix* m, const ApplyArgs<T>& a, hipStream_t s);

template <typename T, bool FUSED, typename V>
void launch_rows(const vbh_matrix* m, const ApplyArgs<T, V>& a, hipStream_t s) {
    if (uses_quads(m, a)) {
        launch_quads<T, V>(m, a, nullptr, s);
        return;
    }
    if (uses_smalls(m, a)) {
        launch_smalls<T, V>(m, a, nullptr, s);
        return;
    }
    if (uses_tiles(m, a)) {
        launch_tiles<T, V>(m, a, nullptr, s);
        return;
    }
    if constexpr (is_mixed<T, V>()) {
        throw Error(VBH_ERR_NOTSUP,
                    "precision 2 (FP32 values, native vectors) supports 1 <= K <= 64 and column-summed dots only");
    } else if (uses_quad_spmv(m, a)) {
        launch_quad_spmv<T>(m, a, FUSED, nullptr, s);
    } else {
        launch_single<T, FUSED>(m, a, s);
    }
}

// The LDS SpMV (K = 1, blocks up to 8), and the row loop with per-column dots.
template <typename T, bool FUSED>
static void launch_single(const vbh_matrix* m, const ApplyArgs<T>& a, hipStream_t s) {
    const RowConfig c = row_config(a.K, m->max_block, m->uniform_bs);
    const dim3 grid(a.G), block(kThreads);
    if (c.spmv_rpp > 0) {
        switch (c.spmv_rpp) {
            case 1: hipLaunchKernelGGL((k_apply_spmv<T, 1, FUSED>), grid, block, 0, s, a); break;
            case 2: hipLaunchKernelGGL((k_apply_spmv<T, 2, FUSED>), grid, block, 0, s, a); break;
            case 4: hipLaunchKernelGGL((k_apply_spmv<T, 4, FUSED>), grid, block, 0, s, a); break;
            default: hipLaunchKernelGGL((k_apply_spmv<T, 8, FUSED>), grid, block, 0, s, a); break;
        }
    } else if constexpr (FUSED) {
        if (c.bs == 4) launch_spmm_family<T, 4>(c.rb, a, s);
        else launch_spmm_family<T, 0>(c.rb, a, s);
    } else {
        throw Error(VBH_ERR_ARG, "internal: no kernel for this product");
    }
    VBH_CHECK_HIP(hipGetLastError());
}

template <typename T, typename V>
bool launch_series(const vbh_matrix* m, const ApplyArgs<T, V>& a, const SeriesAcc<T>& sa, hipStream_t s) {
    if (a.partials != nullptr) return false;
    if (uses_quads(m, a)) {
        launch_quads<T, V>(m, a, &sa, s);
        return true;
    }
    if (uses_smalls(m, a)) {
        launch_smalls<T, V>(m, a, &sa, s);
        return true;
    }
    if (uses_tiles(m, a)) {
        launch_tiles<T, V>(m, a, &sa, s);
        return true;
    }
    if constexpr (is_mixed<T, V>()) {
        return false;
    } else {
        if (uses_quad_spmv(m, a)) {
            launch_quad_spmv<T>(m, a, true, &sa, s);
            return true;
        }
        const RowConfig c = row_config(a.K, m->max_block, m->uniform_bs);
        if (c.spmv_rpp <= 0) return false;
        const dim3 grid(a.G), block(kThreads);
        switch (c.spmv_rpp) {
            case 1: hipLaunchKernelGGL((k_apply_spmv_series<T, 1>), grid, block, 0, s, a, sa); break;
            case 2: hipLaunchKernelGGL((k_apply_spmv_series<T, 2>), grid, block, 0, s, a, sa); break;
            case 4: hipLaunchKernelGGL((k_apply_spmv_series<T, 4>), grid, block, 0, s, a, sa); break;
            default: hipLaunchKernelGGL((k_apply_spmv_series<T, 8>), grid, block, 0, s, a, sa); break;
        }
        VBH_CHECK_HIP(hipGetLastError());
        return true;
    }
}

template <typename T, typename V>
ApplyArgs<T, V> make_args(const vbh_matrix* m, const V* vals, int K, const T* X, int64_t ldx, T* Y, int64_t ldy) {
    m->applied = true;
    ApplyArgs<T, V> a{};
    a.p = m->pattern();
    a.parts = 1;
    a.vals = vals;
    a.K = K;
    a.X = X;
    a.ldx = ldx;
    a.Y = Y;
    a.ldy = ldy;
    a.alpha = 1.0;
    a.split = m->split;
    a.G = m->G;
    return a;
}

template <typename T, typename V>
void apply_plain(vbh_matrix* m, const V* vals, int K, const void* X, int64_t ldx, void* Y, int64_t ldy, hipStream_t s) {
    if (m->nbr == 0 || K == 0) return;
    auto a = make_args<T, V>(m, vals, K, (const T*)X, ldx, (T*)Y, ldy);
    launch_rows<T, false, V>(m, a, s);
}

template <typename T>
void apply_adjoint(vbh_matrix* m, const T* vals, int K, const void* X, int64_t ldx, void* Y, int64_t ldy,
                   hipStream_t s, const AdjointStep<T>* step) {
    if (m->nbc == 0 || K == 0) return;
    ensure_adjoint_plan(m, s);
    ApplyArgs<T> a{};
    a.p = m->pattern();
    a.vals = vals;
    a.K = K;
    a.X = (const T*)X;
    a.ldx = ldx;
    a.Y = (T*)Y;
    a.ldy = ldy;
    a.alpha = 1.0;
    if (step) {
        a.alpha = step->alpha;
        a.beta = step->beta;
        a.gamma = step->Z ? -1.0 : 0.0;
        a.Z = step->Z;
        a.ldz = step->ldz;
    }
    const SeriesAcc<T>* term = step ? &step->term : nullptr;
    const AdjointPlan plan{m->t_ptr, m->t_voff, m->t_rows};
    if (uses_quad_spmv(m, a)) {
        launch_quad_spmv_adjoint<T>(m, a, plan, term, s);
        return;
    }
    if (small_blocks(m)) {
        launch_smalls_adjoint<T>(m, a, plan, term, s);
        return;
    }
    launch_tiles_adjoint<T>(m, a, plan, term, s);
}

void reduce_partials(const double* partials, int G, int E, double* out, bool accumulate, hipStream_t s) {
    hipLaunchKernelGGL(k_reduce_partials, dim3(E), dim3(256), 0, s, partials, G, E, out, accumulate ? 1 : 0);
    VBH_CHECK_HIP(hipGetLastError());
}

template <typename T>
const T* compute_values(vbh_matrix* m, hipStream_t s) {
    if constexpr (std::is_same_v<T, float> || std::is_same_v<T, c64>) {
        ensure_vals32(m, s);
        return (const T*)m->vals32;
    } else {
        return (const T*)m->vals;
    }
}

// explicit instantiations used by kpm.hip
#define VBH_INST2(T, V)                                                                                          \
    template void launch_rows<T, true, V>(const vbh_matrix*, const ApplyArgs<T, V>&, hipStream_t);              \
    template void launch_rows<T, false, V>(const vbh_matrix*, const ApplyArgs<T, V>&, hipStream_t);             \
    template ApplyArgs<T, V> make_args<T, V>(const vbh_matrix*, const V*, int, const T*, int64_t, T*, int64_t); \
    template void apply_plain<T, V>(vbh_matrix*, const V*, int, const void*, int64_t, void*, int64_t, hipStream_t); \
    template bool launch_series<T, V>(const vbh_matrix*, const ApplyArgs<T, V>&, const SeriesAcc<T>&, hipStream_t);
#define VBH_INST(T)                                                          \
    VBH_INST2(T, T)                                                          \
    template const T* compute_values<T>(vbh_matrix*, hipStream_t);          \
    template void apply_adjoint<T>(vbh_matrix*, const T*, int, const void*, int64_t, void*, int64_t, hipStream_t, \
                                   const AdjointStep<T>*);
VBH_INST(double)
VBH_INST(float)
VBH_INST(c128)
VBH_INST(c64)
VBH_INST2(double, float)
VBH_INST2(c128, c64)
#undef VBH_INST
#undef VBH_INST2

}  // namespace vbh

using namespace vbh;

extern "C" {

VBH_API int vbh_spmm(vbh_matrix_t m, int K, const void* X, int ldx, void* Y, int ldy, int precision, void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m, "null matrix");
        VBH_REQUIRE(K >= 0 && ldx >= K && ldy >= K, "leading dimensions must be >= K");
        hipStream_t s = (hipStream_t)stream;
        dispatch_compute(m, precision, [&](auto* tag, auto* vtag) {
            using T = std::remove_pointer_t<decltype(tag)>;
            using V = std::remove_pointer_t<decltype(vtag)>;
            apply_plain<T, V>(m, compute_values<V>(m, s), K, X, ldx, Y, ldy, s);
        });
    });
}

VBH_API int vbh_spmv(vbh_matrix_t m, const void* x, void* y, int precision, void* stream) {
    return vbh_spmm(m, 1, x, 1, y, 1, precision, stream);
}

VBH_API int vbh_spmm_adjoint(vbh_matrix_t m, int K, const void* X, int ldx, void* Y, int ldy, int precision,
                             void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m, "null matrix");
        VBH_REQUIRE(K >= 0 && ldx >= K && ldy >= K, "leading dimensions must be >= K");
        hipStream_t s = (hipStream_t)stream;
        VBH_REQUIRE(precision != 2, "the adjoint supports precision 0 and 1");
        dispatch_compute(m, precision, [&](auto* tag, auto*) {
            using T = std::remove_pointer_t<decltype(tag)>;
            apply_adjoint<T>(m, compute_values<T>(m, s), K, X, ldx, Y, ldy, s);
        });
    });
}

VBH_API int vbh_spmv_adjoint(vbh_matrix_t m, const void* x, void* y, int precision, void* stream) {
    return vbh_spmm_adjoint(m, 1, x, 1, y, 1, precision, stream);
}

VBH_API int vbh_spmm_fused(vbh_matrix_t m, int K, const void* X, int ldx, void* Y, int ldy, double alpha,
                           double beta, double gamma, const void* Z, int ldz, const void* W, int ldw, double* dots,
                           int precision, void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m, "null matrix");
        VBH_REQUIRE(K >= 0 && ldx >= K && ldy >= K, "leading dimensions must be >= K");
        VBH_REQUIRE(gamma == 0.0 || (Z && ldz >= K), "gamma != 0 needs Z with ldz >= K");
        VBH_REQUIRE(!W || ldw >= K, "ldw must be >= K");
        VBH_REQUIRE(!dots || K <= 64, "fused dot products support K <= 64");
        // the epilogue reads X at the owned rows (column i of row i): needs nbc >= nbr
        VBH_REQUIRE(m->nbc >= m->nbr, "fused apply needs the owned columns of a square pattern");
        if (m->nbr == 0 || K == 0) return;
        hipStream_t s = (hipStream_t)stream;
        VBH_REQUIRE(precision != 2 || !dots, "per-column dots support precision 0 and 1");
        dispatch_compute(m, precision, [&](auto* tag, auto* vtag) {
            using T = std::remove_pointer_t<decltype(tag)>;
            using V = std::remove_pointer_t<decltype(vtag)>;
            auto a = make_args<T, V>(m, compute_values<V>(m, s), K, (const T*)X, ldx, (T*)Y, ldy);
            a.alpha = alpha;
            a.beta = beta;
            a.gamma = gamma;
            a.Z = (const T*)Z;
            a.ldz = ldz;
            a.W = (const T*)W;
            a.ldw = ldw;
            a.dot_cols = dots ? K : 0;
            const int G = apply_groups(m, a);
            double* part = nullptr;
            if (dots) part = (double*)scratch(sizeof(double) * 2 * K * G, 2);
            a.partials = part;
            launch_rows<T, true, V>(m, a, s);
            if (dots) reduce_partials(part, G, 2 * K, dots, true, s);
        });
    });
}

}  // extern "C"
