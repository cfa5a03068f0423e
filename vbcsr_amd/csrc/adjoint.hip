// Adjoint of the Chebyshev propagation on gfx950: the stored Chebyshev basis,
// the Clenshaw recurrence with the adjoint operator, and the block-sampled
// outer-product sum (SDDMM) that turns both into the gradient with respect to
// the stored block values.
//
// Forward (examples/ex09_graphene_dynamics.py:102-133, vbcsr/utils.py:71-126):
//   t_0 = x, t_1 = H~ t_0, t_{n+1} = 2 H~ t_n - t_{n-1},  y = sum_n c_n t_n,
//   H~ = (H - center) / half_width.
// Reverse mode, for a real loss L and the gradient convention g_v = dL/dRe v +
// i dL/dIm v (torch's): with lambda = g_y,
//   b_n = conj(c_n) lambda + 2 H~^H b_{n+1} - b_{n+2}   (n >= 1, b_N = b_{N+1} = 0)
//   g_x = b_0 = conj(c_0) lambda + H~^H b_1 - b_2
//   g_{H~} = b_1 t_0^H + 2 sum_{n>=2} b_n t_{n-1}^H,   g_H = g_{H~} / half_width,
// restricted to the stored blocks (the pattern is fixed).  The basis t_n and
// the b_n are arrays of nterms terms of n_rows x K entries.  Term by term (every
// term contiguous) each step of the recurrences gathers and writes dense
// vectors; as column blocks of one row-major array every x entry of a step is a
// cache line of its own (complex128 SpMV steps on 80,000 rows, 64 terms: 21.4
// us as column blocks, 18.9 us on dense vectors).
#include <algorithm>
#include <cstring>

#include "apply.hpp"

namespace vbh {

template <typename T>
__global__ void k_copy_rows(int64_t rows, int K, const T* __restrict__ in, int64_t ldi, T* __restrict__ out,
                            int64_t ldo) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= rows * K) return;
    const int64_t r = e / K;
    const int v = int(e - r * K);
    out[r * ldo + v] = in[r * ldi + v];
}

// bn = c lam over rows x K entries (the last cotangent).
template <typename T>
__global__ void k_scale_rows(int64_t rows, int K, T* __restrict__ bn, int64_t ldb, const T* __restrict__ lam,
                             int64_t ldl, double cre, double cim) {
    using A = typename Wide<T>::type;
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= rows * K) return;
    const int64_t r = e / K;
    const int v = int(e - r * K);
    bn[r * ldb + v] = narrow_to<T>(Sc<A>::make(cre, cim) * widen(lam[r * ldl + v]));
}

// One factor of the outer-product sum: Q = nterms * K vectors of row entries,
// entry q = n * K + v of row i at at[n * term + i * ld + v].
template <typename T>
struct Factors {
    const T* at;
    int64_t term, ld;
    __device__ __forceinline__ int64_t place(int q, int K) const {
        const int n = K == 1 ? q : q / K;
        return int64_t(n) * term + (q - n * K);
    }
};

// G_blk(a,b) += alpha * sum_{q<Q} w_q U[row_a][q] conj(V[col_b][q]) for every
// stored block, w_q = w0 for the first term (q < K) and 1 otherwise; lanes take
// consecutive entries of a block row's contiguous value run.  G is in the
// matrix's own type (FP64 accumulation).
template <typename T, typename G_t>
__global__ __launch_bounds__(kThreads) void k_sddmm(DevPattern p, int K, int Q, Factors<T> u, Factors<T> v, double w0,
                                                    double are, double aim, G_t* __restrict__ Gv,
                                                    const int* __restrict__ split, int Gn) {
    using A = typename Wide<T>::type;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int chunk = xcd_chunk(Gn);
    const A alpha = Sc<A>::make(are, aim);
    for (int i = split[chunk] + wave; i < split[chunk + 1]; i += kWaves) {
        const int r = p.rbs[i];
        const int kb = p.row_ptr[i], ke = p.row_ptr[i + 1];
        if (kb == ke) continue;
        const int64_t v0 = p.voff[kb];
        const int64_t len = p.voff[ke] - v0;
        const int64_t row0 = p.roff[i];
        for (int64_t e = lane; e < len; e += 64) {
            // slot of value e: the last whose panel starts at or before it
            int lo = kb, hi = ke - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (int64_t(r) * (p.meta[mid].y >> 8) <= e) lo = mid;
                else hi = mid - 1;
            }
            const int2 mm = p.meta[lo];
            const int c = mm.y & 255;
            const int in = int(e - int64_t(r) * (mm.y >> 8));
            const int a = in / c, b = in - a * c;
            const T* ur = u.at + (row0 + a) * u.ld;
            const T* vr = v.at + (int64_t(mm.x) + b) * v.ld;
            A first = Sc<A>::zero(), acc = Sc<A>::zero();
#pragma unroll 4
            for (int q = 0; q < K; ++q) first = Sc<A>::fma(widen(ur[q]), widen(Sc<T>::conj(vr[q])), first);
#pragma unroll 8
            for (int q = K; q < Q; ++q)
                acc = Sc<A>::fma(widen(ur[u.place(q, K)]), widen(Sc<T>::conj(vr[v.place(q, K)])), acc);
            const A g = (acc + rscale(w0, first)) * alpha;
            if constexpr (Sc<G_t>::is_complex) {
                Gv[v0 + e] = Gv[v0 + e] + G_t{g.re, g.im};
            } else {
                Gv[v0 + e] += Sc<A>::re(g);
            }
        }
    }
}

// The same for uniform 4 x 4 blocks on the matrix cores: one wavefront per
// block row; product b of v_mfma_f64_4x4x4f64 is slot 4 u + b of the row, an
// instruction contracts four of the Q entries, and its result is the slot's
// 4 x 4 gradient block.  The block row's U entries of 64 q stay in registers
// for all its slots.  Bound by the loads of V (16 bytes a lane in complex128);
// 64 terms of one complex128 column, 200,000 blocks: 530 us with one value a
// lane and a serial sum, 142 us here.
template <typename T, typename G_t>
__global__ __launch_bounds__(kThreads) void k_sddmm_quads(DevPattern p, int K, int Q, Factors<T> u, Factors<T> v,
                                                          double w0, double are, double aim, G_t* __restrict__ Gv,
                                                          int Gn) {
    using A = typename Wide<T>::type;
    constexpr int QS = 16;  // contraction steps of four q per register set
    // U in registers: real entries widened, so that the first term's weight is
    // applied in FP64 as they are loaded; FP32 complex ones (whose registers would
    // be too many) take it after they are widened, steps past that term skipping it
    using UT = std::conditional_t<Sc<T>::is_complex, T, A>;
    constexpr bool late = !std::is_same_v<UT, A>;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int i = xcd_chunk(Gn) * kWaves + __builtin_amdgcn_readfirstlane(wave);
    if (i >= p.nbr) return;
    const int li = lane & 3, lb = (lane >> 2) & 3, lk = lane >> 4;
    const int kb = p.row_ptr[i], ke = p.row_ptr[i + 1];
    const A alpha = Sc<A>::make(are, aim);
    for (int q0 = 0; q0 < Q; q0 += 4 * QS) {
        const int nq = Q - q0 < 4 * QS ? Q - q0 : 4 * QS;
        UT uv[QS];
#pragma unroll
        for (int st = 0; st < QS; ++st) {
            const int q = q0 + 4 * st + lk;
            const int qc = q < Q ? q : Q - 1;
            uv[st] = Sc<UT>::zero();
            if (4 * st >= nq) continue;
            const UT x = UT(u.at[(int64_t(i) * 4 + li) * u.ld + u.place(qc, K)]);
            if (q < Q) uv[st] = !late && q < K ? rscale(w0, x) : x;
        }
        for (int k0 = kb; k0 < ke; k0 += 4) {
            const int slot = k0 + lb < ke ? k0 + lb : ke - 1;
            const T* vr = v.at + (int64_t(p.col_ind[slot]) * 4 + li) * v.ld;
            double re = 0.0, im = 0.0;
#pragma unroll
            for (int s0 = 0; s0 < QS; s0 += 4) {
                if (4 * s0 >= nq) break;
                T vv[4];
                if (4 * (s0 + 4) <= nq) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) vv[t] = vr[v.place(q0 + 4 * (s0 + t) + lk, K)];
                } else {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int q = q0 + 4 * (s0 + t) + lk;
                        vv[t] = *or_zeros(q < Q, vr + v.place(q, K));
                    }
                }
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    A x = widen(uv[s0 + t]);
                    const A y = widen(vv[t]);
                    if (late && q0 + 4 * (s0 + t) < K) x = rscale(q0 + 4 * (s0 + t) + lk < K ? w0 : 1.0, x);
                    if constexpr (Sc<T>::is_complex) {
                        re = __builtin_amdgcn_mfma_f64_4x4x4f64(x.re, y.re, re, 0, 0, 0);
                        im = __builtin_amdgcn_mfma_f64_4x4x4f64(x.im, y.re, im, 0, 0, 0);
                        re = __builtin_amdgcn_mfma_f64_4x4x4f64(x.im, y.im, re, 0, 0, 0);
                        im = __builtin_amdgcn_mfma_f64_4x4x4f64(-x.re, y.im, im, 0, 0, 0);
                    } else {
                        re = __builtin_amdgcn_mfma_f64_4x4x4f64(x, y, re, 0, 0, 0);
                    }
                }
            }
            // lane (j, b, a): entry (a, j) of slot b
            if (k0 + lb < ke) {
                G_t& g = Gv[int64_t(slot) * 16 + lk * 4 + li];
                if constexpr (Sc<G_t>::is_complex) {
                    const A d = A{re, im} * alpha;
                    g = g + G_t{d.re, d.im};
                } else {
                    g += re * are;
                }
            }
        }
    }
}

template <typename T, typename V>
static void sddmm(vbh_matrix* m, int K, int nterms, const Factors<T>& u, const Factors<T>& v, double w0,
                  const double* alpha, V* G, hipStream_t s) {
    const int Q = nterms * K;
    if (m->uniform_bs == 4) {
        const int Gn = ((m->nbr + kWaves - 1) / kWaves + 7) & ~7;
        hipLaunchKernelGGL((k_sddmm_quads<T, V>), dim3(Gn), dim3(kThreads), 0, s, m->pattern(), K, Q, u, v, w0,
                           alpha[0], alpha[1], G, Gn);
    } else {
        hipLaunchKernelGGL((k_sddmm<T, V>), dim3(m->G), dim3(kThreads), 0, s, m->pattern(), K, Q, u, v, w0, alpha[0],
                           alpha[1], G, (const int*)m->split, m->G);
    }
    VBH_CHECK_HIP(hipGetLastError());
}

// t_n at Tb + n * term (rows ld apart), n < nterms; with Y also the series Y =
// sum_n c_n t_n.
template <typename T, typename V>
static void cheb_basis(vbh_matrix* m, int K, const T* X, int64_t ldx, int nterms, T* Tb, int64_t term, int64_t ld,
                       const double* coef, T* Y, int64_t ldy, double center, double half, hipStream_t s) {
    const int64_t N = m->n_rows;
    if (N * K == 0 || nterms <= 0) return;
    const unsigned nb = unsigned((N * K + 255) / 256);
    hipLaunchKernelGGL((k_copy_rows<T>), dim3(nb), dim3(256), 0, s, N, K, X, ldx, Tb, ld);
    VBH_CHECK_HIP(hipGetLastError());
    if (Y) cheb_accum<T>(N, K, X, ldx, Y, ldy, coef, 0, s);
    const V* vals = compute_values<V>(m, s);
    for (int n = 1; n < nterms; ++n) {
        const int st = n - 1;  // produces t_n from t_{n-1} (and t_{n-2})
        auto a = make_args<T, V>(m, vals, K, Tb + st * term, ld, Tb + n * term, ld);
        a.alpha = st == 0 ? 1.0 / half : 2.0 / half;
        a.beta = st == 0 ? -center / half : -2.0 * center / half;
        a.gamma = st == 0 ? 0.0 : -1.0;
        a.Z = st == 0 ? nullptr : Tb + (st - 1) * term;
        a.ldz = ld;
        if (Y) {
            const SeriesAcc<T> sa{Y, ldy, coef[2 * n], coef[2 * n + 1]};
            if (launch_series<T, V>(m, a, sa, s)) continue;
        }
        launch_rows<T, true, V>(m, a, s);
        if (Y) cheb_accum<T>(N, K, Tb + n * term, ld, Y, ldy, coef, n, s);
    }
}

// b_n at B + n * term (rows ld apart): one launch per term, the combination in
// the adjoint kernel's epilogue.
template <typename T>
static void cheb_adjoint(vbh_matrix* m, int K, const T* lam, int64_t ldl, int nterms, const double* coef, T* B,
                         int64_t term, int64_t ld, double center, double half, hipStream_t s) {
    const int64_t N = m->n_rows;
    if (N * K == 0 || nterms <= 0) return;
    const unsigned nb = unsigned((N * K + 255) / 256);
    const T* vals = compute_values<T>(m, s);
    for (int n = nterms - 1; n >= 0; --n) {
        T* bn = B + n * term;
        if (n + 1 == nterms) {
            hipLaunchKernelGGL((k_scale_rows<T>), dim3(nb), dim3(256), 0, s, N, K, bn, ld, lam, ldl, coef[2 * n],
                               -coef[2 * n + 1]);
            VBH_CHECK_HIP(hipGetLastError());
            continue;
        }
        const double s1 = (n == 0 ? 1.0 : 2.0) / half;
        AdjointStep<T> st{};
        st.alpha = s1;
        st.beta = -s1 * center;
        st.Z = n + 2 < nterms ? bn + 2 * term : nullptr;
        st.ldz = ld;
        st.term = SeriesAcc<T>{const_cast<T*>(lam), ldl, coef[2 * n], -coef[2 * n + 1]};
        apply_adjoint<T>(m, vals, K, bn + term, ld, bn, ld, s, &st);
    }
}

}  // namespace vbh

using namespace vbh;

extern "C" {

VBH_API int vbh_cheb_basis(vbh_matrix_t m, int K, const void* X, int ldx, int nterms, void* T, int ldt, double center,
                           double half_width, int precision, void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m && X && T, "null argument");
        VBH_REQUIRE(m->nbc == m->nbr, "the Chebyshev basis needs a square local pattern without ghosts");
        VBH_REQUIRE(K >= 1 && nterms >= 1 && ldx >= K && ldt >= int64_t(nterms) * K, "ldt must be >= nterms*K");
        VBH_REQUIRE(half_width > 0.0, "half_width must be positive");
        VBH_REQUIRE(precision == 0 || precision == 1, "precision must be 0 or 1");
        dispatch_compute(m, precision, [&](auto* tag, auto* vtag) {
            using Tt = std::remove_pointer_t<decltype(tag)>;
            using V = std::remove_pointer_t<decltype(vtag)>;
            cheb_basis<Tt, V>(m, K, (const Tt*)X, ldx, nterms, (Tt*)T, K, ldt, nullptr, nullptr, 0, center, half_width,
                              (hipStream_t)stream);
        });
    });
}

VBH_API int vbh_cheb_adjoint(vbh_matrix_t m, int K, const void* L, int ldl, int nterms, const double* coef, void* B,
                             int ldb, double center, double half_width, int precision, void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m && L && B && coef, "null argument");
        VBH_REQUIRE(m->nbc == m->nbr, "the Chebyshev adjoint needs a square local pattern without ghosts");
        VBH_REQUIRE(K >= 1 && nterms >= 1 && ldl >= K && ldb >= int64_t(nterms) * K, "ldb must be >= nterms*K");
        VBH_REQUIRE(half_width > 0.0, "half_width must be positive");
        VBH_REQUIRE(precision == 0 || precision == 1, "precision must be 0 or 1");
        dispatch_compute(m, precision, [&](auto* tag, auto*) {
            using Tt = std::remove_pointer_t<decltype(tag)>;
            cheb_adjoint<Tt>(m, K, (const Tt*)L, ldl, nterms, coef, (Tt*)B, K, ldb, center, half_width,
                             (hipStream_t)stream);
        });
    });
}

VBH_API int vbh_sddmm(vbh_matrix_t m, int L, const void* U, int ldu, const void* V, int ldv, const double* alpha,
                      void* G, int precision, void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m && G && alpha, "null argument");
        VBH_REQUIRE(L >= 0 && ldu >= L && ldv >= L, "leading dimensions must be >= L");
        VBH_REQUIRE(precision == 0 || precision == 1, "precision must be 0 or 1");
        if (m->nbr == 0 || L == 0 || m->nnz == 0) return;
        VBH_REQUIRE(U && V, "null U or V");
        hipStream_t s = (hipStream_t)stream;
        dispatch_compute(m, precision, [&](auto* tag, auto*) {
            using Tt = std::remove_pointer_t<decltype(tag)>;
            // G has the matrix's own type: double for real, complex128 for complex
            using Gt = std::conditional_t<Sc<Tt>::is_complex, c128, double>;
            sddmm<Tt, Gt>(m, L, 1, Factors<Tt>{(const Tt*)U, 0, ldu}, Factors<Tt>{(const Tt*)V, 0, ldv}, 1.0, alpha,
                          (Gt*)G, s);
        });
    });
}

VBH_API int vbh_cheb_basis_terms(vbh_matrix_t m, int K, const void* X, int ldx, int nterms, void* T, int64_t tstride,
                                 const double* coef, void* Y, int ldy, double center, double half_width, int precision,
                                 void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m && X && T, "null argument");
        VBH_REQUIRE(m->nbc == m->nbr, "the Chebyshev basis needs a square local pattern without ghosts");
        VBH_REQUIRE(K >= 1 && nterms >= 1 && ldx >= K && tstride >= m->n_rows * K, "tstride must be >= n_rows*K");
        VBH_REQUIRE(!Y || (coef && ldy >= K), "the series needs coefficients and ldy >= K");
        VBH_REQUIRE(half_width > 0.0, "half_width must be positive");
        VBH_REQUIRE(precision == 0 || precision == 1, "precision must be 0 or 1");
        dispatch_compute(m, precision, [&](auto* tag, auto* vtag) {
            using Tt = std::remove_pointer_t<decltype(tag)>;
            using V = std::remove_pointer_t<decltype(vtag)>;
            cheb_basis<Tt, V>(m, K, (const Tt*)X, ldx, nterms, (Tt*)T, tstride, K, coef, (Tt*)Y, ldy, center,
                              half_width, (hipStream_t)stream);
        });
    });
}

VBH_API int vbh_cheb_adjoint_terms(vbh_matrix_t m, int K, const void* L, int ldl, int nterms, const double* coef,
                                   void* B, int64_t bstride, double center, double half_width, int precision,
                                   void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m && L && B && coef, "null argument");
        VBH_REQUIRE(m->nbc == m->nbr, "the Chebyshev adjoint needs a square local pattern without ghosts");
        VBH_REQUIRE(K >= 1 && nterms >= 1 && ldl >= K && bstride >= m->n_rows * K, "bstride must be >= n_rows*K");
        VBH_REQUIRE(half_width > 0.0, "half_width must be positive");
        VBH_REQUIRE(precision == 0 || precision == 1, "precision must be 0 or 1");
        dispatch_compute(m, precision, [&](auto* tag, auto*) {
            using Tt = std::remove_pointer_t<decltype(tag)>;
            cheb_adjoint<Tt>(m, K, (const Tt*)L, ldl, nterms, coef, (Tt*)B, bstride, K, center, half_width,
                             (hipStream_t)stream);
        });
    });
}

VBH_API int vbh_sddmm_terms(vbh_matrix_t m, int K, int nterms, const void* U, int64_t ustride, const void* V,
                            int64_t vstride, double first, const double* alpha, void* G, int precision, void* stream) {
    return guard_on(stream, [&] {
        VBH_REQUIRE(m && G && alpha, "null argument");
        VBH_REQUIRE(K >= 0 && nterms >= 0 && int64_t(K) * nterms <= INT32_MAX, "bad term counts");
        VBH_REQUIRE(ustride >= m->n_rows * K && vstride >= m->n_cols * K, "strides must cover a term");
        VBH_REQUIRE(precision == 0 || precision == 1, "precision must be 0 or 1");
        if (m->nbr == 0 || K == 0 || nterms == 0 || m->nnz == 0) return;
        VBH_REQUIRE(U && V, "null U or V");
        dispatch_compute(m, precision, [&](auto* tag, auto*) {
            using Tt = std::remove_pointer_t<decltype(tag)>;
            using Gt = std::conditional_t<Sc<Tt>::is_complex, c128, double>;
            sddmm<Tt, Gt>(m, K, nterms, Factors<Tt>{(const Tt*)U, ustride, K}, Factors<Tt>{(const Tt*)V, vstride, K},
                          first, alpha, (Gt*)G, (hipStream_t)stream);
        });
    });
}

}  // extern "C"
