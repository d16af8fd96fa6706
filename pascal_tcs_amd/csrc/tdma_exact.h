// tdma_exact.h -- tridiagonal lines in PaScaL_TDMA's single-rank operation
// order (PaScaL_TDMA/src/pascal_tdma.f90:487-578 and :715-806, reduced 2-row
// solves of PaScaL_TDMA/src/tdmas.f90:113-212), one lane a line: the line
// solves of tdma.hip and the Poisson y solves of pressure.hip.
//
// One lane owns one system and walks its rows in the reference's order: the
// forward elimination with A fill-in, then the backward elimination with C
// fill-in.  The recurrences are a serial chain (an IEEE division a row on
// the way forward), so what bounds a solve is that chain when there are few
// systems and the traffic of the eliminated rows when there are many:
//   * a workgroup is one wavefront, so a few thousand systems reach every CU,
//     and the rows of the next chunk are loaded while the current one is
//     eliminated (128^3 in 256-thread workgroups with the loads in the
//     chain: 114-122 us a strided solve, 171 us a contiguous one);
//   * the eliminated a, c, d of the last rows of a line stay in LDS, as many
//     as the wavefronts that share a CU leave room for;
//   * the backward elimination runs twice: once without a store, to find the
//     two ends of the solution, and once more, the same operations, to
//     write the solution (counted: 111 B an unknown contiguous, 102 to 104
//     strided at 256x200x256, 49 strided at 128^3, where most rows stay in
//     LDS; 128 and 124 at 512^3 with the eliminated coefficients returned;
//     three passes in place moved 136).
#pragma once

#include <algorithm>
#include <type_traits>

#include "tcs_internal.h"

namespace tcs {
namespace exact_line {

constexpr int EX_W = 64;  // lines per workgroup (one wavefront)
constexpr int EX_U = 8;   // rows of a chunk of strided lines
constexpr int EX_R = 16;  // rows of a chunk of contiguous lines (a 128-byte segment)

// a row as it comes and the eliminated row of one line; NR right-hand sides
// share the matrix recurrences
template <int NR>
struct Row {
    double a, b, c, d[NR];
};
template <int NR>
struct Elim {
    double a, c, d[NR];
};
// rows 1 and 2 normalised by their own diagonal (:503-511)
template <int NR>
__device__ __forceinline__ Elim<NR> first_row(const Row<NR> &w) {
    Elim<NR> e;
    e.a = w.a / w.b;
#pragma unroll
    for (int k = 0; k < NR; k++) e.d[k] = w.d[k] / w.b;
    e.c = w.c / w.b;
    return e;
}
// row j >= 2 entering the forward elimination after row j - 1 (:513-520)
template <int NR>
__device__ __forceinline__ Elim<NR> fwd_row(const Row<NR> &w, const Elim<NR> &p) {
    const double r = 1.0 / (w.b - w.a * p.c);
    Elim<NR> e;
#pragma unroll
    for (int k = 0; k < NR; k++) e.d[k] = r * (w.d[k] - w.a * p.d[k]);
    e.c = r * w.c;
    e.a = -r * w.a * p.a;
    return e;
}
// row j of the backward elimination after row j + 1 (:523-529)
template <int NR>
__device__ __forceinline__ Elim<NR> back_row(const Elim<NR> &e, const Elim<NR> &x) {
    Elim<NR> n;
#pragma unroll
    for (int k = 0; k < NR; k++) n.d[k] = e.d[k] - e.c * x.d[k];
    n.a = e.a - e.c * x.a;
    n.c = -e.c * x.c;
    return n;
}
// rows 2 and n_row of the reduced form to the ends of the solution
// (:531-542): e0 comes back as the reference leaves row 1
template <bool CYC, int NR>
__device__ __forceinline__ void line_ends(Elim<NR> &e0, const Elim<NR> &e1, const Elim<NR> &eN, double (&x1)[NR],
                                          double (&xn)[NR]) {
    {
        const double r = 1.0 / (1.0 - e1.a * e0.c);
#pragma unroll
        for (int k = 0; k < NR; k++) e0.d[k] = r * (e0.d[k] - e0.c * e1.d[k]);
        e0.a = r * e0.a;
        e0.c = -r * e0.c * e1.c;
    }
    if (!CYC) {
        // tdma_many with n2=2, b=1 (tdmas.f90:113-146); x/1.0 is exact
        const double r = 1.0 / (1.0 - eN.a * e0.c);
#pragma unroll
        for (int k = 0; k < NR; k++) {
            xn[k] = r * (eN.d[k] - eN.a * e0.d[k]);
            x1[k] = e0.d[k] - e0.c * xn[k];
        }
    } else {
        // tdma_cycl_many with n2=2 (tdmas.f90:159-212): e(2) is set to -a(2)
        // and then overwritten by e(n2) = -c(n2)
        const double e2 = -eN.c;
#pragma unroll
        for (int k = 0; k < NR; k++) {
            x1[k] = (e0.d[k] - e0.a * eN.d[k] - e0.c * eN.d[k]) / (1.0 + e0.a * e2 + e0.c * e2);
            xn[k] = eN.d[k] + x1[k] * e2;
        }
    }
}

// One line of n_row >= 2 rows: load(j) gives row j, put(j, e) and get(j) keep
// its eliminated form in between, emit(j, e, x) takes the solution x of row
// j with the row's final eliminated form.
template <bool CYC, int NR, class Load, class Put, class Get, class Emit>
__device__ __forceinline__ void solve(int n_row, Load load, Put put, Get get, Emit emit) {
    Elim<NR> e0 = first_row<NR>(load(0)), e1 = first_row<NR>(load(1));
    Row<NR> cur[EX_U], nxt[EX_U];
#pragma unroll
    for (int u = 0; u < EX_U; u++)
        if (2 + u < n_row) cur[u] = load(2 + u);
    put(1, e1);
    Elim<NR> p = e1, pp = e1;  // rows j - 1 and j - 2
    int j0 = 2;
    for (; j0 + 2 * EX_U <= n_row; j0 += EX_U) {
#pragma unroll
        for (int u = 0; u < EX_U; u++) nxt[u] = load(j0 + EX_U + u);
#pragma unroll
        for (int u = 0; u < EX_U; u++) {
            pp = p;
            p = fwd_row<NR>(cur[u], p);
            put(j0 + u, p);
        }
#pragma unroll
        for (int u = 0; u < EX_U; u++) cur[u] = nxt[u];
    }
    for (; j0 < n_row; j0 += EX_U) {
#pragma unroll
        for (int u = 0; u < EX_U; u++)
            if (j0 + EX_U + u < n_row) nxt[u] = load(j0 + EX_U + u);
#pragma unroll
        for (int u = 0; u < EX_U; u++)
            if (j0 + u < n_row) {
                pp = p;
                p = fwd_row<NR>(cur[u], p);
                put(j0 + u, p);
            }
#pragma unroll
        for (int u = 0; u < EX_U; u++) cur[u] = nxt[u];
    }
    const Elim<NR> eN = p, eT = n_row >= 3 ? pp : e1;  // rows n_row and n_row - 1

    // the backward elimination j = n_row - 2 .. 2, OUT: giving out the solution
    double x1[NR], xn[NR];
    auto backward = [&](auto out) {
        constexpr bool OUT = decltype(out)::value;
        auto give = [&](int j, const Elim<NR> &e) {
            if constexpr (OUT) {
                double x[NR];
#pragma unroll
                for (int k = 0; k < NR; k++) x[k] = e.d[k] - e.a * x1[k] - e.c * xn[k];
                emit(j, e, x);
            }
        };
        Elim<NR> x = eT, q[EX_U], r[EX_U];
        int j = n_row - 3;  // next row
#pragma unroll
        for (int u = 0; u < EX_U; u++)
            if (j - u >= 1) q[u] = get(j - u);
        if (n_row >= 3) give(n_row - 2, x);
        for (; j - 2 * EX_U + 1 >= 1; j -= EX_U) {
#pragma unroll
            for (int u = 0; u < EX_U; u++) r[u] = get(j - EX_U - u);
#pragma unroll
            for (int u = 0; u < EX_U; u++) {
                x = back_row<NR>(q[u], x);
                give(j - u, x);
            }
#pragma unroll
            for (int u = 0; u < EX_U; u++) q[u] = r[u];
        }
        for (; j >= 1; j -= EX_U) {
#pragma unroll
            for (int u = 0; u < EX_U; u++)
                if (j - EX_U - u >= 1) r[u] = get(j - EX_U - u);
#pragma unroll
            for (int u = 0; u < EX_U; u++)
                if (j - u >= 1) {
                    x = back_row<NR>(q[u], x);
                    give(j - u, x);
                }
#pragma unroll
            for (int u = 0; u < EX_U; u++) q[u] = r[u];
        }
        return x;  // row 2
    };
    const Elim<NR> x2 = backward(std::integral_constant<bool, false>());
    line_ends<CYC, NR>(e0, x2, eN, x1, xn);
    backward(std::integral_constant<bool, true>());
    emit(0, e0, x1);
    emit(n_row - 1, eN, xn);
}

// The eliminated rows of a wavefront's lines kept in LDS, [row][value][lane].
template <int NR>
struct Kept {
    static constexpr int VALUES = 2 + NR;
    static constexpr int ROW_BYTES = VALUES * EX_W * (int)sizeof(double);
    double *v;
    int lane;
    __device__ __forceinline__ void put(int row, const Elim<NR> &e) const {
        double *q = v + (size_t)row * (VALUES * EX_W) + lane;
        q[0] = e.a;
        q[EX_W] = e.c;
#pragma unroll
        for (int k = 0; k < NR; k++) q[(2 + k) * EX_W] = e.d[k];
    }
    __device__ __forceinline__ Elim<NR> get(int row) const {
        const double *q = v + (size_t)row * (VALUES * EX_W) + lane;
        Elim<NR> e;
        e.a = q[0];
        e.c = q[EX_W];
#pragma unroll
        for (int k = 0; k < NR; k++) e.d[k] = q[(2 + k) * EX_W];
        return e;
    }
};
// How many: what 160 KB a CU leave each of the wavefronts that share it
// (these kernels hold one a SIMD).
template <int NR>
inline int kept_rows(long lines, int n_row) {
    const long waves = (lines + EX_W - 1) / EX_W;
    const int per_cu = (int)std::min<long>(4, (waves + 255) / 256);
    return std::min(n_row - 1, (156 * 1024 / per_cu) / Kept<NR>::ROW_BYTES);
}
constexpr int KEPT_LDS = 160 * 1024;  // dynamic LDS limit to ask for

}  // namespace exact_line
}  // namespace tcs
