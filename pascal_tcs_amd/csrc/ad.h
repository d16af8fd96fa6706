// ad.h -- exact derivatives of the per-cell formulas of the step.
//
// The stage rows (thermal, momentum) and the cell updates (block
// corrections, pressure right-hand side, projection) are templates over the
// scalar type S and the field access P: a cell evaluates its formula with
// P[idx] loads from its input fields.  Instantiated with S = double and raw
// pointers they are the step itself.  The adjoint instantiates them with
// reverse-mode numbers (Rev, rev.h): one evaluation and one sweep back give
// the cell's vector-Jacobian product, exactly (the same operations with
// their derivatives), and no formula is differentiated by hand.  Functions
// of one value (the property polynomials) go through forward-mode numbers
// (Dual) and enter it as one operation.
#pragma once

#include <type_traits>
#include <utility>

#include "tcs_internal.h"

namespace tcs {

// ---- scalars ---------------------------------------------------------------
struct Dual {
    double v, d;
    __host__ __device__ Dual() : v(0.0), d(0.0) {}
    __host__ __device__ Dual(double x) : v(x), d(0.0) {}
    __host__ __device__ Dual(double x, double y) : v(x), d(y) {}
};
__device__ __forceinline__ Dual operator-(Dual a) { return Dual(-a.v, -a.d); }
__device__ __forceinline__ Dual operator+(Dual a, Dual b) { return Dual(a.v + b.v, a.d + b.d); }
__device__ __forceinline__ Dual operator-(Dual a, Dual b) { return Dual(a.v - b.v, a.d - b.d); }
__device__ __forceinline__ Dual operator*(Dual a, Dual b) { return Dual(a.v * b.v, a.d * b.v + a.v * b.d); }
__device__ __forceinline__ Dual operator/(Dual a, Dual b) {
    const double q = a.v / b.v;
    return Dual(q, (a.d - q * b.d) / b.v);
}
__device__ __forceinline__ Dual operator+(Dual a, double b) { return Dual(a.v + b, a.d); }
__device__ __forceinline__ Dual operator+(double a, Dual b) { return Dual(a + b.v, b.d); }
__device__ __forceinline__ Dual operator-(Dual a, double b) { return Dual(a.v - b, a.d); }
__device__ __forceinline__ Dual operator-(double a, Dual b) { return Dual(a - b.v, -b.d); }
__device__ __forceinline__ Dual operator*(Dual a, double b) { return Dual(a.v * b, a.d * b); }
__device__ __forceinline__ Dual operator*(double a, Dual b) { return Dual(a * b.v, a * b.d); }
__device__ __forceinline__ Dual operator/(Dual a, double b) { return Dual(a.v / b, a.d / b); }
__device__ __forceinline__ Dual operator/(double a, Dual b) {
    const double q = a / b.v;
    return Dual(q, -q * b.d / b.v);
}

// Reverse-mode values (rev.h; a formula's outputs are Rev, its named values
// and inputs nodes of its expressions).
struct Rev;
template <class S>
constexpr bool is_rev() { return std::is_same<S, Rev>::value; }
template <class A>
__device__ auto rev_of(A &&x, double v, double p);
template <class A, class B>
__device__ auto rev_of2(A &&x, B &&y, double v, double px, double py);

// as<S>(e): a named value of a cell formula, of type S (in the reverse pass
// the expression's own type).
template <class S, class E>
__device__ __forceinline__ auto as(E &&e) {
    if constexpr (is_rev<S>()) return std::decay_t<E>(std::forward<E>(e));
    else return (S)e;
}
// passed ? a() : b().  The reverse pass takes both (what it records must not
// depend on the cell) and weights them 1 and 0.
template <class S, class A, class B>
__device__ __forceinline__ auto pick(bool passed, A a, B b) {
    if constexpr (is_rev<S>()) {
        auto x = a();
        auto y = b();
        const double v = passed ? x.v : y.v;
        return rev_of2(std::move(x), std::move(y), v, passed ? 1.0 : 0.0, passed ? 0.0 : 1.0);
    } else {
        return passed ? (S)a() : (S)b();
    }
}
// x with the wall terms f(x) in wall-term mode WM: 0 computes them, 1 skips
// them where near is false (not in the reverse pass), 2 leaves them out
template <class S, int WM, class X, class F>
__device__ __forceinline__ auto with_walls(bool near, const X &x, F f) {
    if constexpr (is_rev<S>()) {
        // what is recorded must not depend on the cell
        static_assert(WM != 1, "wall terms of the reverse pass: computed (0) or left out (2)");
        if constexpr (WM == 0) return f(x);
        else return rev_of(x, x.v, 1.0);
    } else if constexpr (WM == 0) {
        return (S)f(x);
    } else if constexpr (WM == 1) {
        S y = x;
        if (near) y = f(x);
        return y;
    } else {
        return x;
    }
}

// ---- field access ----------------------------------------------------------
// the step: raw pointers
struct RawW {
    __device__ __forceinline__ const double *operator()(int, const double *p) const { return p; }
};

// A value type of the adjoint (neither double nor float).  The stage rows
// have no branch on j for these: the reverse pass's operations are the same
// for every cell.
template <class S>
constexpr bool is_dual() { return !std::is_same<S, double>::value && !std::is_same<S, float>::value; }

// The mixed form's rows: FP32 arithmetic on the FP32 twins of the arrays
// they read.  In that form every array a stage row or block correction reads
// (state, increments, (j, k) tables, wall tables, stale scalars) lives in
// one FP64 arena and has an FP32 twin at the same element offset of an FP32
// arena, so the twin of p is f + (p - d).
struct F32Ptr {
    const float *p;
    __device__ __forceinline__ float operator[](size_t i) const { return p[i]; }
};
struct TwinW {
    const double *d;  // the FP64 arena
    const float *f;   // its FP32 twin
    __device__ __forceinline__ F32Ptr operator()(int, const double *p) const { return F32Ptr{f + (p - d)}; }
};
inline TwinW twin_w(const tcs_ctx *c) { return TwinW{c->a64, c->a32}; }
// the FP32 twin of an array of the mixed form's arena (null outside it)
inline float *twin(const tcs_ctx *c, const double *p) {
    if (!c->a64 || p < c->a64 || p >= c->a64 + c->an) return nullptr;
    return c->a32 + (p - c->a64);
}

// The input set of a formula evaluated on one thread: (field, index) of
// every load, without repeats (the stale viscosities).
constexpr int AD_MAXIN = 128;
struct Rec {
    int n;
    int fid[AD_MAXIN];
    long idx[AD_MAXIN];
    __device__ void add(int f, long i) {
        for (int r = 0; r < n; r++)
            if (fid[r] == f && idx[r] == i) return;
        if (n < AD_MAXIN) {
            fid[n] = f;
            idx[n] = i;
        }
        n++;  // n > AD_MAXIN reports an overflow
    }
};
struct RecPtr {
    const double *p;
    int f;
    Rec *rec;
    __device__ __forceinline__ double operator[](size_t i) const {
        rec->add(f, (long)i);
        return p[i];
    }
};
// one input seeded with derivative 1
struct SeedPtr {
    const double *p;
    long seed;
    __device__ __forceinline__ Dual operator[](size_t i) const { return Dual(p[i], (long)i == seed ? 1.0 : 0.0); }
};

}  // namespace tcs
