// rev.h -- reverse-mode derivatives of the per-cell formulas, in registers.
//
// A cell formula (ad.h) instantiated with S = Rev builds its derivatives from
// the language's own order of destruction: every named value of the formula
// is a local variable that holds its expression's partial derivatives and an
// adjoint; the outputs, assigned last, add their adjoints to the values they
// were made of, and when the formula returns its values are destroyed in
// the reverse of their order of definition, each handing its adjoint on to
// its operands, down to the inputs' accumulators.  No tape: after inlining
// it is straight-line code on registers, about three times the formula's
// operations.
//
// Rules for a formula: a value is defined once (const auto x = as<S>(...)),
// in the body of the formula function (not in a block or a function it
// calls), and a function it calls returns one expression of named values.
#pragma once

#include <utility>

#include "ad.h"

namespace tcs {

struct NodeTag {};
template <class T>
constexpr bool node_v = std::is_base_of<NodeTag, std::decay_t<T>>::value;

// a named value or an input: its value and where its adjoint is collected
struct Ref : NodeTag {
    double v;
    double *adj;
    __device__ __forceinline__ Ref(double x, double *a) : v(x), adj(a) {}
    __device__ __forceinline__ void back(double w) const {
#pragma clang fp contract(fast)
        *adj = *adj + w;
    }
};
// an operand of an operation: a Ref to a named value, or the node itself
// when it is a temporary of the expression
template <class T>
__device__ __forceinline__ auto operand(T &&t) {
    if constexpr (std::is_same<std::decay_t<T>, Ref>::value) {
        return Ref(t);
    } else if constexpr (std::is_lvalue_reference<T>::value) {
        t.live = true;
        return Ref(t.v, &t.adj);
    } else {
        return std::decay_t<T>(std::move(t));
    }
}

// operations with one or two differentiated operands: the value and its
// partial derivatives
template <class A>
struct Un : NodeTag {
    A a;
    double v, p;
    mutable double adj = 0.0;
    mutable bool live = false;  // a named value that was used
    __device__ __forceinline__ Un(A &&x, double val, double d) : a(std::move(x)), v(val), p(d) {}
    __device__ __forceinline__ Un(Un &&o) : a(std::move(o.a)), v(o.v), p(o.p) {}
    __device__ __forceinline__ void back(double w) const {
#pragma clang fp contract(fast)
        a.back(w * p);
    }
    __device__ __forceinline__ ~Un() {
        if (live) back(adj);
    }
};
template <class A, class B>
struct Bin : NodeTag {
    A a;
    B b;
    double v, pa, pb;
    mutable double adj = 0.0;
    mutable bool live = false;
    __device__ __forceinline__ Bin(A &&x, B &&y, double val, double da, double db)
        : a(std::move(x)), b(std::move(y)), v(val), pa(da), pb(db) {}
    __device__ __forceinline__ Bin(Bin &&o)
        : a(std::move(o.a)), b(std::move(o.b)), v(o.v), pa(o.pa), pb(o.pb) {}
    __device__ __forceinline__ void back(double w) const {
#pragma clang fp contract(fast)
        a.back(w * pa);
        b.back(w * pb);
    }
    __device__ __forceinline__ ~Bin() {
        if (live) back(adj);
    }
};
// v = f(x) with the derivative p; v = f(x, y) with px, py
template <class A>
__device__ __forceinline__ auto rev_of(A &&x, double v, double p) {
    auto o = operand(std::forward<A>(x));
    return Un<decltype(o)>(std::move(o), v, p);
}
template <class A, class B>
__device__ __forceinline__ auto rev_of2(A &&x, B &&y, double v, double px, double py) {
    auto o = operand(std::forward<A>(x));
    auto q = operand(std::forward<B>(y));
    return Bin<decltype(o), decltype(q)>(std::move(o), std::move(q), v, px, py);
}
#define REV_IF2 std::enable_if_t<node_v<A> && node_v<B>, int> = 0
#define REV_IF1 std::enable_if_t<node_v<A> && std::is_arithmetic<std::decay_t<B>>::value, int> = 0
#define REV_IF0 std::enable_if_t<std::is_arithmetic<std::decay_t<A>>::value && node_v<B>, int> = 0
template <class A, std::enable_if_t<node_v<A>, int> = 0>
__device__ __forceinline__ auto operator-(A &&a) { return rev_of(std::forward<A>(a), -a.v, -1.0); }
template <class A, class B, REV_IF2>
__device__ __forceinline__ auto operator+(A &&a, B &&b) {
    return rev_of2(std::forward<A>(a), std::forward<B>(b), a.v + b.v, 1.0, 1.0);
}
template <class A, class B, REV_IF2>
__device__ __forceinline__ auto operator-(A &&a, B &&b) {
    return rev_of2(std::forward<A>(a), std::forward<B>(b), a.v - b.v, 1.0, -1.0);
}
template <class A, class B, REV_IF2>
__device__ __forceinline__ auto operator*(A &&a, B &&b) {
    return rev_of2(std::forward<A>(a), std::forward<B>(b), a.v * b.v, b.v, a.v);
}
template <class A, class B, REV_IF2>
__device__ __forceinline__ auto operator/(A &&a, B &&b) {
    const double r = 1.0 / b.v, q = a.v * r;
    return rev_of2(std::forward<A>(a), std::forward<B>(b), q, r, -q * r);
}
template <class A, class B, REV_IF1>
__device__ __forceinline__ auto operator+(A &&a, const B &b) { return rev_of(std::forward<A>(a), a.v + (double)b, 1.0); }
template <class A, class B, REV_IF1>
__device__ __forceinline__ auto operator-(A &&a, const B &b) { return rev_of(std::forward<A>(a), a.v - (double)b, 1.0); }
template <class A, class B, REV_IF1>
__device__ __forceinline__ auto operator*(A &&a, const B &b) { return rev_of(std::forward<A>(a), a.v * (double)b, (double)b); }
template <class A, class B, REV_IF1>
__device__ __forceinline__ auto operator/(A &&a, const B &b) {
    const double r = 1.0 / (double)b;
    return rev_of(std::forward<A>(a), a.v * r, r);
}
template <class A, class B, REV_IF0>
__device__ __forceinline__ auto operator+(const A &a, B &&b) { return rev_of(std::forward<B>(b), (double)a + b.v, 1.0); }
template <class A, class B, REV_IF0>
__device__ __forceinline__ auto operator-(const A &a, B &&b) { return rev_of(std::forward<B>(b), (double)a - b.v, -1.0); }
template <class A, class B, REV_IF0>
__device__ __forceinline__ auto operator*(const A &a, B &&b) { return rev_of(std::forward<B>(b), (double)a * b.v, (double)a); }
template <class A, class B, REV_IF0>
__device__ __forceinline__ auto operator/(const A &a, B &&b) {
    const double r = 1.0 / b.v, q = (double)a * r;
    return rev_of(std::forward<B>(b), q, -q * r);
}
#undef REV_IF2
#undef REV_IF1
#undef REV_IF0

// An output of a formula: its adjoint, handed on when the output is assigned.
struct Rev {
    double seed = 0.0;
    template <class E>
    __device__ __forceinline__ void operator=(E &&e) {
        if constexpr (node_v<E>) operand(std::forward<E>(e)).back(seed);
    }
};

// Inputs.  Each differentiated field has an accumulator for every offset
// (dk, dj, di) of its elements around the cell; `used` and the element `at`
// of those a formula reads, and whose element it is: the lane's own, its x
// row's, every cell's.  After inlining the offsets are constants and the
// accumulators registers.
constexpr int REV_REL = 27;
enum { IN_CELL = 0, IN_ROW = 1, IN_ALL = 2 };
struct FieldBars {
    double adj[REV_REL];
    size_t at[REV_REL];
    bool used[REV_REL];
    int kind;
};
struct RevPtr {
    const double *p;
    FieldBars *b;
    bool diff;  // the field is differentiated
    double *sink;
    __device__ __forceinline__ Ref input(size_t q, int rel, int kind) const {
        if (!diff) return Ref(p[q], sink);
        b->used[rel] = true;
        b->at[rel] = q;
        b->kind = kind;
        return Ref(p[q], &b->adj[rel]);
    }
    __device__ __forceinline__ Ref operator[](const RelCell &c) const { return input(c.q, c.rel, IN_CELL); }
    __device__ __forceinline__ Ref operator[](const RelRow &c) const { return input(c.q, c.rel, IN_ROW); }
    __device__ __forceinline__ Ref operator[](int s) const { return input((size_t)s, s, IN_ALL); }
};
template <int ND>
struct RevW {
    FieldBars *bars;
    double *sink;
    __device__ __forceinline__ RevPtr operator()(int f, const double *p) const {
        return RevPtr{p, bars + (f < ND ? f : 0), f < ND, sink};
    }
};

struct OutBars {
    const double *p[4];
    int full;  // p in the fields' layout (1) or the interior layout (0)
    // rows of a solved stage instead (lam not null): their adjoints from
    // lambda = A^-T xbar and the solution x, -lambda x' with x' the solution
    // at the row before, at the row and after it on the stage's line, and
    // lambda for the right-hand side (has_d)
    const double *lam, *x;
    int axis, jlo, cyc, has_d;
};
// the line through interior cell q along `axis` (0 x, 1 y, 2 z), rows j >= jlo:
// position, length and stride of the line, and the cells before and after q
// on it (cyclically), with hp, hn whether the line has them
struct LinePos {
    int pos, n;
    long prev, next;
    bool hp, hn;
};
__device__ __forceinline__ LinePos line_pos(const Grid &g, int axis, int jlo, int cyc, int i, int j, int k) {
    const long n1 = g.n1m, q = (long)g.r3(i, j, k);
    const long stride = axis == 0 ? 1 : axis == 1 ? n1 : n1 * g.n2m;
    const int n = axis == 0 ? g.n1m : axis == 1 ? g.n2m - jlo + 1 : g.n3m;
    const int pos = axis == 0 ? i - 1 : axis == 1 ? j - jlo : k - 1;
    const long wrap = (long)(n - 1) * stride;
    return {pos, n, pos > 0 ? q - stride : q + wrap, pos < n - 1 ? q + stride : q - wrap, pos > 0 || cyc,
            pos < n - 1 || cyc};
}
template <int NF>
struct InBars {
    double *p[NF];  // adjoints of the input fields (the first Cell::ND are used)
};

// sum over aligned groups of lw lanes (a power of two)
__device__ __forceinline__ double lane_sum(double s, int lw) {
    for (int o = lw >> 1; o >= 1; o >>= 1) s += __shfl_xor(s, o);
    return s;
}
// *p += s with the FP64 atomic add of the L2 (HIP's atomicAdd on a double is
// a compare-and-swap loop, which neighbouring cells adding to shared inputs
// kept retrying: 224 against 67 ms an adjoint step at 128^3).  The adjoint
// arrays are device allocations (coarse-grained), which these atomics serve.
__device__ __forceinline__ void add_to(double *p, double s) {
    if (s != 0.0) unsafeAtomicAdd(p, s);
}

// The adjoints of the inputs of field F, offsets N.., into its adjoint array.
// IN_CELL inputs: the three x offsets of one (dk, dj) are the elements q - 1,
// q, q + 1, so each lane passes its outer two to its neighbours and adds one
// value (the end lanes of the row add theirs).  IN_ROW inputs are summed
// over the x row first; IN_ALL ones go to all[], which the kernel sums over
// its planes.
template <int N>
__device__ __forceinline__ void rev_scatter(const FieldBars &t, double *bar, int lw, int lane, bool act,
                                            double *all) {
    if constexpr (N < REV_REL) {
        constexpr int lo = N, c = N + 1, hi = N + 2;
        if (t.used[lo] || t.used[c] || t.used[hi]) {
            if (t.kind == IN_CELL) {
                const size_t q = t.used[c] ? t.at[c] : t.used[lo] ? t.at[lo] + 1 : t.at[hi] - 1;
                double s = t.used[c] ? t.adj[c] : 0.0;
                if (t.used[lo]) {
                    const double v = __shfl_down(t.adj[lo], 1);
                    if (lane != lw - 1) s += v;
                    if (act && lane == 0) add_to(bar + q - 1, t.adj[lo]);
                }
                if (t.used[hi]) {
                    const double v = __shfl_up(t.adj[hi], 1);
                    if (lane != 0) s += v;
                    if (act && lane == lw - 1) add_to(bar + q + 1, t.adj[hi]);
                }
                if (act) add_to(bar + q, s);
            } else {
                auto one = [&](int u) {
                    if (!t.used[u]) return;
                    if (t.kind == IN_ROW) {
                        const double s = lane_sum(t.adj[u], lw);
                        if (act && lane == 0) add_to(bar + t.at[u], s);
                    } else if (u < 6) {
                        all[u] += t.adj[u];
                    }
                };
                one(lo);
                one(c);
                one(hi);
            }
        }
        rev_scatter<N + 3>(t, bar, lw, lane, act, all);
    }
}
template <int ND, int F>
__device__ __forceinline__ void rev_scatter_fields(const FieldBars *t, double *const *bars, int lw, int lane,
                                                   bool act, double *all) {
    if constexpr (F < ND) {
        rev_scatter<0>(t[F], bars[F], lw, lane, act, all);
        rev_scatter_fields<ND, F + 1>(t, bars, lw, lane, act, all);
    }
}

// One cell: the adjoints w of its outputs in, its formula (in wall-term mode
// WM where it has one), the inputs' adjoints out.
template <int WM, class Cell>
__device__ __forceinline__ void cell_reverse(const Cell &cell, int i, int j, int k, const double (&w)[4],
                                             const InBars<Cell::NF> &ib, int lw, int lane, bool act, double *all) {
    constexpr int ND = Cell::ND;
    FieldBars t[ND] = {};
    double sink = 0.0;
    {
        Rev a{w[0]}, b{w[1]}, c{w[2]}, d{w[3]};
        const Rel ri{i, 0}, rj{j, 0}, rk{k, 0};
        if constexpr (WM >= 0) cell.template eval<Rev, WM>(RevW<ND>{t, &sink}, ri, rj, rk, a, b, c, d);
        else cell.template eval<Rev>(RevW<ND>{t, &sink}, ri, rj, rk, a, b, c, d);
    }
    rev_scatter_fields<ND, 0>(t, ib.p, lw, lane, act, all);
}

// rows whose wall terms can be left out away from the walls (wall_free(j))
template <class Cell, class = void>
struct HasWalls {
    static constexpr bool value = false;
};
template <class Cell>
struct HasWalls<Cell, std::void_t<decltype(&Cell::wall_free)>> {
    static constexpr bool value = true;
};

// Vector-Jacobian products of the cells (i, j, k), i in [1, n1m], j in [jlo,
// jhi], k in [1, n3m]: the cell's eval gives up to four outputs, whose
// adjoints are ob; each input's share is added to ib.  A wavefront takes
// 64 / lw rows j of lw = min(64, n1m) cells, VJP_KB planes k one after the
// other.  At 128^3 on one MI355X a backward step went from 38.3 to 5.0 ms
// with this pass (forward-mode passes over four inputs at a time before: the
// dW z rows 8.11 -> 0.33 ms, the thermal z rows 3.76 -> 0.22 ms).  The
// momentum z rows hold 260-310 registers and run one wavefront per SIMD.
constexpr int VJP_KB = 4;  // divides n3m, a power of two >= 4
// Copies of the stale scalars' adjoints, summed afterwards: every wavefront
// adds to them, and adds to one address follow each other (dW x at 128^3:
// 223 us with one copy).
constexpr int REV_STALE = 256, REV_STALE_STRIDE = 16;
template <class Cell>
__global__ void __launch_bounds__(64)
k_cell_vjp(Cell cell, int jlo, int jhi, int lw, OutBars ob, InBars<Cell::NF> ib) {
    const Grid &g = cell.g;
    const int lane = threadIdx.x % lw;
    const int i = blockIdx.x * lw + lane + 1;
    int j = jlo + blockIdx.y * (64 / lw) + threadIdx.x / lw;
    const bool act = j <= jhi;
    j = act ? j : jhi;  // lanes past the last row take part with zero adjoints
    double all[6] = {};
#pragma unroll 1
    for (int kk = 0; kk < VJP_KB; kk++) {
        const int k = blockIdx.z * VJP_KB + kk + 1;
        const size_t q = ob.full ? g.ix(i, j, k) : g.r3(i, j, k);
        double w[4];
        if (ob.lam) {
            const LinePos L = line_pos(g, ob.axis, ob.jlo, ob.cyc, i, j, k);
            const double l = act ? ob.lam[q] : 0.0;
            w[0] = L.hp ? -l * ob.x[L.prev] : 0.0;
            w[1] = -l * ob.x[q];
            w[2] = L.hn ? -l * ob.x[L.next] : 0.0;
            w[3] = ob.has_d ? l : 0.0;
        } else {
#pragma unroll
            for (int o = 0; o < 4; o++) w[o] = (act && ob.p[o]) ? ob.p[o][q] : 0.0;
        }
        const bool any = w[0] != 0.0 || w[1] != 0.0 || w[2] != 0.0 || w[3] != 0.0;
        if (__ballot(any) == 0) continue;
        if constexpr (HasWalls<Cell>::value) {
            if (__ballot(!cell.wall_free(j)) == 0) cell_reverse<2>(cell, i, j, k, w, ib, lw, lane, act, all);
            else cell_reverse<0>(cell, i, j, k, w, ib, lw, lane, act, all);
        } else {
            cell_reverse<-1>(cell, i, j, k, w, ib, lw, lane, act, all);
        }
    }
    if constexpr (Cell::STALE >= 0) {
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const double s = lane_sum(all[q], 64);
            const unsigned w = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
            if (threadIdx.x == 0) add_to(ib.p[Cell::STALE] + q + REV_STALE_STRIDE * (w % REV_STALE), s);
        }
    }
}

}  // namespace tcs
