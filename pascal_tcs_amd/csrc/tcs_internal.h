// tcs_internal.h -- context layout and device helpers shared by the HIP
// translation units of libpascal_tcs.  Not part of the C-ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <initializer_list>
#include <string>
#include <utility>

#include "../../include/pascal_tcs.h"
#include "device_once.h"

namespace tcs {

void set_error(const std::string &msg);

// Per-label HIP-event timing of kernel launches and stage entry points
// (the device counterpart of the reference's labelled timers,
// PaScaL_TDMA/src/timer.f90).  Active only while a context has it enabled;
// every launch in this library goes through TCS_LAUNCH.
struct Profiler;
struct AdjWork;  // adjoint fields and the step's kept values (adjoint.hip)
void prof_begin(const char *label, hipStream_t s);
void prof_end(hipStream_t s);

#define TCS_HIP(expr)                                                          \
    do {                                                                       \
        hipError_t _e = (expr);                                                \
        if (_e != hipSuccess) {                                                \
            ::tcs::set_error(std::string(#expr) + ": " + hipGetErrorString(_e)); \
            return TCS_E_HIP;                                                  \
        }                                                                      \
    } while (0)

#define TCS_LAUNCH_CHECK()                                                     \
    do {                                                                       \
        hipError_t _e = hipGetLastError();                                     \
        if (_e != hipSuccess) {                                                \
            ::tcs::set_error(std::string("kernel launch: ") + hipGetErrorString(_e)); \
            return TCS_E_HIP;                                                  \
        }                                                                      \
    } while (0)

#define TCS_LAUNCH(st, label, kern, grd, blk, lds, ...)                        \
    do {                                                                       \
        ::tcs::prof_begin(label, st);                                          \
        hipLaunchKernelGGL(kern, grd, blk, lds, st, __VA_ARGS__);              \
        ::tcs::prof_end(st);                                                   \
        TCS_LAUNCH_CHECK();                                                    \
    } while (0)

#define TCS_TRY(expr)                                                          \
    do {                                                                       \
        int _r = (expr);                                                       \
        if (_r != TCS_OK) return _r;                                           \
    } while (0)

// An index of a cell formula in the adjoint's reverse pass: the index v and
// its constant offset o in {-1, 0, 1} from the cell's own, which names the
// input's accumulator (rev.h).  RelCell: element q of a field, rel from the
// three offsets; RelRow: element q of a (j, k) table.
struct Rel {
    int v, o;
    __host__ __device__ __forceinline__ operator int() const { return v; }
};
__device__ __forceinline__ Rel operator+(Rel a, int d) { return Rel{a.v + d, a.o + d}; }
__device__ __forceinline__ Rel operator-(Rel a, int d) { return Rel{a.v - d, a.o - d}; }
struct RelCell {
    size_t q;
    int rel;
};
struct RelRow {
    size_t q;
    int rel;
};
// the fixed plane v read by a cell formula in the place of the neighbour at
// offset o
__device__ __forceinline__ int at_plane(int, int v, int) { return v; }
__device__ __forceinline__ Rel at_plane(Rel, int v, int o) { return Rel{v, o}; }

// Grid description passed by value to every stencil kernel.
// Full fields: (0:n1m+1, 0:n2m+1, 0:n3m+1), i fastest, rows P1 >= N1
// elements apart (a multiple of 16) and each field allocated FIELD_FRONT
// elements after a 128-byte boundary, so the interior run i = 1.. of every
// row starts on a 128-byte line: a 16-cell row segment is one cache line.
// Interior work arrays: (1:n1m, 1:n2m, 1:n3m), i fastest.
constexpr int FIELD_FRONT = 15;
inline int field_pitch(int N1) { return (N1 + 15) / 16 * 16; }
struct Grid {
    int n1m, n2m, n3m;
    int N1, N2, N3;  // full extents n?m+2
    int P1;          // row pitch of the full fields
    int wrap;        // kernels that have the code for it write periodic ghosts and wall rows
    const double *dx1, *dx2, *dx3, *dmx1, *dmx2, *dmx3;
    const double *rdx1, *rdx2, *rdx3, *rdmx1, *rdmx2, *rdmx3;  // their reciprocals
    // the six tables (dx1, dmx1, dx2, dmx2, dx3, dmx3) back to back rounded to
    // float, then their reciprocals in the same order (the mixed form's rows)
    const float *fmet;
    const int *jC, *jS;
    __device__ __forceinline__ size_t ix(int i, int j, int k) const {
        return (size_t)i + (size_t)P1 * ((size_t)j + (size_t)N2 * (size_t)k);
    }
    __device__ __forceinline__ size_t b2(int i, int k) const { return (size_t)i + (size_t)N1 * (size_t)k; }
    __device__ __forceinline__ size_t t2(int j, int k) const { return (size_t)j + (size_t)N2 * (size_t)k; }
    __device__ __forceinline__ size_t r3(int i, int j, int k) const {
        return (size_t)(i - 1) + (size_t)n1m * ((size_t)(j - 1) + (size_t)n2m * (size_t)(k - 1));
    }
    // The periodic images in x and z of F(i, j, k) = v (element q): a kernel
    // that makes a whole field leaves its rows as the ghost-cell update would.
    // Called in a branch of the few wavefronts for which edge() holds, after
    // the stores of the cells themselves: tested cell by cell at each store,
    // the images cost blockLdU 0.5 of 1.8 ms at 512^3.
    template <class E>
    __device__ __forceinline__ void images(E *F, int i, int k, size_t q, E v) const {
        const long di = i == 1 ? n1m : i == n1m ? -n1m : 0;
        if (di) F[(long)q + di] = v;
        if (k == 1 || k == n3m) {
            const long dk = (k == 1 ? (long)n3m : -(long)n3m) * P1 * N2;
            F[(long)q + dk] = v;
            if (di) F[(long)q + dk + di] = v;
        }
    }
    // whether cells i0..i0+ib-1, j, k0..k0+kb-1 touch the edge of the
    // interior; ib and kb divide n1m and n3m
    __device__ __forceinline__ bool edge(int i0, int ib, int j, int k0, int kb) const {
        return j == 1 || j == n2m || i0 == 1 || i0 + ib > n1m || k0 == 1 || k0 + kb > n3m;
    }
    // F's wall row next to row j, if there is one, from src's, with its
    // images: the thread of an edge row brings over the wall row of a second
    // buffer, or with src = F renews a wall row's ghosts
    template <class E, class E0>
    __device__ __forceinline__ void wall(E *F, const E0 *src, int i, int j, int k) const {
        for (int s = 0; s < 2; s++) {
            if (s ? j != n2m : j != 1) continue;
            const size_t q = ix(i, s ? j + 1 : 0, k);
            const E v = (E)src[q];
            F[q] = v;
            images(F, i, k, q, v);
        }
    }
    // The cells of a full field outside the interior, numbered: the faces i in
    // {0, n1m+1} (all j, k), then j in {0, n2m+1} (interior i, all k), then k
    // in {0, n3m+1} (interior i and j)
    __host__ __device__ size_t shell_size() const {
        return (size_t)2 * N2 * N3 + (size_t)2 * n1m * N3 + (size_t)2 * n1m * n2m;
    }
    __device__ __forceinline__ size_t shell_cell(size_t q) const {
        const size_t fi = (size_t)2 * N2 * N3, fj = (size_t)2 * n1m * N3;
        const int side = (int)(q % 2);  // the faces' sizes are even
        if (q < fi) {
            const size_t r = q / 2;
            return ix(side ? N1 - 1 : 0, (int)(r % N2), (int)(r / N2));
        }
        if ((q -= fi) < fj) {
            const size_t r = q / 2;
            return ix((int)(r % n1m) + 1, side ? N2 - 1 : 0, (int)(r / n1m));
        }
        const size_t r = (q - fj) / 2;
        return ix((int)(r % n1m) + 1, (int)(r / n1m) + 1, side ? N3 - 1 : 0);
    }
    __device__ __forceinline__ RelCell ix(Rel i, Rel j, Rel k) const {
        return RelCell{ix(i.v, j.v, k.v), (k.o + 1) * 9 + (j.o + 1) * 3 + (i.o + 1)};
    }
    __device__ __forceinline__ RelCell b2(Rel i, Rel k) const { return RelCell{b2(i.v, k.v), 13 + i.o}; }
    __device__ __forceinline__ RelRow t2(Rel j, Rel k) const {
        return RelRow{t2(j.v, k.v), (k.o + 1) * 3 + (j.o + 1)};
    }
};

// Polynomial property coefficients and nondimensional constants.
struct Phys {
    double Ct, Cmu, Cmt, Cmp, DeltaT;
    double a10, a11, a12, a13, a14, a15;
    double b10, b11, b12, b13, b14, b15;
    double c10, c11, c12, c13, c14, c15;
    double d10, d11, d12, d13, d14, d15;
    double KPP0, Rho0, Cp0, Mu0, a12pera11;
    // the fast forms' property polynomials, from the coefficients above:
    // c10/KPP0, Rho0*Cp0, and the numerator of d(1/(rho cp)) as a quintic
    double kppS, rcS, dircN[6];
};

}  // namespace tcs

struct tcs_ctx {
    tcs_params prm;
    tcs::Phys phys;
    int n1m, n2m, n3m;
    int N1, N2, N3;
    int P1;  // row pitch of the full fields (field_pitch(N1))
    size_t nfull, nint, nwall, ntab;
    int h1p, h3p;
    int device;
    int tdma_split;          // tcs_params.tdma_split
    hipStream_t stream;

    // host copies of the metrics
    double *h_dx1, *h_dx2, *h_dx3, *h_dmx1, *h_dmx2, *h_dmx3;
    // device metrics / masks
    double *dx1, *dx2, *dx3, *dmx1, *dmx2, *dmx3;
    double *rmet;            // 1/dx1, 1/dmx1, 1/dx2, 1/dmx2, 1/dx3, 1/dmx3 back to back,
                             // then the float tables of Grid::fmet
    int *jC, *jS;

    double *f[TCS_NFIELD];  // INVRHO / MU hold (0:n2sub,0:n3sub) tables
    // second buffers of T, U, V, W, dPhat, dP0: tcs_step writes their
    // updates there (the reads of the old values stay undisturbed) and swaps;
    // outside tcs_step their contents are dead (field uploads and downloads
    // stage through spare[TCS_T])
    double *spare[TCS_NFIELD];
    double *wall[TCS_NWALL];

    // ADI scratch (interior size each)
    double *am, *ac, *ap, *rhs;
    // stale scalars of the momentum stages (mu1,mu2 of dV; mu1..mu4 of dW)
    double *stale;

    // Poisson
    double *prhs;            // interior
    double *spec_x;          // complex (h1p, n2m, n3m), kx fastest
    double *spec_y;          // complex (h1p, n3m, n2m), kx fastest then kz
    double *pA, *pC;         // TDMA scratch (h1p*n3m, n2m)
    double *dxk2, *dzk;      // wave numbers
    double *ptab;            // y coefficients am(j), ap(j), ac(j) of the Poisson systems
    double *tw1, *tw3;       // twiddles (n/2 complex each)
    double *linesum, *planesum, *scal;  // mean reduction
    double *red;             // reduction scratch
    double *h_pinned;        // pinned host scalars
    tcs::Profiler *prof;     // null unless profiling is enabled
    tcs::AdjWork *adj;       // null until an adjoint entry is called
    int cfl_valid;           // cfl_max holds mpi_Post_CFL's maximum for the current fields
    double cfl_max;
    // routine calls held back so that the next call can fuse with them
    // (PEND_* bits; tcs::flush_pending runs them as called)
    int pend;
    double pend_dt_ldv, pend_dt_ldu, pend_dt_rhs;
    // Set within tcs_step, which knows that every field a kernel writes whole
    // is followed by its ghost-cell update.  The routines called one by one
    // leave the ghosts to tcs_ghostcell_update, as a caller may look at them
    // in between.
    int wrap;
    // Whether the kernels of a step write the periodic ghosts and the wall
    // rows of their fields themselves (Grid::edge, images, wall; LineOut::gx).
    // On a small grid they do, instead of 13 launches that cost 5 us each.
    // Past 2^23 cells the fields are followed by ghost-cell updates, which
    // bring the wall rows of a second buffer along, and the kernels are those
    // without ghost code: the stores of the images, one per line of memory,
    // and the registers they take in kernels at their bandwidth cost more than
    // the launches (at 512^3 written by the kernels 32.3 ms a step, 53.0 in
    // the exact form and 24.7 in the mixed; by launches 32.1, 51.9 and 24.5).
    // Kernels against launches, plain and mixed: 64^3 211 us against 224 and
    // 288 against 301; 256x128x128 1.11 ms against 1.12 and 0.85 against 0.87;
    // 256x128x256 (2^23) 2.16 against 2.15 and 1.56 against 1.57.
    bool wrap_fields() const { return wrap && nint <= ((size_t)1 << 23); }
    // The mixed form (precision 2): every array its stage rows and block
    // corrections read (T, U, V, W, P and the second buffers of T, U, V, W;
    // dU, dV, dW; the Mu and invRho tables; the wall tables; the stale
    // scalars) is carved from one FP64 arena a64 of an elements, and the
    // FP32 arena a32 holds each one's twin at the same element offset.  The
    // twins of the increments dU, dV, dW are where the mixed form keeps them
    // (the FP64 arrays are filled from them on download); the others are
    // FP32 copies of the FP64 arrays, current while their TWIN_* bit is set
    // in twin_ok.  Null / 0 in the FP64 forms.
    double *a64;
    float *a32;
    size_t an, aused;
    unsigned twin_ok;

    tcs::Grid grid() const {
        tcs::Grid g;
        g.n1m = n1m; g.n2m = n2m; g.n3m = n3m;
        g.N1 = N1; g.N2 = N2; g.N3 = N3;
        g.P1 = P1;
        g.wrap = wrap;
        g.dx1 = dx1; g.dx2 = dx2; g.dx3 = dx3;
        g.rdx1 = rmet; g.rdmx1 = rmet + N1; g.rdx2 = rmet + 2 * N1; g.rdmx2 = g.rdx2 + N2;
        g.rdx3 = g.rdx2 + 2 * N2; g.rdmx3 = g.rdx3 + N3;
        g.fmet = reinterpret_cast<const float *>(rmet + 2 * (N1 + N2 + N3));
        g.dmx1 = dmx1; g.dmx2 = dmx2; g.dmx3 = dmx3;
        g.jC = jC; g.jS = jS;
        return g;
    }
};

namespace tcs {

// Reductions that end in the same launch: thread 0 of each workgroup leaves
// its value(s) with last_put and then asks last_arrive, true in the workgroup
// that arrives last, whose threads read every value with last_get.  A
// put's exchange has been performed where all XCDs see it when its old value
// is back, and last_arrive's add is issued after that, so no fence is needed:
// a release per workgroup writes back and an acquire drops the whole of its
// XCD's L2 (1024 workgroups of a reduction over 64^3 cells: 31 us).
__device__ __forceinline__ unsigned long long last_swap(double *p, double v) {
    return __hip_atomic_exchange(reinterpret_cast<unsigned long long *>(p), (unsigned long long)__double_as_longlong(v),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void last_put(double *p, double v) {
    const unsigned long long old = last_swap(p, v);
    asm volatile("" ::"v"(old) : "memory");  // wait for it
}
__device__ __forceinline__ void last_put(double *p, double v, double *p1, double v1) {
    const unsigned long long old = last_swap(p, v), old1 = last_swap(p1, v1);
    asm volatile("" ::"v"(old), "v"(old1) : "memory");
}
__device__ __forceinline__ bool last_arrive(unsigned *count, unsigned n) {
    const bool last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    if (last) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return last;
}
__device__ __forceinline__ double last_get(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Dynamic LDS past 64 KiB (gfx950: 160 KiB per CU) needs the kernel's limit
// raised, on each device: to be called before a launch, with the most that
// any of the kernel's launches asks for.
int lds_limit(const void *kernel, size_t most, DeviceSet &raised);

// launch helpers -------------------------------------------------------------
inline dim3 interior_block() { return dim3(64, 4, 1); }
// Row j = blockIdx.y * 4 + threadIdx.y + 1 of a kernel launched with
// interior_block(): the 64 threads of a wavefront share threadIdx.y, so j is
// the same on every lane, and readfirstlane lets the compiler see it (the
// (j, k) tables and j's metrics are then loaded once per wavefront).
__device__ __forceinline__ int wave_row_j() {
    return __builtin_amdgcn_readfirstlane((int)(blockIdx.y * blockDim.y + threadIdx.y + 1));
}
inline dim3 interior_grid(int nx, int ny, int nz) {
    return dim3((unsigned)((nx + 63) / 64), (unsigned)((ny + 3) / 4), (unsigned)nz);
}
// Cell-update stencil kernels where a thread takes KB consecutive k planes
// of one (i, j) (KB <= 4 divides n3m, a power of two >= 4): the values a
// plane shares with the next are loaded once.
inline dim3 cell_grid(int nx, int ny, int nz, int kb, dim3 blk = interior_block(), int ib = 1) {
    return dim3((unsigned)((nx / ib + blk.x - 1) / blk.x), (unsigned)((ny + blk.y - 1) / blk.y), (unsigned)(nz / kb));
}

// Where a solve puts its solution: back into D (mode 0), or into an
// FP64 field F at F[base + s0*ss0 + s1*ss1 + row*rs], stored (mode 1),
// added to what F holds (mode 2), or added to what Fin holds at the same
// place (mode 3: F a second buffer of the field), or stored into the FP32
// field G (mode 4: the mixed form's increments) -- the last sweep of an ADI
// stage writes the increment straight into its module array.
struct LineOut {
    double *F = nullptr;
    const double *Fin = nullptr;
    float *G = nullptr;  // mode 4: the FP32 field G at the same place, stored; modes 1-3 of FP32
                         // lines: G (when set) also receives the FP32 copy of the FP64 value
    long base = 0, ss0 = 0, ss1 = 0, rs = 0;
    int mode = 0;
    // > 0: gx x gz lines of n_row rows, written with their periodic ghosts in
    // s0 and s1 and with the wall rows before and after them (mode 3: Fin's)
    int gx = 0, gz = 0, n_row = 0;
    bool zero_walls = false;  // (gx > 0) the wall rows become zero (dV's)
    void wrap_to(const tcs_ctx *c, int nr) {
        if (c->wrap_fields()) { gx = c->n1m; gz = c->n3m; n_row = nr; }
    }
};
namespace part {
// F[o] = v and its images on the periodic ghost lines di in s0 and dk in s1
// away (0: none), stored with the value still in registers: read back from the
// line's own stores afterwards, the images took 50 us of a 110 us solve at
// 256^3, in the few workgroups that have them.
template <typename E>
__device__ __forceinline__ void put_line(E *F, long o, E v, long di, long dk) {
    F[o] = v;
    if (di) F[o + di] = v;
    if (dk) {
        F[o + dk] = v;
        if (di) F[o + dk + di] = v;
    }
}
}  // namespace part

// TDMA launcher (exact PaScaL order) on strided systems:
//   system (s0, s1) starts at base + s0*ss0 + s1*ss1, rows step rs.
// Right-hand sides from Din, solutions to Dout (which may be Din); A and C
// are overwritten, with keep by the reference's modified coefficients.  out
// (mode 1, non-cyclic strided systems): the solutions into a field instead,
// Dout overwritten.
int ptdma_exact_launch(double *A, const double *B, double *C, const double *Din, double *Dout, int n0, long ss0,
                       int n1, long ss1, int n_row, long rs, bool cyclic, bool keep, hipStream_t st,
                       const LineOut &out = LineOut());
// The same systems split into parts (PaScaL_TDMA's multi-rank algorithm,
// one thread per rank); n_row in [2, 512]; strided lines need ss0 = 1.
bool ptdma_part_plan(int n_row, int &P, int &w1, int &w2);
int ptdma_part_launch(double *A, const double *B, double *C, double *D, int n0, long ss0, int n1, long ss1,
                      int n_row, long rs, bool cyclic, hipStream_t st, const LineOut &out = LineOut());
// right-hand sides from Din, solutions to Dout (which may be Din)
int ptdma_part_launch(const double *A, const double *B, const double *C, const double *Din, double *Dout, int n0,
                      long ss0, int n1, long ss1, int n_row, long rs, bool cyclic, hipStream_t st);
// FP32 lines (the mixed form's ADI solves), same algorithm and layouts.
int ptdma_part_launch(float *A, const float *B, float *C, float *D, int n0, long ss0, int n1, long ss1,
                      int n_row, long rs, bool cyclic, hipStream_t st, const LineOut &out = LineOut());
// ADI sweep of a context: split solve when the context asks for it and the
// line length allows, else the single-rank order.
inline int ptdma_sweep(const tcs_ctx *c, double *A, const double *B, double *C, const double *Din, double *Dout,
                       int n0, long ss0, int n1, long ss1, int n_row, long rs, bool cyclic) {
    int P, w1, w2;
    if (c->tdma_split && ptdma_part_plan(n_row, P, w1, w2) && (rs == 1 || ss0 == 1))
        return ptdma_part_launch(A, B, C, Din, Dout, n0, ss0, n1, ss1, n_row, rs, cyclic, c->stream);
    return ptdma_exact_launch(A, B, C, Din, Dout, n0, ss0, n1, ss1, n_row, rs, cyclic, false, c->stream);
}
inline int ptdma_sweep(const tcs_ctx *c, double *A, const double *B, double *C, double *D, int n0, long ss0,
                       int n1, long ss1, int n_row, long rs, bool cyclic) {
    return ptdma_sweep(c, A, B, C, D, D, n0, ss0, n1, ss1, n_row, rs, cyclic);
}
// FP32 sweep of the mixed form: always the split solve (lines <= 512 rows).
inline int ptdma_sweep(const tcs_ctx *c, float *A, const float *B, float *C, float *D, int n0, long ss0, int n1,
                       long ss1, int n_row, long rs, bool cyclic) {
    return ptdma_part_launch(A, B, C, D, n0, ss0, n1, ss1, n_row, rs, cyclic, c->stream);
}

// Stage entry points of the kernel translation units (thermal, momentum,
// pressure).  Each of them is compiled three times: into namespace `exact`
// with FP contraction off (the reference's operation order, precision 0),
// into namespace `fast` with contraction and reciprocal arithmetic allowed
// (precision 1), and into namespace `mixed`, the fast arithmetic with FP32
// ADI scratch and FP32 line solves (precision 2).  TCS_FORM names the
// namespace a translation unit builds, TCS_SCRATCH its scratch type.
// The *_into / *_pseudo routines are tcs_step's fused forms: thermal's last
// sweep writes T + dT into a second buffer (when the lines are split); the
// block corrections also write the pseudo-update U + dU, V + dV, W + dW and
// the projection the new dPhat, dP0 into second buffers.
#define TCS_STAGE_DECLS                                                                 \
    int thermal_solver(tcs_ctx *c, double dt);                                          \
    int thermal_coeffi(tcs_ctx *c);                                                     \
    int momentum_coeffi(tcs_ctx *c);                                                    \
    int momentum_solvedU(tcs_ctx *c, double dt);                                        \
    int momentum_solvedV(tcs_ctx *c, double dt);                                        \
    int momentum_solvedW(tcs_ctx *c, double dt);                                        \
    int momentum_blockLdV(tcs_ctx *c, double dt);                                       \
    int momentum_blockLdU(tcs_ctx *c, double dt);                                       \
    int momentum_pseudoupdate(tcs_ctx *c);                                              \
    int pressure_rhs(tcs_ctx *c, double dt);                                            \
    int pressure_poisson(tcs_ctx *c);                                                   \
    int pressure_poisson_rhs(tcs_ctx *c, double dt);                                    \
    int pressure_projection(tcs_ctx *c, double dt);                                     \
    int thermal_solver_into(tcs_ctx *c, double dt, double *Tn, bool *written);          \
    int momentum_blockLdV_pseudo(tcs_ctx *c, double dt, double *Vn);                    \
    int momentum_blockLdU_pseudo(tcs_ctx *c, double dt, double *Un, double *Wn);        \
    int pressure_projection_into(tcs_ctx *c, double dt, double *dPhatn, double *dP0n);
namespace exact { TCS_STAGE_DECLS }
namespace fast { TCS_STAGE_DECLS }
namespace mixed { TCS_STAGE_DECLS }
#undef TCS_STAGE_DECLS
// up to FieldSet::MAX full fields for one launch (blockIdx.y picks one)
struct FieldSet {
    static constexpr int MAX = 6;
    double *f[MAX];
};
struct FieldSet32 {
    float *f[FieldSet::MAX];
};
int halo(tcs_ctx *c, double *f);
// walls (not empty: one for each field, or null): the buffers that the fields'
// wall rows are brought over from, with their ghosts
int halo(tcs_ctx *c, std::initializer_list<double *> fields, std::initializer_list<const double *> walls = {});
// the same ghost-cell update of FP32 fields (the mixed form's increments)
int halo(tcs_ctx *c, std::initializer_list<float *> fields);
// The mixed form's FP32 twins of FP64 arrays (tcs_ctx::a32): which are
// current (tcs_ctx::twin_ok), making them current, and the increment of a
// field as the form keeps it (the FP64 array, or its FP32 twin).
enum {
    TWIN_T = 1, TWIN_U = 2, TWIN_V = 4, TWIN_W = 8, TWIN_P = 16,
    TWIN_TAB = 32,    // Mu, invRho
    TWIN_WALL = 64,   // the eight wall tables
    TWIN_STALE = 128  // the stale scalars of the momentum stages
};
int ensure_twins(tcs_ctx *c, unsigned bits);
// FP32 increment twin -> FP64 array (downloads of dU, dV, dW in the mixed
// form) and back (uploads)
int increment_to_fp64(tcs_ctx *c, int id);
int increment_from_fp64(tcs_ctx *c, int id);
// copy the cells outside the interior (x/z ghosts, wall rows) of fields into
// the second buffers that are to become them
int copy_shell(tcs_ctx *c, std::initializer_list<int> ids);
// Routine entries that hold their launches back: tcs_momentum_blockLdV, the
// ghost-cell update of dV after it and tcs_momentum_blockLdU wait for
// tcs_momentum_pseudoupdateUVW (which then runs the block corrections with
// the pseudo-update fused in), tcs_pressure_rhs waits for
// tcs_pressure_poisson_fft2 (the right-hand side made inside the x
// transform).  Every other entry point runs what is held first, unfused.
enum { PEND_LDV = 1, PEND_HALO_DV = 2, PEND_LDU = 4, PEND_RHS = 8 };
int flush_pending(tcs_ctx *c);
int post_div(tcs_ctx *c, double *out);
int post_cfl(tcs_ctx *c, double *maxuovx);
int nusselt(tcs_ctx *c, double Tup, double Tbt, double *nb, double *nt);
void adjoint_free(tcs_ctx *c);

}  // namespace tcs
