// adjoint.hip -- the discrete adjoint of one MPM-STD step (src/main.f90:131-203
// in the plain FP64 form, precision 0).
//
// The stage units are compiled here a fourth time, into namespace tcs::adj,
// so the adjoint uses the step's own row and cell formulas.  tcs_adjoint_step
// first runs the step forward from the context's state, keeping the inputs
// every nonlinear part needs and the three ADI solutions of every stage;
// then it walks the step backwards:
//   * halos, wall extrapolation, the dP mean: their transposes (the ghost
//     adjoints go to the periodic sources, the mean projection is symmetric);
//   * cell updates (projection, dPhat history, block corrections, pressure
//     RHS, pseudo-update): vector-Jacobian products of the cell formulas
//     (rev.h: one reverse pass a cell);
//   * each ADI stage x = A^-1 d: lambda = A^-T xbar by the transposed line
//     solve (the stage's rows, stored where the transposed systems have them,
//     solved as the step solves its lines: split when they are), row adjoints
//     abar_i = -lambda_i x_{i-1}, bbar_i = -lambda_i x_i, cbar_i = -lambda_i
//     x_{i+1}, dbar_i = lambda_i, then the rows' vector-Jacobian product;
//   * the Poisson solve: the same FFT pipeline with every wavenumber's
//     y-system transposed (the pinned mean mode's row projection after the
//     solve, the zeroed imaginary parts before it), which is the exact
//     transpose because the modified wavenumbers are even in kx and kz.
// The adjoint fields of the state (T, U, V, W, P, dPhat, dP0) and of the
// temperature wall arrays are kept in the context.
#define TCS_FORM adj
#define TCS_REV
#include "rev.h"
#include "momentum.hip"
#include "pressure.hip"
#include "thermal.hip"

#include <algorithm>
#include <utility>

namespace tcs {
namespace adj {

constexpr int NSTATE = 7;
constexpr int STATE_IDS[NSTATE] = {TCS_T, TCS_U, TCS_V, TCS_W, TCS_P, TCS_DPHAT, TCS_DP0};
enum { ST_T, ST_U, ST_V, ST_W, ST_P, ST_DPHAT, ST_DP0 };
enum { STG_T, STG_U, STG_V, STG_W };

}  // namespace adj

struct AdjWork {
    double *b[adj::NSTATE];         // adjoints of the state fields
    double *bdU, *bdV, *bdW, *bdP;  // of the increments (within a step)
    double *bMu, *biR, *bstale;     // of the (j,k) tables and the stale scalars
    double *bwall[TCS_NWALL];       // of the wall arrays
    double *tmp[4];                 // full-size work
    double *s0[adj::NSTATE];        // state at the start of the step
    // and within it, of what a later stage overwrites: dU and dV as solved,
    // U, V, W before the projection
    double *sdU1, *sdV1, *sU1, *sV1, *sW1;
    double *X[4][3];                // ADI stage solutions (interior layout)
    double *lam, *rint;             // interior layout
    double *psum;                   // partial sums of the dP mean, then the mean; a counter
    std::vector<void *> all;
};

namespace adj {

// ---- transposes of the linear pieces -----------------------------------------

// k_halo transposed: every ghost's adjoint goes to its periodic source (the
// same enumeration as k_halo; sources are never x or z ghosts)
__global__ void k_halo_adj(Grid g, FieldSet fs) {
    double *__restrict__ b = fs.f[blockIdx.y];  // one field per grid row
    const int N1 = g.N1, N2 = g.N2, N3 = g.N3;
    const int n1m = g.n1m, n3m = g.n3m;
    const size_t nx = (size_t)2 * N2 * N3, nz = (size_t)2 * N1 * N2;
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t dst, src;
    if (q < nx) {
        const int side = (int)(q % 2);
        const size_t r = q / 2;
        const int j = (int)(r % N2), k = (int)(r / N2);
        if (k == 0 || k == N3 - 1) return;
        dst = g.ix(side ? n1m + 1 : 0, j, k);
        src = g.ix(side ? 1 : n1m, j, k);
    } else if (q < nx + nz) {
        const size_t r = q - nx;
        const int side = (int)(r % 2);
        const size_t t = r / 2;
        const int i = (int)(t % N1), j = (int)(t / N1);
        const int is = (i == 0) ? n1m : (i == n1m + 1 ? 1 : i);
        dst = g.ix(i, j, side ? n3m + 1 : 0);
        src = g.ix(is, j, side ? 1 : n3m);
    } else {
        return;
    }
    const double v = b[dst];
    b[dst] = 0.0;
    if (v != 0.0) unsafeAtomicAdd(b + src, v);  // the L2's FP64 atomic (not a compare-and-swap loop)
}

int halo_adj(tcs_ctx *c, std::initializer_list<double *> fields) {
    FieldSet fs{};
    int nf = 0;
    for (double *b : fields) {
        if (nf == FieldSet::MAX) return TCS_E_ARG;
        fs.f[nf++] = b;
    }
    const size_t n = (size_t)2 * c->N2 * c->N3 + (size_t)2 * c->N1 * c->N2;
    TCS_LAUNCH(c->stream, "adj_halo", k_halo_adj, dim3((unsigned)((n + 255) / 256), (unsigned)nf), dim3(256), 0,
               c->grid(), fs);
    return TCS_OK;
}

// k_wall_extrap transposed
__global__ void k_wall_extrap_adj(Grid g, double *__restrict__ b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int k = blockIdx.y + 1;
    if (i > g.n1m) return;
    const double *dmx2 = g.dmx2;
    const int n2sub = g.n2m + 1, n2msub = g.n2m;
    const double s = dmx2[1] + dmx2[2];
    const double a0 = (s * s) / ((s * s) - (dmx2[1] * dmx2[1]));
    const double b0 = (dmx2[1] * dmx2[1]) / ((s * s) - (dmx2[1] * dmx2[1]));
    const double t = dmx2[n2sub] + dmx2[n2msub];
    const double a1 = (t * t) / ((t * t) - (dmx2[n2sub] * dmx2[n2sub]));
    const double b1 = (dmx2[n2sub] * dmx2[n2sub]) / ((t * t) - (dmx2[n2sub] * dmx2[n2sub]));
    const double gb = b[g.ix(i, 0, k)], gt = b[g.ix(i, n2sub, k)];
    b[g.ix(i, 0, k)] = 0.0;
    b[g.ix(i, n2sub, k)] = 0.0;
    b[g.ix(i, 1, k)] += a0 * gb;
    b[g.ix(i, 2, k)] -= b0 * gb;
    b[g.ix(i, n2msub, k)] += a1 * gt;
    b[g.ix(i, n2sub - 2, k)] -= b1 * gt;
}

int wall_extrap_adj(tcs_ctx *c, double *b) {
    TCS_LAUNCH(c->stream, "adj_wall_extrap", k_wall_extrap_adj, dim3((c->n1m + 63) / 64, c->n3m), dim3(64), 0,
               c->grid(), b);
    return TCS_OK;
}

// The interior's mean into out[SUM_BLOCKS] (out: partial sums, the mean, a
// counter): the last workgroup adds the partial sums in their order.
constexpr int SUM_BLOCKS = 512;
__device__ __forceinline__ double block_sum(double v, double *s) {
    s[threadIdx.x] = v;
    __syncthreads();
    for (int h = 128; h >= 1; h >>= 1) {
        if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
        __syncthreads();
    }
    v = s[0];
    __syncthreads();
    return v;
}
__global__ void __launch_bounds__(256) k_interior_mean(Grid g, const double *__restrict__ b, double *out) {
    __shared__ double s[256];
    __shared__ bool last;
    const size_t n = (size_t)g.n1m * g.n2m * g.n3m;
    double v = 0.0;
    for (size_t q = (size_t)blockIdx.x * 256 + threadIdx.x; q < n; q += (size_t)gridDim.x * 256) {
        const size_t r = q / g.n1m;
        v += b[g.ix((int)(q - r * g.n1m) + 1, (int)(r % g.n2m) + 1, (int)(r / g.n2m) + 1)];
    }
    v = block_sum(v, s);
    if (threadIdx.x == 0) {
        last_put(out + blockIdx.x, v);
        last = last_arrive(reinterpret_cast<unsigned *>(out + SUM_BLOCKS + 1), gridDim.x);
    }
    __syncthreads();
    if (!last) return;
    v = 0.0;
    for (unsigned q = threadIdx.x; q < gridDim.x; q += 256) v += last_get(out + q);
    v = block_sum(v, s);
    if (threadIdx.x == 0) out[SUM_BLOCKS] = v / ((double)g.n1m * (double)g.n2m * (double)g.n3m);
}

// r (interior layout) = the interior of b minus the mean, and b's interior 0
__global__ void k_take_mean(Grid g, const double *__restrict__ mean, double *__restrict__ b, double *__restrict__ r) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
    const int k = blockIdx.z + 1;
    if (i > g.n1m || j > g.n2m) return;
    const size_t q = g.ix(i, j, k);
    r[g.r3(i, j, k)] = b[q] - mean[0];
    b[q] = 0.0;
}

// b at (i, j, k), element q, plus what its periodic images hold, which are
// set to zero: k_halo_adj's fold for the one cell that has those images
__device__ __forceinline__ double fold_images(const Grid &g, double *b, int i, int k, size_t q) {
    double v = b[q];
    auto take = [&](long d) {
        v += b[(long)q + d];
        b[(long)q + d] = 0.0;
    };
    const long di = i == 1 ? g.n1m : i == g.n1m ? -g.n1m : 0;
    if (di) take(di);
    if (k == 1 || k == g.n3m) {
        const long dk = (k == 1 ? (long)g.n3m : -(long)g.n3m) * g.P1 * g.N2;
        take(dk);
        if (di) take(dk + di);
    }
    return v;
}
// The ghost-cell update of b transposed, then r (interior layout) = its
// interior (0 for rows j < jlo).  ZERO: b (ghosts and wall rows too) ends
// as zero, the stage having replaced the field; otherwise b stays.
template <bool ZERO>
__global__ void k_take(Grid g, int jlo, double *b, double *__restrict__ r) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
    const int k = blockIdx.z + 1;
    if (i > g.n1m || j > g.n2m) return;
    const size_t q = g.ix(i, j, k);
    const double v = fold_images(g, b, i, k, q);
    b[q] = ZERO ? 0.0 : v;
    r[g.r3(i, j, k)] = j >= jlo ? v : 0.0;
    for (int s = 0; s < 2; s++) {
        if (s ? j != g.n2m : j != 1) continue;
        const size_t o = g.ix(i, s ? j + 1 : 0, k);
        const double w = fold_images(g, b, i, k, o);
        b[o] = ZERO ? 0.0 : w;
    }
}

// Work on several arrays in one launch, an array a grid row
struct Arrays {
    static constexpr int MAX = 20;
    double *dst[MAX];
    const double *src[MAX];
    size_t n[MAX];
    int count = 0;
    void add(double *d, const double *s, size_t len) {
        dst[count] = d;
        src[count] = s;
        n[count++] = len;
    }
};
// dst = src, or 0 where src is null
__global__ void __launch_bounds__(256) k_copy_arrays(Arrays a) {
    double *__restrict__ dst = a.dst[blockIdx.y];
    const double *__restrict__ src = a.src[blockIdx.y];
    const size_t n = a.n[blockIdx.y], st = (size_t)gridDim.x * 256;
    if (src)
        for (size_t q = (size_t)blockIdx.x * 256 + threadIdx.x; q < n; q += st) dst[q] = src[q];
    else
        for (size_t q = (size_t)blockIdx.x * 256 + threadIdx.x; q < n; q += st) dst[q] = 0.0;
}
static int copy_arrays(tcs_ctx *c, const Arrays &a) {
    size_t most = 1;
    for (int q = 0; q < a.count; q++) most = std::max(most, a.n[q]);
    TCS_LAUNCH(c->stream, "adj_copy", k_copy_arrays, dim3((unsigned)std::min<size_t>((most + 1023) / 1024, 1024), a.count),
               dim3(256), 0, a);
    return TCS_OK;
}

// transposed Poisson y-systems, one (kx, kz) system per thread (the rows of
// k_poisson_tdma: A = amj, B = acj - dxk2 - dzk, C = apj, the mean mode's
// first row pinned); imaginary parts zeroed before, the pinned row after
__global__ void k_poisson_tdma_T(int n3m, int h1p, int n2m, int h3p, const double *__restrict__ amj,
                                 const double *__restrict__ apj, const double *__restrict__ acj,
                                 const double *__restrict__ dxk2, const double *__restrict__ dzk,
                                 double2 *S, double *cw) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int nsys = n3m * h1p;
    if (s >= nsys) return;
    const int kx = s / n3m, kz = s - kx * n3m;
    const size_t rs = (size_t)nsys;
    double2 *d = S + s;
    double *cp = cw + s;
    const double shift = dxk2[kx], zk = dzk[kz];
    const bool pin = (kx == 0 && kz == 0);
    const bool zim = (kx == 0 && (kz == 0 || kz == h3p - 1));
    auto A = [&](int jj) { return (pin && jj == 0) ? 0.0 : amj[jj]; };
    auto B = [&](int jj) { return (pin && jj == 0) ? 1.0 : acj[jj] - shift - zk; };
    auto C = [&](int jj) { return (pin && jj == 0) ? 0.0 : apj[jj]; };
    // row jj of the transpose: (C(jj-1), B(jj), A(jj+1)); ends dropped
    // (non-cyclic).  The rows come U at a time, the next ones in flight.
    constexpr int U = 8;
    double cprev = 0.0, dr = 0.0, di = 0.0;
    double2 v[U], nv[U];
#pragma unroll
    for (int u = 0; u < U; u++)
        if (u < n2m) v[u] = d[(size_t)u * rs];
    for (int j0 = 0; j0 < n2m; j0 += U) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (j0 + U + u < n2m) nv[u] = d[(size_t)(j0 + U + u) * rs];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int jj = j0 + u;
            if (jj >= n2m) break;
            const double at = jj > 0 ? C(jj - 1) : 0.0;
            const double ct = jj < n2m - 1 ? A(jj + 1) : 0.0;
            const double m = 1.0 / (B(jj) - at * cprev);
            const double vi = zim ? 0.0 : v[u].y;
            dr = (v[u].x - at * dr) * m;
            di = (vi - at * di) * m;
            cprev = ct * m;
            cp[(size_t)jj * rs] = cprev;
            d[(size_t)jj * rs] = make_double2(dr, di);
        }
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = nv[u];
    }
    double xr = dr, xi = di, w[U], nw[U];
#pragma unroll
    for (int u = 0; u < U; u++)
        if (n2m - 2 - u >= 0) { v[u] = d[(size_t)(n2m - 2 - u) * rs]; w[u] = cp[(size_t)(n2m - 2 - u) * rs]; }
    for (int j0 = n2m - 2; j0 >= 0; j0 -= U) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (j0 - U - u >= 0) { nv[u] = d[(size_t)(j0 - U - u) * rs]; nw[u] = cp[(size_t)(j0 - U - u) * rs]; }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int jj = j0 - u;
            if (jj < 0) break;
            xr = v[u].x - w[u] * xr;
            xi = v[u].y - w[u] * xi;
            d[(size_t)jj * rs] = make_double2(xr, xi);
        }
#pragma unroll
        for (int u = 0; u < U; u++) { v[u] = nv[u]; w[u] = nw[u]; }
    }
    if (pin) d[0] = make_double2(0.0, d[0].y);
}

// ---- ADI stage transposes ------------------------------------------------------

// A stage's rows (rows3d's) with the transposed systems' coefficients: aT_i =
// c_{i-1} and cT_i = a_{i+1}, each coefficient stored where the transposed
// row has it
template <class Row>
__global__ void __launch_bounds__(256) k_rows3d_T(Row row, int axis, int jlo, int cyc, double *__restrict__ aT,
                                                  double *__restrict__ b, double *__restrict__ cT) {
    const Grid &g = row.g;
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = wave_row_j();
    if (i > g.n1m || j > g.n2m || j < jlo) return;
#pragma unroll
    for (int q = 0; q < ROWS3D_KB; q++) {
        const int k = blockIdx.z * ROWS3D_KB + q + 1;
        double am, ac, ap, d;
        row(i, j, k, am, ac, ap, d);
        const LinePos L = line_pos(g, axis, jlo, cyc, i, j, k);
        const size_t o = g.r3(i, j, k);
        b[o] = ac;
        if (L.hp) cT[L.prev] = am;
        else aT[o] = 0.0;
        if (L.hn) aT[L.next] = ap;
        else cT[o] = 0.0;
    }
}

template <class Cell>
int cell_vjp(tcs_ctx *c, AdjWork *w, const Cell &cell, int jlo, OutBars ob, InBars<Cell::NF> ib) {
    const int lw = std::min(64, c->n1m), rows = 64 / lw;
    const dim3 blk(64), grd((unsigned)(c->n1m / lw), (unsigned)((c->n2m - jlo + rows) / rows),
                            (unsigned)(c->n3m / VJP_KB));
    TCS_LAUNCH(c->stream, "adj_cell_vjp", (k_cell_vjp<Cell>), grd, blk, 0, cell, jlo, c->n2m, lw, ob, ib);
    return TCS_OK;
}

// Line geometry of a stage's solves over the rows j >= jlo (as the forward
// stages launch them): (n0, ss0, n1, ss1, n_row, rs) and the offset of row jlo.
struct LineGeom {
    long off;
    int n0;
    long ss0;
    int n1;
    long ss1;
    int n_row;
    long rs;
};
static LineGeom geom(const tcs_ctx *c, int axis, int jlo) {
    const long n1 = c->n1m, n12 = (long)c->n1m * c->n2m, off = (long)(jlo - 1) * n1;
    const int nl = c->n2m - jlo + 1;
    if (axis == 2) return {off, c->n1m, 1, nl, n1, c->n3m, n12};
    if (axis == 0) return {off, nl, n1, c->n3m, n12, c->n1m, 1};
    return {off, c->n1m, 1, c->n3m, n12, nl, n1};
}

static int sweep(tcs_ctx *c, double *A, const double *B, double *C, const double *Din, double *Dout, int axis,
                 int jlo, bool cyc) {
    const LineGeom L = geom(c, axis, jlo);
    return ptdma_sweep(c, A + L.off, B + L.off, C + L.off, Din + L.off, Dout + L.off, L.n0, L.ss0, L.n1, L.ss1, L.n_row, L.rs, cyc);
}

// One stage backwards.  On entry w->lam holds xbar (interior layout, rows
// j >= jlo); on exit it holds lambda = A^-T xbar, which is the adjoint of the
// stage's right-hand side (the previous stage's solution for x and y
// stages; the rows' own d for the z stage, HAS_D).
template <bool HAS_D, class Row>
int stage_adj(tcs_ctx *c, AdjWork *w, const Row &row, int axis, int jlo, bool cyc, const double *X,
              InBars<Row::NF> ib) {
    TCS_LAUNCH(c->stream, "adj_rows", k_rows3d_T<Row>,
               cell_grid(c->n1m, c->n2m, c->n3m, ROWS3D_KB, interior_block(), 1), interior_block(), 0, row, axis, jlo,
               (int)cyc, c->am, c->ac, c->ap);
    TCS_TRY(sweep(c, c->am, c->ac, c->ap, w->lam, w->lam, axis, jlo, cyc));
    const OutBars ob{{}, 0, w->lam, X, axis, jlo, (int)cyc, (int)HAS_D};
    return cell_vjp(c, w, row, jlo, ob, ib);
}

// ---- small kernels -----------------------------------------------------------

// U += dU, V += dV (j >= 2; times 0 at j = 1), W += dW transposed
__global__ void k_pseudo_adj(Grid g, const double *__restrict__ bU, const double *__restrict__ bV,
                             const double *__restrict__ bW, double *__restrict__ bdU, double *__restrict__ bdV,
                             double *__restrict__ bdW) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
    const int k = blockIdx.z + 1;
    if (i > g.n1m || j > g.n2m) return;
    const size_t q = g.ix(i, j, k);
    bdU[q] += bU[q];
    bdV[q] += j >= 2 ? bV[q] : bV[q] * 0.0;
    bdW[q] += bW[q];
}

// Mu, invRho tables from T(n1sub, j, k) transposed
__global__ void k_coeffi_adj(Grid g, Phys p, const double *__restrict__ T, const double *__restrict__ bMu,
                             const double *__restrict__ biR, double *__restrict__ bT) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int k = blockIdx.y;
    if (j >= g.N2) return;
    const size_t q = g.ix(g.n1m + 1, j, k);
    Dual mu, ir;
    mu_ir_of_T(p, Dual(T[q], 1.0), mu, ir);
    bT[q] += mu.d * bMu[g.t2(j, k)] + ir.d * biR[g.t2(j, k)];
}

// the stale viscosities transposed: the copies of their adjoints summed,
// then, on one thread, six outputs of a few inputs
__global__ void __launch_bounds__(64) k_stale_adj(Grid g, const double *__restrict__ Mu,
                                                  const double *__restrict__ bstale, double *__restrict__ bMu) {
    double b[6];
    for (int q = 0; q < 6; q++) {
        double s = 0.0;
        for (int c = threadIdx.x; c < REV_STALE; c += 64) s += bstale[q + REV_STALE_STRIDE * c];
        b[q] = lane_sum(s, 64);
    }
    if (threadIdx.x != 0) return;
    Rec rec;
    rec.n = 0;
    double v[6];
    stale_values<double>(g, RecPtr{Mu, 0, &rec}, v);
    for (int r = 0; r < rec.n && r < AD_MAXIN; r++) {
        Dual o[6];
        stale_values<Dual>(g, SeedPtr{Mu, rec.idx[r]}, o);
        double s = 0.0;
        for (int q = 0; q < 6; q++) s += o[q].d * b[q];
        bMu[rec.idx[r]] += s;
    }
}

// the wall Nusselt number's gradient, times weight: Nu_bottom =
// sum over the interior (TBCbt - T(i,1,k)) / dmx2(1) * L2 / (n1m n3m dT)
__global__ void k_nusselt_adj(Grid g, double wgt, double *__restrict__ bT, double *__restrict__ bTbt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int k = blockIdx.y + 1;
    if (i > g.n1m) return;
    bT[g.ix(i, 1, k)] -= wgt;
    bTbt[g.b2(i, k)] += wgt;
}

// ---- the step forward, keeping what the adjoint needs ----------------------------

// A stage's increment (interior layout) into its field: stored (MODE 1, 0 in
// rows j < j0 and, with j0 > 1, in the wall rows) or added (MODE 2), with the
// field's ghost-cell update; S (not null) keeps a copy of the whole field.
template <int MODE>
__global__ void k_store_keep(Grid g, int j0, const double *__restrict__ inc, double *F, double *S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
    const int k = blockIdx.z + 1;
    if (i > g.n1m || j > g.n2m) return;
    auto put = [&](size_t q, double v) {
        F[q] = v;
        g.images(F, i, k, q, v);
        if (!S) return;
        S[q] = v;
        g.images(S, i, k, q, v);
    };
    const size_t q = g.ix(i, j, k);
    const double v = j >= j0 ? inc[g.r3(i, j, k)] : 0.0;
    put(q, MODE == 1 ? v : F[q] + v);
    for (int s = 0; s < 2; s++) {
        if (s ? j != g.n2m : j != 1) continue;
        const size_t o = g.ix(i, s ? j + 1 : 0, k);
        put(o, j0 > 1 ? 0.0 : F[o]);
    }
}
template <int MODE>
static int store_keep(tcs_ctx *c, int j0, const double *inc, double *F, double *S) {
    TCS_LAUNCH(c->stream, "adj_fwd_store", k_store_keep<MODE>, interior_grid(c->n1m, c->n2m, c->n3m),
               interior_block(), 0, c->grid(), j0, inc, F, S);
    return TCS_OK;
}

// the fields' ghost-cell updates, and copies of the whole fields
__global__ void k_halo_keep(Grid g, Arrays a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
    const int k = blockIdx.z % g.n3m + 1, f = blockIdx.z / g.n3m;
    if (i > g.n1m || j > g.n2m) return;
    double *S = a.dst[f], *F = const_cast<double *>(a.src[f]);
    const int w0 = j == 1 ? 0 : j, w1 = j == g.n2m ? j + 1 : j;
    for (int jj = w0; jj <= w1; jj++) {
        const size_t q = g.ix(i, jj, k);
        const double v = F[q];
        S[q] = v;
        g.images(F, i, k, q, v);
        g.images(S, i, k, q, v);
    }
}

// ADI of one increment (or of T), forward: the three solutions into X[0..2],
// each solve from the one before it
template <class RZ, class RX, class RY>
static int adi_forward(tcs_ctx *c, const RZ &rz, const RX &rx, const RY &ry, int jlo, double *const (&X)[3]) {
    double *am = c->am, *ac = c->ac, *ap = c->ap;
    TCS_TRY(rows3d_launch<true>(c, "adj_fwd_rows", rz, jlo, am, ac, ap, X[0]));
    TCS_TRY(sweep(c, am, ac, ap, X[0], X[0], 2, jlo, true));
    TCS_TRY(rows3d_launch<false>(c, "adj_fwd_rows", rx, jlo, am, ac, ap, X[1]));
    TCS_TRY(sweep(c, am, ac, ap, X[0], X[1], 0, jlo, true));
    TCS_TRY(rows3d_launch<false>(c, "adj_fwd_rows", ry, jlo, am, ac, ap, X[2]));
    TCS_TRY(sweep(c, am, ac, ap, X[1], X[2], 1, jlo, false));
    return TCS_OK;
}

// T, dW, the tables, the stale scalars and dP keep the values that the
// backward pass needs until the step's end; what is overwritten is copied.
// (A copy and a solve's right-hand side or increment moved by launches of
// their own, and the adjoints' folds, packs and clears likewise: 286 kernels
// and copies a step, 139 now; a backward step at 32x45x64 0.91 -> 0.52 ms, at
// 128^3 4.84 -> 3.76 ms, the transposed systems split as the forward ones are.)
static int forward_keep(tcs_ctx *c, AdjWork *w, double dt) {
    const Grid g = c->grid();
    double **f = c->f;
    {
        Arrays a;
        for (int s = 0; s < NSTATE; s++) a.add(w->s0[s], f[STATE_IDS[s]], c->nfull);
        TCS_TRY(copy_arrays(c, a));
    }
    // thermal
    TCS_TRY(adi_forward(c, ThermalZ{g, c->phys, dt, f[TCS_T], f[TCS_U], f[TCS_V], f[TCS_W], c->wall[TCS_TBCUP],
                                    c->wall[TCS_TBCBT]},
                        ThermalX{g, c->phys, dt, f[TCS_T], f[TCS_U]}, ThermalY{g, c->phys, dt, f[TCS_T], f[TCS_V]}, 1,
                        w->X[STG_T]));
    TCS_TRY(store_keep<2>(c, 1, w->X[STG_T][2], f[TCS_T], nullptr));
    TCS_TRY(momentum_coeffi(c));
    // solvedU
    TCS_TRY(adi_forward(c, DUZ{g, c->phys, dt, f[TCS_U], f[TCS_V], f[TCS_W], f[TCS_P], f[TCS_T], f[TCS_MU],
                               f[TCS_INVRHO], c->wall[TCS_UBCUP], c->wall[TCS_UBCBT], c->wall[TCS_VBCUP],
                               c->wall[TCS_VBCBT]},
                        DUX{g, c->phys, dt, f[TCS_U], f[TCS_MU], f[TCS_INVRHO]},
                        DUY{g, c->phys, dt, f[TCS_V], f[TCS_MU], f[TCS_INVRHO]}, 1, w->X[STG_U]));
    TCS_TRY(store_keep<1>(c, 1, w->X[STG_U][2], f[TCS_DU], w->sdU1));
    // solvedV (rows j >= 2)
    TCS_TRY(adi_forward(c, DVZ{g, c->phys, dt, f[TCS_U], f[TCS_V], f[TCS_W], f[TCS_P], f[TCS_DU], f[TCS_MU],
                               f[TCS_INVRHO], c->wall[TCS_VBCUP], c->wall[TCS_VBCBT]},
                        DVX{g, c->phys, dt, f[TCS_U], f[TCS_INVRHO], c->stale},
                        DVY{g, c->phys, dt, f[TCS_V], f[TCS_MU], f[TCS_INVRHO]}, 2, w->X[STG_V]));
    TCS_TRY(store_keep<1>(c, 2, w->X[STG_V][2], f[TCS_DV], w->sdV1));
    // solvedW
    TCS_TRY(adi_forward(c, DWZ{g, c->phys, dt, f[TCS_U], f[TCS_V], f[TCS_W], f[TCS_P], f[TCS_DU], f[TCS_DV],
                               f[TCS_MU], f[TCS_INVRHO], c->wall[TCS_VBCUP], c->wall[TCS_VBCBT],
                               c->wall[TCS_WBCUP], c->wall[TCS_WBCBT]},
                        DWX{g, c->phys, dt, f[TCS_U], f[TCS_INVRHO], c->stale},
                        DWY{g, c->phys, dt, f[TCS_V], f[TCS_INVRHO], c->stale}, 1, w->X[STG_W]));
    TCS_TRY(store_keep<1>(c, 1, w->X[STG_W][2], f[TCS_DW], nullptr));
    // block corrections, pseudo-update
    TCS_TRY(momentum_blockLdV(c, dt));
    TCS_TRY(halo(c, f[TCS_DV]));
    TCS_TRY(momentum_blockLdU(c, dt));
    TCS_TRY(momentum_pseudoupdate(c));
    {
        Arrays a;
        a.add(w->sU1, f[TCS_U], c->nfull);
        a.add(w->sV1, f[TCS_V], c->nfull);
        a.add(w->sW1, f[TCS_W], c->nfull);
        TCS_LAUNCH(c->stream, "adj_fwd_keep", k_halo_keep, interior_grid(c->n1m, c->n2m, c->n3m * a.count),
                   interior_block(), 0, g, a);
    }
    // pressure
    TCS_TRY(pressure_rhs(c, dt));
    TCS_TRY(pressure_poisson(c));
    TCS_TRY(halo(c, f[TCS_DP]));
    TCS_TRY(pressure_projection(c, dt));
    return halo(c, {f[TCS_U], f[TCS_V], f[TCS_W], f[TCS_P], f[TCS_DPHAT]});
}

// ---- the step backwards ----------------------------------------------------------

// Before a cell update that overwrites fields' interior rows j >= jlo: their
// new adjoints (dst) start as the old ones (src) outside those cells
// (untouched values pass through) and zero inside (filled by the update's
// product).
__global__ void k_overwrite_begin(Grid g, int jlo, Arrays a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z % g.N3, f = blockIdx.z / g.N3;
    if (i >= g.N1 || j >= g.N2) return;
    const bool in = i >= 1 && i <= g.n1m && j >= jlo && j <= g.n2m && k >= 1 && k <= g.n3m;
    const size_t q = g.ix(i, j, k);
    a.dst[f][q] = in ? 0.0 : a.src[f][q];
}
static int overwrite_begin(tcs_ctx *c, int jlo, std::initializer_list<std::pair<double *, const double *>> fields) {
    Arrays a;
    for (const auto &f : fields) a.add(f.first, f.second, c->nfull);
    TCS_LAUNCH(c->stream, "adj_begin", k_overwrite_begin, interior_grid(c->N1, c->N2, c->N3 * a.count),
               interior_block(), 0, c->grid(), jlo, a);
    return TCS_OK;
}

template <bool ZERO>
static int take(tcs_ctx *c, int jlo, double *b, double *r) {
    TCS_LAUNCH(c->stream, "adj_take", k_take<ZERO>, interior_grid(c->n1m, c->n2m, c->n3m), interior_block(), 0,
               c->grid(), jlo, b, r);
    return TCS_OK;
}

static int backward(tcs_ctx *c, AdjWork *w, double dt) {
    const Grid g = c->grid();
    const dim3 blk = interior_block(), grd = interior_grid(c->n1m, c->n2m, c->n3m);
    double **b = w->b;
    const double *Mu = c->f[TCS_MU], *iR = c->f[TCS_INVRHO];
    const double *TBCup = c->wall[TCS_TBCUP], *TBCbt = c->wall[TCS_TBCBT];
    // halos after the projection
    TCS_TRY(halo_adj(c, {b[ST_DPHAT], b[ST_P], b[ST_W], b[ST_V], b[ST_U]}));
    // P wall extrapolation; dPhat / dP0 history; projection
    TCS_TRY(wall_extrap_adj(c, b[ST_P]));
    {
        const DPhatUpdate cell{g, c->f[TCS_DP], w->s0[ST_DPHAT], w->s0[ST_DP0]};
        TCS_TRY(overwrite_begin(c, 1, {{w->tmp[0], b[ST_DPHAT]}, {w->tmp[1], b[ST_DP0]}}));
        TCS_TRY(cell_vjp(c, w, cell, 1, OutBars{{b[ST_DPHAT], b[ST_DP0], nullptr, nullptr}, 1},
                         InBars<3>{{w->bdP, w->tmp[0], w->tmp[1]}}));
        std::swap(b[ST_DPHAT], w->tmp[0]);
        std::swap(b[ST_DP0], w->tmp[1]);
    }
    {
        const Projection cell{g, c->phys, dt, iR, c->f[TCS_DP], w->s0[ST_DPHAT], w->s0[ST_DP0],
                              w->sU1, w->sV1, w->sW1, w->s0[ST_P]};
        TCS_TRY(overwrite_begin(c, 1, {{w->tmp[0], b[ST_U]}, {w->tmp[1], b[ST_V]}, {w->tmp[2], b[ST_W]},
                                       {w->tmp[3], b[ST_P]}}));
        TCS_TRY(cell_vjp(c, w, cell, 1, OutBars{{b[ST_U], b[ST_V], b[ST_W], b[ST_P]}, 1},
                         InBars<8>{{w->biR, w->bdP, b[ST_DPHAT], b[ST_DP0], w->tmp[0], w->tmp[1], w->tmp[2],
                                    w->tmp[3]}}));
        for (int q = 0; q < 4; q++) std::swap(b[ST_U + q], w->tmp[q]);
    }
    // Poisson: halo(dP), wall extrapolation, mean, then the transposed solve
    TCS_TRY(halo_adj(c, {w->bdP}));
    TCS_TRY(wall_extrap_adj(c, w->bdP));
    TCS_LAUNCH(c->stream, "adj_mean", k_interior_mean, dim3((unsigned)std::min<size_t>(SUM_BLOCKS, (c->nint + 2047) / 2048)),
               dim3(256), 0, g, w->bdP, w->psum);
    TCS_LAUNCH(c->stream, "adj_take_mean", k_take_mean, grd, blk, 0, g, w->psum + SUM_BLOCKS, w->bdP, w->rint);
    {
        const int n2m = c->n2m, n3m = c->n3m, h1p = c->h1p;
        double2 *spec = (double2 *)c->spec_x;
        TCS_TRY(fft_x_fwd_launch(c, "adj_fft_x_fwd", w->rint, spec));
        TCS_TRY(fft_z_launch<-1>(c, "adj_fft_z", spec));
        const int nsys = n3m * h1p;
        TCS_LAUNCH(c->stream, "adj_poisson_T", k_poisson_tdma_T, dim3((nsys + 63) / 64), dim3(64), 0, n3m, h1p, n2m,
                   c->h3p, c->ptab, c->ptab + n2m, c->ptab + 2 * n2m, c->dxk2, c->dzk, spec, c->pC);
        TCS_TRY(fft_z_launch<+1>(c, "adj_fft_z", spec));
        TCS_TRY(fft_x_inv_launch(c, "adj_fft_x_inv", spec, w->tmp[0]));
    }
    // pressure right-hand side
    {
        const PressureRHS cell{g, c->phys, dt, w->sU1, w->sV1, w->sW1, w->s0[ST_DPHAT], iR,
                               c->wall[TCS_VBCUP], c->wall[TCS_VBCBT]};
        TCS_TRY(cell_vjp(c, w, cell, 1, OutBars{{w->tmp[0], nullptr, nullptr, nullptr}, 1},
                         InBars<7>{{b[ST_U], b[ST_V], b[ST_W], b[ST_DPHAT], w->biR, nullptr, nullptr}}));
    }
    // halos of U, V, W; pseudo-update
    TCS_TRY(halo_adj(c, {b[ST_W], b[ST_V], b[ST_U]}));
    TCS_LAUNCH(c->stream, "adj_pseudo", k_pseudo_adj, grd, blk, 0, g, b[ST_U], b[ST_V], b[ST_W], w->bdU, w->bdV,
               w->bdW);
    // blockLdU, halo(dV), blockLdV, halo(dW)
    {
        const BlockLdU cell{g, c->phys, dt, w->s0[ST_U], c->f[TCS_DV], c->f[TCS_DW], Mu, iR, w->sdU1};
        TCS_TRY(overwrite_begin(c, 1, {{w->tmp[0], w->bdU}}));
        TCS_TRY(cell_vjp(c, w, cell, 1, OutBars{{w->bdU, nullptr, nullptr, nullptr}, 1},
                         InBars<6>{{b[ST_U], w->bdV, w->bdW, w->bMu, w->biR, w->tmp[0]}}));
        std::swap(w->bdU, w->tmp[0]);
    }
    TCS_TRY(halo_adj(c, {w->bdV}));
    {
        const BlockLdV cell{g, c->phys, dt, w->s0[ST_V], c->f[TCS_DW], Mu, iR, w->sdV1};
        TCS_TRY(overwrite_begin(c, 2, {{w->tmp[0], w->bdV}}));
        TCS_TRY(cell_vjp(c, w, cell, 2, OutBars{{w->bdV, nullptr, nullptr, nullptr}, 1},
                         InBars<5>{{b[ST_V], w->bdW, w->bMu, w->biR, w->tmp[0]}}));
        std::swap(w->bdV, w->tmp[0]);
    }
    // solvedW: dW's interior is the y stage's solution
    TCS_TRY(take<true>(c, 1, w->bdW, w->lam));
    {
        const DWZ rz{g, c->phys, dt, w->s0[ST_U], w->s0[ST_V], w->s0[ST_W], w->s0[ST_P], w->sdU1, w->sdV1, Mu,
                     iR, c->wall[TCS_VBCUP], c->wall[TCS_VBCBT], c->wall[TCS_WBCUP], c->wall[TCS_WBCBT]};
        const DWX rx{g, c->phys, dt, w->s0[ST_U], iR, c->stale};
        const DWY ry{g, c->phys, dt, w->s0[ST_V], iR, c->stale};
        TCS_TRY(stage_adj<false>(c, w, ry, 1, 1, false, w->X[STG_W][2], InBars<3>{{b[ST_V], w->biR, w->bstale}}));
        TCS_TRY(stage_adj<false>(c, w, rx, 0, 1, true, w->X[STG_W][1], InBars<3>{{b[ST_U], w->biR, w->bstale}}));
        TCS_TRY(stage_adj<true>(c, w, rz, 2, 1, true, w->X[STG_W][0],
                                InBars<12>{{b[ST_U], b[ST_V], b[ST_W], b[ST_P], w->bdU, w->bdV, w->bMu, w->biR,
                                            nullptr, nullptr, nullptr, nullptr}}));
    }
    // solvedV: rows j >= 2; dV's other rows are zeroed in the forward step
    TCS_TRY(take<true>(c, 2, w->bdV, w->lam));
    {
        const DVZ rz{g, c->phys, dt, w->s0[ST_U], w->s0[ST_V], w->s0[ST_W], w->s0[ST_P], w->sdU1, Mu, iR,
                     c->wall[TCS_VBCUP], c->wall[TCS_VBCBT]};
        const DVX rx{g, c->phys, dt, w->s0[ST_U], iR, c->stale};
        const DVY ry{g, c->phys, dt, w->s0[ST_V], Mu, iR};
        TCS_TRY(stage_adj<false>(c, w, ry, 1, 2, false, w->X[STG_V][2], InBars<3>{{b[ST_V], w->bMu, w->biR}}));
        TCS_TRY(stage_adj<false>(c, w, rx, 0, 2, true, w->X[STG_V][1], InBars<3>{{b[ST_U], w->biR, w->bstale}}));
        TCS_TRY(stage_adj<true>(c, w, rz, 2, 2, true, w->X[STG_V][0],
                                InBars<9>{{b[ST_U], b[ST_V], b[ST_W], b[ST_P], w->bdU, w->bMu, w->biR, nullptr,
                                           nullptr}}));
    }
    // solvedU
    TCS_TRY(take<true>(c, 1, w->bdU, w->lam));
    {
        const DUZ rz{g, c->phys, dt, w->s0[ST_U], w->s0[ST_V], w->s0[ST_W], w->s0[ST_P], c->f[TCS_T], Mu, iR,
                     c->wall[TCS_UBCUP], c->wall[TCS_UBCBT], c->wall[TCS_VBCUP], c->wall[TCS_VBCBT]};
        const DUX rx{g, c->phys, dt, w->s0[ST_U], Mu, iR};
        const DUY ry{g, c->phys, dt, w->s0[ST_V], Mu, iR};
        TCS_TRY(stage_adj<false>(c, w, ry, 1, 1, false, w->X[STG_U][2], InBars<3>{{b[ST_V], w->bMu, w->biR}}));
        TCS_TRY(stage_adj<false>(c, w, rx, 0, 1, true, w->X[STG_U][1], InBars<3>{{b[ST_U], w->bMu, w->biR}}));
        TCS_TRY(stage_adj<true>(c, w, rz, 2, 1, true, w->X[STG_U][0],
                                InBars<11>{{b[ST_U], b[ST_V], b[ST_W], b[ST_P], b[ST_T], w->bMu, w->biR, nullptr,
                                            nullptr, nullptr, nullptr}}));
    }
    // stale viscosities and the Mu / invRho tables (from T after the thermal stage)
    TCS_LAUNCH(c->stream, "adj_stale", k_stale_adj, dim3(1), dim3(64), 0, g, Mu, w->bstale, w->bMu);
    TCS_LAUNCH(c->stream, "adj_coeffi", k_coeffi_adj, dim3((c->N2 + 63) / 64, c->N3), dim3(64), 0, g, c->phys, c->f[TCS_T],
               w->bMu, w->biR, b[ST_T]);
    // thermal: T1 = T0 + x3 on the interior
    TCS_TRY(take<false>(c, 1, b[ST_T], w->lam));
    {
        const ThermalZ rz{g, c->phys, dt, w->s0[ST_T], w->s0[ST_U], w->s0[ST_V], w->s0[ST_W], TBCup, TBCbt};
        const ThermalX rx{g, c->phys, dt, w->s0[ST_T], w->s0[ST_U]};
        const ThermalY ry{g, c->phys, dt, w->s0[ST_T], w->s0[ST_V]};
        TCS_TRY(stage_adj<false>(c, w, ry, 1, 1, false, w->X[STG_T][2], InBars<2>{{b[ST_T], b[ST_V]}}));
        TCS_TRY(stage_adj<false>(c, w, rx, 0, 1, true, w->X[STG_T][1], InBars<2>{{b[ST_T], b[ST_U]}}));
        TCS_TRY(stage_adj<true>(c, w, rz, 2, 1, true, w->X[STG_T][0],
                                InBars<6>{{b[ST_T], b[ST_U], b[ST_V], b[ST_W], w->bwall[TCS_TBCUP],
                                           w->bwall[TCS_TBCBT]}}));
    }
    // the step's own tables and scalars start from zero next time
    Arrays z;
    z.add(w->bMu, nullptr, c->ntab);
    z.add(w->biR, nullptr, c->ntab);
    z.add(w->bstale, nullptr, REV_STALE * REV_STALE_STRIDE);
    return copy_arrays(c, z);
}

}  // namespace adj

void adjoint_free(tcs_ctx *c) {
    if (!c->adj) return;
    for (void *p : c->adj->all) (void)hipFree(p);
    delete c->adj;
    c->adj = nullptr;
}

static int adjoint_alloc(tcs_ctx *c) {
    if (c->adj) return TCS_OK;
    AdjWork *w = new AdjWork();
    c->adj = w;
    // full fields get the step's layout (FIELD_FRONT elements in front)
    auto get = [&](double **p, size_t n) -> int {
        const size_t front = n == c->nfull ? FIELD_FRONT + 1 : 0;
        void *q = nullptr;
        if (hipMalloc(&q, (std::max<size_t>(n, 1) + front) * sizeof(double)) != hipSuccess) return TCS_E_HIP;
        w->all.push_back(q);
        if (hipMemset(q, 0, (std::max<size_t>(n, 1) + front) * sizeof(double)) != hipSuccess) return TCS_E_HIP;
        *p = (double *)q + (front ? FIELD_FRONT : 0);
        return TCS_OK;
    };
    int rc = TCS_OK;
    for (int s = 0; s < adj::NSTATE && rc == TCS_OK; s++) rc |= get(&w->b[s], c->nfull) | get(&w->s0[s], c->nfull);
    for (double **p : {&w->bdU, &w->bdV, &w->bdW, &w->bdP, &w->sdU1, &w->sdV1, &w->sU1, &w->sV1, &w->sW1, &w->tmp[0],
                        &w->tmp[1], &w->tmp[2], &w->tmp[3]})
        rc |= get(p, c->nfull);
    for (double **p : {&w->bMu, &w->biR}) rc |= get(p, c->ntab);
    rc |= get(&w->bstale, (size_t)REV_STALE * REV_STALE_STRIDE) | get(&w->psum, adj::SUM_BLOCKS + 2);
    for (int q = 0; q < TCS_NWALL; q++) rc |= get(&w->bwall[q], c->nwall);
    for (int s = 0; s < 4; s++)
        for (int q = 0; q < 3; q++) rc |= get(&w->X[s][q], c->nint);
    for (double **p : {&w->lam, &w->rint}) rc |= get(p, c->nint);
    if (rc != TCS_OK) {
        adjoint_free(c);
        set_error("tcs_adjoint: device allocation failed");
        return TCS_E_HIP;
    }
    return TCS_OK;
}

}  // namespace tcs

using namespace tcs;

extern "C" int tcs_adjoint_zero(tcs_ctx *c) {
    if (!c) return TCS_E_ARG;
    TCS_TRY(flush_pending(c));
    TCS_TRY(adjoint_alloc(c));
    AdjWork *w = c->adj;
    adj::Arrays z;
    static_assert(adj::NSTATE + TCS_NWALL + 4 <= adj::Arrays::MAX, "one launch");
    for (int s = 0; s < adj::NSTATE; s++) z.add(w->b[s], nullptr, c->nfull);
    for (int q = 0; q < TCS_NWALL; q++) z.add(w->bwall[q], nullptr, c->nwall);
    for (double *p : {w->bdU, w->bdV, w->bdW, w->bdP}) z.add(p, nullptr, c->nfull);
    return adj::copy_arrays(c, z);
}

static double *adjoint_array(tcs_ctx *c, int32_t kind, int32_t id, size_t &n) {
    AdjWork *w = c->adj;
    if (kind == 0) {
        for (int s = 0; s < adj::NSTATE; s++)
            if (adj::STATE_IDS[s] == id) {
                n = c->nfull;
                return w->b[s];
            }
        return nullptr;
    }
    if (kind == 1 && id >= 0 && id < TCS_NWALL) {
        n = c->nwall;
        return w->bwall[id];
    }
    return nullptr;
}

extern "C" int tcs_adjoint_copy(tcs_ctx *c, int32_t kind, int32_t id, int32_t to_adjoint, double *dev) {
    if (!c || !dev) return TCS_E_ARG;
    TCS_TRY(flush_pending(c));
    TCS_TRY(adjoint_alloc(c));
    size_t n = 0;
    double *a = adjoint_array(c, kind, id, n);
    if (!a) {
        set_error("tcs_adjoint_copy: kind 0 takes a state field id (T, U, V, W, P, dPhat, dP0), kind 1 a wall id");
        return TCS_E_ARG;
    }
    if (kind == 0) {
        // dev holds the reference layout (rows N1 apart), the adjoint field rows P1 apart
        const size_t pd = (size_t)c->N1 * sizeof(double), pa = (size_t)c->P1 * sizeof(double);
        const size_t rows = (size_t)c->N2 * c->N3;
        if (to_adjoint) TCS_HIP(hipMemcpy2DAsync(a, pa, dev, pd, pd, rows, hipMemcpyDeviceToDevice, c->stream));
        else TCS_HIP(hipMemcpy2DAsync(dev, pd, a, pa, pd, rows, hipMemcpyDeviceToDevice, c->stream));
        return TCS_OK;
    }
    if (to_adjoint) TCS_HIP(hipMemcpyAsync(a, dev, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    else TCS_HIP(hipMemcpyAsync(dev, a, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    return TCS_OK;
}

extern "C" int tcs_adjoint_add_nusselt(tcs_ctx *c, double weight, double Tup, double Tbt) {
    if (!c) return TCS_E_ARG;
    TCS_TRY(flush_pending(c));
    TCS_TRY(adjoint_alloc(c));
    const Grid g = c->grid();
    const double wgt = weight * c->prm.L2 / (Tbt - Tup) / c->h_dmx2[1] / ((double)c->n1m * (double)c->n3m);
    TCS_LAUNCH(c->stream, "adj_nusselt", adj::k_nusselt_adj, dim3((c->n1m + 63) / 64, c->n3m), dim3(64), 0, g, wgt,
               c->adj->b[adj::ST_T], c->adj->bwall[TCS_TBCBT]);
    return TCS_OK;
}

extern "C" int tcs_adjoint_step(tcs_ctx *c, double dt) {
    if (!c) return TCS_E_ARG;
    TCS_TRY(flush_pending(c));
    if (c->prm.precision != 0) {
        set_error("tcs_adjoint_step: the adjoint differentiates the plain FP64 step (precision 0)");
        return TCS_E_ARG;
    }
    if (c->nfull + FIELD_FRONT + 1 > ((size_t)1 << 28)) {  // the interface's limit
        set_error("tcs_adjoint_step: the full fields must hold fewer than 2^28 values");
        return TCS_E_ARG;
    }
    TCS_TRY(adjoint_alloc(c));
    c->cfl_valid = 0;
    TCS_TRY(adj::forward_keep(c, c->adj, dt));
    TCS_TRY(adj::backward(c, c->adj, dt));
    // the step is over when the entry returns: buffers given to
    // tcs_adjoint_copy before it may be written again, and a device error is
    // this call's
    TCS_HIP(hipStreamSynchronize(c->stream));
    return TCS_OK;
}
