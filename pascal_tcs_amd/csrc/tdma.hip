// tdma.hip -- batched tridiagonal solves with PaScaL_TDMA's single-rank
// operation order (PaScaL_TDMA/src/pascal_tdma.f90:487-578 and :715-806,
// reduced 2-row solves of PaScaL_TDMA/src/tdmas.f90:113-212).
//
// The kernels here move rows between memory and the one-lane lines of
// tdma_exact.h.
#include "tdma_exact.h"

#include <mutex>

namespace tcs {

namespace {

using namespace exact_line;

// Lines strided in memory: line l = s0 + n0*s1 starts at s0*ss0 + s1*ss1,
// rows rs apart.  A, C and Dout also hold the eliminated rows j < jl (the
// rows j >= jl are kept in LDS); KEEP: A and C come back as the reference
// leaves them.  FIELD: the solution goes into the field of out (stored) and
// not into Dout, with its ghosts and wall rows where out asks for them (the
// momentum y stages of the single-rank order; by a kernel of its own the
// stores took 50 us a stage at 256x200x256).
template <bool CYC, bool KEEP, bool FIELD = false>
__global__ void __launch_bounds__(EX_W)
k_ptdma_exact(double *A, const double *B, double *C, const double *Din, double *Dout, int n0, long ss0, long ss1,
              long lines, int n_row, long rs, int jl, LineOut out) {
    extern __shared__ double lds[];
    const Kept<1> keep{lds, (int)threadIdx.x};
    const long line = (long)blockIdx.x * EX_W + threadIdx.x;
    if (line >= lines) return;  // no barrier below: a lane reads only what it wrote
    const long s1 = line / n0, base = (line - s1 * n0) * ss0 + s1 * ss1;
    double *a = A + base, *c = C + base, *d = Dout + base;
    const double *b = B + base, *din = Din + base;
    const long s0 = line - s1 * n0, fb = out.base + s0 * out.ss0 + s1 * out.ss1;
    long di = 0, dk = 0;
    if (FIELD && out.gx > 0) {
        di = s0 == 0 ? out.gx * out.ss0 : s0 == out.gx - 1 ? -out.gx * out.ss0 : 0;
        dk = s1 == 0 ? out.gz * out.ss1 : s1 == out.gz - 1 ? -out.gz * out.ss1 : 0;
    }
    solve<CYC, 1>(
        n_row,
        [&](int j) {
            const long o = (long)j * rs;
            return Row<1>{a[o], b[o], c[o], {din[o]}};
        },
        [&](int j, const Elim<1> &e) {
            if (j >= jl) {
                keep.put(j - jl, e);
            } else {
                const long o = (long)j * rs;
                a[o] = e.a; c[o] = e.c; d[o] = e.d[0];
            }
        },
        [&](int j) {
            if (j >= jl) return keep.get(j - jl);
            const long o = (long)j * rs;
            return Elim<1>{a[o], c[o], {d[o]}};
        },
        [&](int j, const Elim<1> &e, const double (&x)[1]) {
            const long o = (long)j * rs;
            if constexpr (FIELD) part::put_line<double>(out.F, fb + (long)j * out.rs, x[0], di, dk);
            else d[o] = x[0];
            if constexpr (KEEP) { a[o] = e.a; c[o] = e.c; }
        });
    if (FIELD && out.gx > 0) {
        const long lo = fb - out.rs, hi = fb + (long)n_row * out.rs;
        part::put_line<double>(out.F, lo, out.F[lo], di, dk);
        part::put_line<double>(out.F, hi, out.F[hi], di, dk);
    }
}

// Systems whose rows are contiguous in memory (the x sweep of an (i,j,k)
// array): line (s0, s1) starts at s0*ss0 + s1*ss1.  The rows come in chunks
// of EX_R of the workgroup's 64 lines, loaded along the lines (128-byte
// segments) one chunk ahead and turned through LDS, so each lane still walks
// its own line.  The eliminated rows of a chunk go back to the chunk's own
// memory in the order of the lanes (lane l of row r is value r*64 + l of the
// chunk), where the backward passes read them without turning; only the
// solution (and with KEEP a and c) is turned back.
template <bool CYC, bool KEEP>
__global__ void __launch_bounds__(EX_W)
k_ptdma_exact_rows(double *A, const double *B, double *C, const double *Din, double *Dout, int n0, long ss0,
                   long ss1, int n_row) {
    constexpr int P = EX_R + 1;  // padded row of the tile
    __shared__ double tile[4][EX_W * P];
    const int lane = threadIdx.x;
    const int s0a = blockIdx.x * EX_W;
    const int nl = min(EX_W, n0 - s0a);  // lines here
    const long lb = (long)s0a * ss0 + (long)blockIdx.y * ss1;
    const bool act = lane < nl;
    const int nch = (n_row + EX_R - 1) / EX_R;
    double *TA = tile[0] + lane * P, *TB = tile[1] + lane * P, *TC = tile[2] + lane * P, *TD = tile[3] + lane * P;
    const int ql = lane / EX_R, qr = lane % EX_R;  // along the lines: line 4q + ql, row qr of the chunk
    // value (r, lane) of the chunk at row r0 with nr rows; the last, shorter one
    // stays in its lines' order (packing it, or fewer lines, by divisions took
    // a third of the time: 647 us a line of 1000 rows, 414 now)
    auto spot = [&](int r0, int nr, int r) {
        if (nr < EX_R) return lb + (long)lane * ss0 + r0 + r;
        if (nl == EX_W) return lb + (long)(r * 4 + ql) * ss0 + r0 + qr;
        const unsigned v = r * nl + lane;
        return lb + (long)(v / EX_R) * ss0 + r0 + v % EX_R;
    };
    double va[EX_R], vb[EX_R], vc[EX_R], vd[EX_R];
    auto fetch = [&](int ch) {  // a chunk's rows into registers, along the lines
        const int r0 = ch * EX_R;
#pragma unroll
        for (int q = 0; q < EX_R; q++) {
            const int l = q * 4 + ql;
            if (l < nl && r0 + qr < n_row) {
                const long o = lb + (long)l * ss0 + r0 + qr;
                va[q] = A[o]; vb[q] = B[o]; vc[q] = C[o]; vd[q] = Din[o];
            }
        }
    };
    Elim<1> e0{}, e1{}, p{}, pp{};
    fetch(0);
    for (int ch = 0; ch < nch; ch++) {
        const int r0 = ch * EX_R, nr = min(EX_R, n_row - r0);
#pragma unroll
        for (int q = 0; q < EX_R; q++) {
            const int o = (q * 4 + ql) * P + qr;
            tile[0][o] = va[q]; tile[1][o] = vb[q]; tile[2][o] = vc[q]; tile[3][o] = vd[q];
        }
        __syncthreads();
        if (ch + 1 < nch) fetch(ch + 1);
        if (act) {
            auto row = [&](int r) {
                const int j = r0 + r;
                const Row<1> w{TA[r], TB[r], TC[r], {TD[r]}};
                pp = p;
                if (j >= 2) {
                    p = fwd_row<1>(w, p);
                } else {
                    p = first_row<1>(w);
                    if (j == 0) e0 = p;
                    else e1 = p;
                }
                const long o = spot(r0, nr, r);
                A[o] = p.a; C[o] = p.c; Dout[o] = p.d[0];
            };
            if (nr == EX_R) {
#pragma unroll
                for (int r = 0; r < EX_R; r++) row(r);
            } else {
                for (int r = 0; r < nr; r++) row(r);
            }
        }
        __syncthreads();
    }
    const Elim<1> eN = p, eT = n_row >= 3 ? pp : e1;

    double x1[1] = {0.0}, xn[1] = {0.0};
    auto backward = [&](auto out) {
        constexpr bool OUT = decltype(out)::value;
        Elim<1> x = eT, q[EX_R];
        auto get = [&](int ch) {
            const int r0 = ch * EX_R, nr = min(EX_R, n_row - r0);
#pragma unroll
            for (int r = 0; r < EX_R; r++)
                if (act && r < nr) {
                    const long o = spot(r0, nr, r);
                    q[r].a = A[o]; q[r].c = C[o]; q[r].d[0] = Dout[o];
                }
        };
        get(nch - 1);
        for (int ch = nch - 1; ch >= 0; ch--) {
            const int r0 = ch * EX_R, nr = min(EX_R, n_row - r0);
            Elim<1> w[EX_R];
#pragma unroll
            for (int r = 0; r < EX_R; r++) w[r] = q[r];
            if (ch > 0) get(ch - 1);
#pragma unroll
            for (int r = EX_R - 1; r >= 0; r--) {
                const int j = r0 + r;
                if (r >= nr) continue;
                if (j >= 1 && j <= n_row - 3) x = back_row<1>(w[r], x);
                if constexpr (OUT) {
                    double v = x.d[0] - x.a * x1[0] - x.c * xn[0], ka = x.a, kc = x.c;
                    if (j == n_row - 1) { v = xn[0]; ka = eN.a; kc = eN.c; }
                    if (j == 0) { v = x1[0]; ka = e0.a; kc = e0.c; }
                    TD[r] = v;
                    if constexpr (KEEP) { TA[r] = ka; TC[r] = kc; }
                }
            }
            if constexpr (OUT) {
                // every lane has its own rows of this chunk in registers before
                // the solution takes their place in memory
                __syncthreads();
#pragma unroll
                for (int u = 0; u < EX_R; u++) {
                    const int l = u * 4 + ql, o = l * P + qr;
                    if (l < nl && qr < nr) {
                        const long t = lb + (long)l * ss0 + r0 + qr;
                        Dout[t] = tile[3][o];
                        if constexpr (KEEP) { A[t] = tile[0][o]; C[t] = tile[2][o]; }
                    }
                }
                __syncthreads();
            }
        }
        return x;
    };
    const Elim<1> x2 = backward(std::integral_constant<bool, false>());
    line_ends<CYC, 1>(e0, x2, eN, x1, xn);
    backward(std::integral_constant<bool, true>());
}

}  // namespace

int ptdma_exact_launch(double *A, const double *B, double *C, const double *Din, double *Dout, int n0, long ss0,
                       int n1, long ss1, int n_row, long rs, bool cyclic, bool keep, hipStream_t st,
                       const LineOut &out) {
    if (n0 <= 0 || n1 <= 0) return TCS_OK;
    if (n_row < 2 || n1 > 65535) {
        set_error("ptdma: n_row must be >= 2 and the outer system count <= 65535");
        return TCS_E_ARG;
    }
#define EXACT_PICK(kern) \
    (cyclic ? (keep ? kern<true, true> : kern<true, false>) : (keep ? kern<false, true> : kern<false, false>))
    const bool field = out.mode == 1;
    if (out.mode != 0 && (!field || rs == 1 || cyclic || keep)) {
        set_error("ptdma: field output is stored from non-cyclic strided lines only");
        return TCS_E_ARG;
    }
    if (rs == 1) {
        // planes of few lines without gaps between them are one plane, so that
        // workgroups are full (3000 planes of 1 line of 301 rows 493 us, now
        // 167; of 5 lines 557, 221; above half a workgroup's lines a plane
        // what is saved may go into a last round of a few workgroups: 2000
        // planes of 33 lines of 33 rows 92 us, 120 as one)
        if (2 * n0 <= EX_W && ss1 == (long)n0 * ss0 && (long)n0 * n1 <= INT32_MAX) {
            n0 *= n1;
            n1 = 1;
        }
        const dim3 grd((unsigned)((n0 + EX_W - 1) / EX_W), (unsigned)n1);
        TCS_LAUNCH(st, cyclic ? "ptdma_rows_cyclic" : "ptdma_rows", EXACT_PICK(k_ptdma_exact_rows), grd, dim3(EX_W),
                   0, A, B, C, Din, Dout, n0, ss0, ss1, n_row);
        return TCS_OK;
    }
    const long lines = (long)n0 * n1;
    const int kept = kept_rows<1>(lines, n_row), lds = kept * Kept<1>::ROW_BYTES;
    const auto kern = field ? k_ptdma_exact<false, false, true> : EXACT_PICK(k_ptdma_exact);
    static DeviceSet raised[5];
    TCS_TRY(lds_limit((const void *)kern, KEPT_LDS, raised[field ? 4 : 2 * cyclic + keep]));
    TCS_LAUNCH(st, cyclic ? "ptdma_cyclic" : "ptdma", kern, dim3((unsigned)((lines + EX_W - 1) / EX_W)), dim3(EX_W),
               lds, A, B, C, Din, Dout, n0, ss0, ss1, lines, n_row, rs, n_row - kept, out);
#undef EXACT_PICK
    return TCS_OK;
}

}  // namespace tcs

using namespace tcs;

static int many_solve(double *A, const double *B, double *C, double *D, int32_t n_sys,
                      int32_t n_row, bool cyc, void *stream) {
    if (!A || !B || !C || !D || n_sys < 0 || n_row < 2) {
        set_error("ptdma_many_solve: null pointer or n_row < 2");
        return TCS_E_ARG;
    }
    // (n_sys, n_row): the systems adjacent, their rows n_sys apart
    if (n_sys == 1)  // one system: its rows are contiguous
        return ptdma_exact_launch(A, B, C, D, D, 1, 1, 1, 0, n_row, 1, cyc, true, (hipStream_t)stream);
    return ptdma_exact_launch(A, B, C, D, D, n_sys, 1, 1, 0, n_row, n_sys, cyc, true, (hipStream_t)stream);
}

extern "C" int ptdma_many_solve_dev(double *A, const double *B, double *C, double *D, int32_t n_sys,
                                    int32_t n_row, void *stream) {
    return many_solve(A, B, C, D, n_sys, n_row, false, stream);
}

extern "C" int ptdma_many_solve_cycle_dev(double *A, const double *B, double *C, double *D,
                                          int32_t n_sys, int32_t n_row, void *stream) {
    return many_solve(A, B, C, D, n_sys, n_row, true, stream);
}

extern "C" int ptdma_many_solve_host(double *A, double *B, double *C, double *D, int32_t n_sys,
                                     int32_t n_row, int32_t cyclic) {
    if (!A || !B || !C || !D || n_sys <= 0 || n_row < 2) {
        set_error("ptdma_many_solve_host: bad arguments");
        return TCS_E_ARG;
    }
    size_t bytes = (size_t)n_sys * (size_t)n_row * sizeof(double);
    double *d[4] = {nullptr, nullptr, nullptr, nullptr};
    double *h[4] = {A, B, C, D};
    int rc = TCS_OK;
    for (int q = 0; q < 4 && rc == TCS_OK; q++) {
        if (hipMalloc(&d[q], bytes) != hipSuccess) { set_error("hipMalloc failed"); rc = TCS_E_NOMEM; }
        else if (hipMemcpy(d[q], h[q], bytes, hipMemcpyHostToDevice) != hipSuccess) { set_error("H2D copy failed"); rc = TCS_E_HIP; }
    }
    if (rc == TCS_OK) rc = many_solve(d[0], d[1], d[2], d[3], n_sys, n_row, cyclic != 0, nullptr);
    if (rc == TCS_OK && hipDeviceSynchronize() != hipSuccess) { set_error("ptdma kernel failed"); rc = TCS_E_HIP; }
    if (rc == TCS_OK) {
        for (int q : {0, 2, 3})
            if (hipMemcpy(h[q], d[q], bytes, hipMemcpyDeviceToHost) != hipSuccess) { set_error("D2H copy failed"); rc = TCS_E_HIP; }
    }
    for (int q = 0; q < 4; q++)
        if (d[q]) (void)hipFree(d[q]);
    return rc;
}

// ---- host solve without device allocation ---------------------------------
// ptdma_many_solve_host stages the four host arrays in device buffers it
// allocates and frees on every call.  The variant below stages them in one
// file-scope device array instead (each GPU the library runs on holds its
// own copy until the process ends), so a caller that must not allocate --
// or that calls the solve plane by plane in a loop -- pays only the copies.
// Four arrays of at most NOALLOC_MAX doubles each (4 x 16 MiB).  Every call
// on a GPU shares that GPU's array: calls that overlap on one GPU (from
// several host threads) race.  The array needs no clearing: each call
// overwrites the part it uses before any kernel reads it.
constexpr size_t NOALLOC_MAX = (size_t)1 << 21;
static __device__ __align__(256) double scratch[4 * NOALLOC_MAX];

constexpr int NOALLOC_DEVICES = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[NOALLOC_DEVICES];  // device address of `scratch` per device

// the current device's address of `scratch`, looked up once per device
static int scratch_address(double **out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_DEVICES) {
        set_error("ptdma_many_solve_host_noalloc: no usable current device");
        return TCS_E_HIP;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error(std::string("ptdma_many_solve_host_noalloc: hipGetSymbolAddress failed: ") +
                      hipGetErrorString(e));
            return TCS_E_HIP;
        }
        g_scratch_ptr[dev] = (double *)p;
    }
    *out = g_scratch_ptr[dev];
    return TCS_OK;
}

extern "C" int ptdma_many_solve_host_noalloc(double *A, double *B, double *C, double *D, int32_t n_sys,
                                             int32_t n_row, int32_t cyclic) {
    if (!A || !B || !C || !D || n_sys <= 0 || n_row < 2) {
        set_error("ptdma_many_solve_host_noalloc: bad arguments");
        return TCS_E_ARG;
    }
    const size_t n = (size_t)n_sys * (size_t)n_row;
    if (n > NOALLOC_MAX) {
        set_error("ptdma_many_solve_host_noalloc: n_sys*n_row = " + std::to_string(n) + " exceeds the maximum " +
                  std::to_string(NOALLOC_MAX) + " of the static staging array (use ptdma_many_solve_host)");
        return TCS_E_ARG;
    }
    double *base = nullptr;
    TCS_TRY(scratch_address(&base));
    const size_t bytes = n * sizeof(double);
    double *d[4] = {base, base + NOALLOC_MAX, base + 2 * NOALLOC_MAX, base + 3 * NOALLOC_MAX};
    double *h[4] = {A, B, C, D};
    for (int q = 0; q < 4; q++)
        if (hipMemcpy(d[q], h[q], bytes, hipMemcpyHostToDevice) != hipSuccess) {
            set_error("ptdma_many_solve_host_noalloc: H2D copy failed");
            return TCS_E_HIP;
        }
    TCS_TRY(many_solve(d[0], d[1], d[2], d[3], n_sys, n_row, cyclic != 0, nullptr));
    if (hipStreamSynchronize(nullptr) != hipSuccess) {
        set_error("ptdma_many_solve_host_noalloc: kernel failed");
        return TCS_E_HIP;
    }
    for (int q : {0, 2, 3})
        if (hipMemcpy(h[q], d[q], bytes, hipMemcpyDeviceToHost) != hipSuccess) {
            set_error("ptdma_many_solve_host_noalloc: D2H copy failed");
            return TCS_E_HIP;
        }
    return TCS_OK;
}

extern "C" int ptdma_single_solve_dev(double *A, const double *B, double *C, double *D, int32_t n_row,
                                      int32_t cyclic, void *stream) {
    return many_solve(A, B, C, D, 1, n_row, cyclic != 0, stream);
}

extern "C" int ptdma_single_solve_host(double *A, double *B, double *C, double *D, int32_t n_row, int32_t cyclic) {
    return ptdma_many_solve_host(A, B, C, D, 1, n_row, cyclic);
}

extern "C" int ptdma_axis_solve_dev(double *A, const double *B, double *C, double *D, int32_t n1,
                                    int32_t n2, int32_t n3, int32_t axis, int32_t cyclic, void *stream) {
    if (!A || !B || !C || !D || n1 <= 0 || n2 <= 0 || n3 <= 0 || axis < 0 || axis > 2) {
        set_error("ptdma_axis_solve_dev: bad arguments");
        return TCS_E_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    long s1 = n1, s2 = (long)n1 * n2;
    switch (axis) {
    case 0:  // rows along i: systems (j,k)
        return ptdma_exact_launch(A, B, C, D, D, n2, s1, n3, s2, n1, 1, cyclic != 0, true, st);
    case 1:  // rows along j: systems (i,k)
        return ptdma_exact_launch(A, B, C, D, D, n1, 1, n3, s2, n2, s1, cyclic != 0, true, st);
    default:  // rows along k: systems (i,j)
        return ptdma_exact_launch(A, B, C, D, D, n1, 1, n2, s1, n3, s2, cyclic != 0, true, st);
    }
}
