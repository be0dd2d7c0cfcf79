// ppf_tdma.hip -- batched Thomas solver on explicit coefficient arrays.
//
// Replaces the one-rank branch of PaScaL_TDMA_many_solve_cuda
// (01_Fortran/PaScaL_TDMA/src/pascal_tdma_cuda.f90:230-269) which launches
// tdma_many_cuda (tdmas_cuda.f90:35-102).  One thread per system; system index
// fastest in memory, so every row access of a wavefront is one contiguous
// 512-byte segment.  The recurrence keeps the previous row in registers
// instead of the reference's shared-memory pipeline copies, and the
// arithmetic is evaluated without contraction in the reference's order
// (d/b, c/b; r = 1/(b - a c'); d' = r (d - a d'); c' = r c; d -= c' d_next), so
// results are bitwise equal to the reference Thomas on the same inputs.
#include <hip/hip_runtime.h>

#include <new>

#include "../../include/pascal_poisson_fft.h"

struct ppf_tdma_plan {
    int nx, ny, nz;
    double *e;  // correction vector of the cyclic solve (nx*ny*nz)
};

namespace {

// One thread solves one system, row after row, so what bounds these kernels is
// the latency of a row's loads unless they are issued ahead: rows come in
// chunks (U of the elimination, V of the substitutions, whose rows take less
// time than their loads' latency), the next chunk's loads in flight while the
// current one is solved, and a chunk's stores are younger than the loads that
// follow it in the chain, so nothing waits for them.  One-wave workgroups
// spread a few thousand systems over as many CUs as there are waves.  256^3
// (many systems): 291 -> 200 us, 6.0 TB/s of the 72 bytes a row moves; cyclic
// 6000 systems of 90 rows: 57 -> 28 us and 256 of 512 rows 363 -> 138, where a
// row's chain of a correctly rounded division and the products that use it
// (about 0.2 us) is what is left.
//
// A chunk costs its registers (4 arrays x U rows x 2 chunks), which short
// systems do not use and whose waves they miss: up to 8 rows (4, 8) is taken,
// 4M systems of 2 rows 53 us against 60 with (8, 16), cyclic of 3 rows 136
// against 163 with (4, 16).  The cyclic kernel holds a third vector: U = 8 left
// it one wave per SIMD (65536 systems of 400 rows 556 us, 542 with 4).
//
// Past the last row a chunk's loads are left out: clamped to that row instead,
// 4M systems of 3 rows took 194 us instead of 96, cyclic 309 instead of 136, 1M
// of 20 rows 228 instead of 214.  The tests of it cost 1.3% where waves are few
// and lines long (256^3 with its refill 304.5 us, clamped 300.7), so the plain
// form clamps from 128 rows on, where a chunk is little of a line.
constexpr int kTdmaThreads = 64;
// millions of systems fill the chip whatever the workgroup's size, and its
// launches are then fewer: 4M systems of 12 rows 492 -> 472 us (490,000 of 20
// rows 101.6, 102.8)
inline int tdma_threads(long nsys) { return nsys >= 1L << 21 ? 4 * kTdmaThreads : kTdmaThreads; }
constexpr int kTdmaShort = 8, kTdmaLong = 128;  // rows up to, and from which, as above

// U rows of the N arrays src, from row k0 in steps of DIR, clamped to the ends or
// as far as there are rows
template <int N, int U, int DIR, bool CLAMP>
struct TdmaRows {
    double v[N][U];
    __device__ __forceinline__ void load(const double *const (&src)[N], size_t ns, long s, int k0, int nrow) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int k = k0 + DIR * u;
            if (CLAMP) k = DIR > 0 ? (k < nrow ? k : nrow - 1) : (k > 0 ? k : 0);
            else if (DIR > 0 ? k >= nrow : k < 0) break;
#pragma unroll
            for (int n = 0; n < N; ++n) v[n][u] = src[n][(size_t)k * ns + s];
        }
    }
};

template <int U, int V, bool CLAMP>
__global__ void __launch_bounds__(4 * kTdmaThreads)
k_tdma_many(const double *__restrict__ a, const double *__restrict__ b, double *c, double *d, long nsys, int nrow) {
#pragma clang fp contract(off)
    const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsys) return;
    const size_t ns = (size_t)nsys;
    double dp, cp;
    {
        const double *const src[4] = {a, b, c, d};
        TdmaRows<4, U, 1, CLAMP> cur, nxt;
        cur.load(src, ns, s, 1, nrow);
        dp = d[s] / b[s];
        cp = c[s] / b[s];
        d[s] = dp;
        c[s] = cp;
        for (int k0 = 1; k0 < nrow; k0 += U) {
            if (k0 + U < nrow) nxt.load(src, ns, s, k0 + U, nrow);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (k0 + u < nrow) {
                    const size_t q = (size_t)(k0 + u) * ns + (size_t)s;
                    const double ak = cur.v[0][u];
                    const double r = 1.0 / (cur.v[1][u] - ak * cp);
                    dp = r * (cur.v[3][u] - ak * dp);
                    cp = r * cur.v[2][u];
                    d[q] = dp;
                    c[q] = cp;
                }
            }
            cur = nxt;
        }
    }
    const double *const src[2] = {c, d};
    TdmaRows<2, V, -1, CLAMP> cur, nxt;
    cur.load(src, ns, s, nrow - 2, nrow);
    for (int k0 = nrow - 2; k0 >= 0; k0 -= V) {
        if (k0 - V >= 0) nxt.load(src, ns, s, k0 - V, nrow);
#pragma unroll
        for (int u = 0; u < V; ++u) {
            if (k0 - u >= 0) {
                dp = cur.v[1][u] - cur.v[0][u] * dp;
                d[(size_t)(k0 - u) * ns + (size_t)s] = dp;
            }
        }
        cur = nxt;
    }
}

// Cyclic Thomas, op order of tdma_cycl_many_cuda (tdmas_cuda.f90:114-217):
// rows 1..n-1 are reduced for d' and the correction vector e (e_1 = -a_1,
// e_{n-1} = -c_{n-1}, zero between: constants here, not stored and read back),
// x_0 follows from row 0, then x_k = d'_k + x_0 e_k.  x_0 uses rows 1 and n-1 of
// d and e after the backward loop, which for n = 2 (one row) are the forward
// values.
template <int U, int V, bool CLAMP>
__global__ void __launch_bounds__(4 * kTdmaThreads)
k_tdma_cycl_many(const double *__restrict__ a, const double *__restrict__ b, double *c, double *d, double *e, long nsys,
                 int nrow) {
#pragma clang fp contract(off)
    const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsys) return;
    const size_t ns = (size_t)nsys;
    const int last = nrow - 1;
    const double a0 = a[s], b0 = b[s], c0 = c[s], d0 = d[s];
    double d1 = d[ns + s], b1 = b[ns + s], c1 = c[ns + s], e1 = last == 1 ? -c1 : -a[ns + s];
    {
        const double *const src[4] = {a, b, c, d};
        TdmaRows<4, U, 1, CLAMP> cur, nxt;
        cur.load(src, ns, s, 2, nrow);
        d1 = d1 / b1;
        c1 = c1 / b1;
        e1 = e1 / b1;
        d[ns + s] = d1;
        c[ns + s] = c1;
        e[ns + s] = e1;
        for (int k0 = 2; k0 < nrow; k0 += U) {
            if (k0 + U < nrow) nxt.load(src, ns, s, k0 + U, nrow);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u;
                if (k < nrow) {
                    const size_t q = (size_t)k * ns + (size_t)s;
                    const double ak = cur.v[0][u];
                    const double ek = k == last ? -cur.v[2][u] : 0.0;
                    const double r = 1.0 / (cur.v[1][u] - ak * c1);
                    d1 = r * (cur.v[3][u] - ak * d1);
                    e1 = r * (ek - ak * e1);
                    c1 = r * cur.v[2][u];
                    e[q] = e1;
                    d[q] = d1;
                    c[q] = c1;
                }
            }
            cur = nxt;
        }
    }
    const double dn = d1, en = e1;  // row n-1
    {
        const double *const src[3] = {c, d, e};
        TdmaRows<3, V, -1, CLAMP> cur, nxt;
        cur.load(src, ns, s, nrow - 2, nrow);
        for (int k0 = nrow - 2; k0 >= 1; k0 -= V) {
            if (k0 - V >= 1) nxt.load(src, ns, s, k0 - V, nrow);
#pragma unroll
            for (int u = 0; u < V; ++u) {
                if (k0 - u >= 1) {
                    const size_t q = (size_t)(k0 - u) * ns + (size_t)s;
                    d1 = cur.v[1][u] - cur.v[0][u] * d1;
                    e1 = cur.v[2][u] - cur.v[0][u] * e1;
                    d[q] = d1;
                    e[q] = e1;
                }
            }
            cur = nxt;
        }
    }
    const double x0 = (d0 - a0 * dn - c0 * d1) / (b0 + a0 * en + c0 * e1);
    d[s] = x0;
    const double *const src[2] = {d, e};
    TdmaRows<2, V, 1, CLAMP> cur, nxt;
    cur.load(src, ns, s, 1, nrow);
    for (int k0 = 1; k0 < nrow; k0 += V) {
        if (k0 + V < nrow) nxt.load(src, ns, s, k0 + V, nrow);
#pragma unroll
        for (int u = 0; u < V; ++u)
            if (k0 + u < nrow) d[(size_t)(k0 + u) * ns + (size_t)s] = cur.v[0][u] + x0 * cur.v[1][u];
        cur = nxt;
    }
}

}  // namespace

extern "C" {

int ppf_tdma_plan_many_create(int nx_sys, int ny_sys, int nz_row, ppf_tdma_plan **plan) {
    if (!plan) return PPF_ERR_INVALID_ARG;
    *plan = nullptr;
    if (nx_sys <= 0 || ny_sys <= 0 || nz_row <= 0) return PPF_ERR_INVALID_ARG;
    ppf_tdma_plan *p = new (std::nothrow) ppf_tdma_plan{nx_sys, ny_sys, nz_row, nullptr};
    if (!p) return PPF_ERR_ALLOC;
    // the cyclic solve's correction vector, as the reference plan's e_buff
    // for one rank (pascal_tdma_cuda.f90:108-201)
    if (hipMalloc(&p->e, sizeof(double) * (size_t)nx_sys * ny_sys * nz_row) != hipSuccess) {
        delete p;
        return PPF_ERR_ALLOC;
    }
    *plan = p;
    return PPF_OK;
}

int ppf_tdma_many_solve(ppf_tdma_plan *p, const double *a, const double *b, double *c, double *d, void *stream) {
    if (!p || !a || !b || !c || !d) return PPF_ERR_INVALID_ARG;
    const long nsys = (long)p->nx * p->ny;
    const int nt = tdma_threads(nsys);
    const auto kernel = p->nz <= kTdmaShort  ? k_tdma_many<4, 8, false>
                        : p->nz < kTdmaLong ? k_tdma_many<8, 16, false>
                                            : k_tdma_many<8, 16, true>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((nsys + nt - 1) / nt)), dim3(nt), 0,
                       static_cast<hipStream_t>(stream), a, b, c, d, nsys, p->nz);
    return hipGetLastError() == hipSuccess ? PPF_OK : PPF_ERR_HIP;
}

int ppf_tdma_many_solve_cycle(ppf_tdma_plan *p, const double *a, const double *b, double *c, double *d,
                              void *stream) {
    if (!p || !a || !b || !c || !d) return PPF_ERR_INVALID_ARG;
    if (p->nz < 2) return PPF_ERR_SIZE;
    const long nsys = (long)p->nx * p->ny;
    const int nt = tdma_threads(nsys);
    const auto kernel = p->nz <= kTdmaShort ? k_tdma_cycl_many<4, 8, false> : k_tdma_cycl_many<4, 16, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((nsys + nt - 1) / nt)), dim3(nt), 0,
                       static_cast<hipStream_t>(stream), a, b, c, d, p->e, nsys, p->nz);
    return hipGetLastError() == hipSuccess ? PPF_OK : PPF_ERR_HIP;
}

int ppf_tdma_plan_many_destroy(ppf_tdma_plan *p) {
    if (!p) return PPF_ERR_INVALID_ARG;
    if (p->e) (void)hipFree(p->e);
    delete p;
    return PPF_OK;
}

}  // extern "C"
