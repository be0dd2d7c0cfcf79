// ppf_aux.hpp -- small non-template kernels of the solve path (z row table,
// reductions, the device-side refinement test, ghost faces, the copy
// yardstick), with internal linkage so several translation units may include
// them.
#pragma once

#include "ppf_kernels.hpp"

namespace ppf {

// z row coefficients for one solve as a table (read by the residual forms):
// zam[k], zap[k] (k < n3m), then zap[n3m..n3m+3] = the wall extrapolation
// coefficients.
static __global__ void __launch_bounds__(256)
k_zcoef(const double *__restrict__ dx3, const double *__restrict__ dmx3, int n3m, double *__restrict__ zam,
        double *__restrict__ zap) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n3m) z_row(dx3, dmx3, n3m, k, zam[k], zap[k]);
    if (k == 0) z_wall_bc(dmx3, n3m, zap + n3m);
}

// Totals of the per-workgroup triples (sum r^2, sum f^2, sum x) in a fixed
// order (deterministic).  With check set it is also the device-side
// refinement test (below; check.gate is the gate to test and close, the same
// one that gates this kernel), which saves a launch per test.
struct GateTest {
    int *gate = nullptr;
    double tol = 0.0;
    int count = 0;
    double *res_out = nullptr;
    bool nan_closes = false;  // a NaN residual closes the gate (the host sees it)
};
static __global__ void __launch_bounds__(256) k_reduce3(const double *__restrict__ partial, int n, double *__restrict__ out,
                                                 const int *__restrict__ gate, GateTest check = GateTest{},
                                                 double *__restrict__ host = nullptr) {
    if (gated_off(gate)) return;
    __shared__ double red[256];
    double a = 0.0, b = 0.0, c = 0.0;
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        a += partial[3 * q];
        b += partial[3 * q + 1];
        c += partial[3 * q + 2];
    }
    a = block_sum<256>(a, red);
    b = block_sum<256>(b, red);
    c = block_sum<256>(c, red);
    if (threadIdx.x == 0) {
        out[0] = a;
        out[1] = b;
        out[2] = c;
        if (host) {  // pinned host memory, read after the stream is synchronised
            host[0] = a;
            host[1] = b;
            host[2] = c;
        }
        if (check.gate && check.gate[0] != 0) {
            const double rel = b > 0 ? sqrt(a / b) : sqrt(a);
            *check.res_out = rel;
            check.gate[1] += check.count;
            check.gate[0] = (rel <= check.tol || (check.nan_closes && rel != rel)) ? 0 : 1;
        }
    }
}

// Device-side refinement test.  k_gate_init opens the gate (gate[0] = 1: more
// sweeps may run) and sets the sweep count gate[1]; the test (k_reduce3 with
// a GateTest, while the gate is open) stores ||r||/||f|| of the totals it
// just reduced in res_out, counts the sweep that produced them (count = 1
// after a gated sweep) and closes the gate once the residual is <= tol (a
// NaN residual keeps it open, so the sweeps run out and the caller sees the
// miss).
static __global__ void k_gate_init(int *__restrict__ gate, int sweeps) {
    gate[0] = 1;
    gate[1] = sweeps;
}

// Ghost layers of P from its interior, every ghost cell in one launch.  The
// reference's order is wall extrapolation p0 = BC_a p1 - BC_b p2 along x, y, z
// (cuda_neumann_BC / apply_bc_on_direction, fft_3d_poisson.f90:798-852), then
// the periodic wraps along x, y, z (cuda_ghostcell_update on one rank,
// :666-796), each over the full ghosted ranges of the other axes.  A cell that
// is a ghost along several axes therefore holds the last of these steps applied
// to the earlier ones: its wrapped indices are replaced first, and what remains
// is z's extrapolation of y's of x's, at most eight interior cells.  (As up to
// six dependent face kernels the launches cost more than the faces: 112 x 96 x
// 130 3 x 3.4 us and the gaps between them, now 4.4 us; 512^3 27 us, as before.)
struct GhostArgs {
    int n[3];
    int per[3];
    const double *dmx[3];
};
static __global__ void __launch_bounds__(256) k_ghosts(double *__restrict__ P, GhostArgs g) {
    const long L1 = g.n[0] + 2, L2 = g.n[1] + 2;
    const unsigned l1 = (unsigned)L1;
    const unsigned nz = l1 * (unsigned)L2, ny = l1 * g.n[2], nx = (unsigned)g.n[1] * g.n[2];  // cells of one face per axis
    __shared__ double ws[6][2];  // wall weights of the low and the high end, per axis
    if (threadIdx.x < 6) {
        const int a = threadIdx.x >> 1, n = g.n[a], hi = threadIdx.x & 1;
        const double *m = g.dmx[a];
        const double d1 = hi ? m[n + 1] : m[1], d2 = hi ? m[n] : m[2], s = d1 + d2;
        ws[threadIdx.x][0] = s * s / (s * s - d1 * d1);
        ws[threadIdx.x][1] = d1 * d1 / (s * s - d1 * d1);
    }
    __syncthreads();
    unsigned q = blockIdx.x * blockDim.x + threadIdx.x;  // (extents up to 1024, 1024 and 4096: below 2^25 cells in all)
    int at[3];
    if (q < 2 * nz) {
        at[2] = q < nz ? 0 : g.n[2] + 1;
        q = q < nz ? q : q - nz;
        at[1] = (int)(q / l1);
        at[0] = (int)(q % l1);
    } else if ((q -= 2 * nz) < 2 * ny) {
        at[1] = q < ny ? 0 : g.n[1] + 1;
        q = q < ny ? q : q - ny;
        at[2] = 1 + (int)(q / l1);
        at[0] = (int)(q % l1);
    } else if ((q -= 2 * ny) < 2 * nx) {
        // both ends of a row on adjacent lanes: a row's high ghost and the next
        // row's low one share a cache line
        at[0] = (q & 1) ? g.n[0] + 1 : 0;
        q >>= 1;
        at[2] = 1 + (int)(q / (unsigned)g.n[1]);
        at[1] = 1 + (int)(q % (unsigned)g.n[1]);
    } else {
        return;
    }
    // per axis: the value is wa v[ia] - wb v[ib] (wb = 0: v[ia] itself)
    int ia[3], ib[3];
    double wa[3], wb[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int n = g.n[a], i = at[a];
        ia[a] = ib[a] = i;
        wa[a] = 1.0;
        wb[a] = 0.0;
        if (i != 0 && i != n + 1) continue;
        if (g.per[a]) {
            ia[a] = ib[a] = i == 0 ? n : 1;
        } else {
            wa[a] = ws[2 * a + (i != 0)][0];
            wb[a] = ws[2 * a + (i != 0)][1];
            ia[a] = i == 0 ? 1 : n;
            ib[a] = i == 0 ? 2 : n - 1;
        }
    }
    auto row = [&](int k, int j) {
        const double *r = P + ((long)k * L2 + j) * L1;
        return wb[0] == 0.0 ? r[ia[0]] : wa[0] * r[ia[0]] - wb[0] * r[ib[0]];
    };
    auto plane = [&](int k) { return wb[1] == 0.0 ? row(k, ia[1]) : wa[1] * row(k, ia[1]) - wb[1] * row(k, ib[1]); };
    P[((long)at[2] * L2 + at[1]) * L1 + at[0]] =
        wb[2] == 0.0 ? plane(ia[2]) : wa[2] * plane(ia[2]) - wb[2] * plane(ib[2]);
}

// Streaming copy, the measured-bandwidth yardstick for the pass kernels and
// the calibration of HBM byte counters: one nontemporal 16-byte load and
// store per thread, one workgroup per 4 KiB.  Of the copy shapes measured at
// 1 GiB on MI355X this one is the fastest (6.5 TB/s; a persistent grid-stride
// loop 4.8-6.1 TB/s, hipMemcpy 5.1 TB/s).
using D2v = double __attribute__((ext_vector_type(2)));
static __global__ void __launch_bounds__(256) k_copy(D2v *__restrict__ dst, const D2v *__restrict__ src, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) st_stream(&dst[i], ld_stream(&src[i]));
}

}  // namespace ppf
