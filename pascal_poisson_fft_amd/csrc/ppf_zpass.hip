// ppf_zpass.hip -- host launcher of pass 3 (the z Thomas solves) for FP64 and
// FP32 workspaces: the shapes of the partitioned register Thomas k_zpart, the
// one-thread-per-line k_zthomas, and the choice among them.
#include <type_traits>

#include "ppf_plan.hpp"

namespace ppf {

namespace {
// The shape of a plan that was not tuned, from the line length and the number
// of 16-column workgroups.  z stage in us, 256 x 256 lines (65536 columns)
// unless another grid is named, this rule's shape against the neighbours:
//  * up to 512 rows, about 16 partitions: S P then fills whole groups of four
//    waves, one for each SIMD (a six-wave workgroup of 28 or 32 rows gets one
//    place where two would fit): 300 rows K=20 102, K=32 107, K=16 117;
//    448 rows K=28 127, 32 141, 16 147; 200 rows K=20 54, K=16 57, K=32 60;
//  * 513..768 rows K = 24, whose 128 registers admit two 512-thread
//    workgroups per CU: 768 rows 253, K=28 294, K=32 310 (1024 x 1024 x 768:
//    2.61 ms, K=32 3.90 ms);
//  * FP32 workspaces up to 256 and near 512 rows take 32 columns, whole
//    128-byte rows: 256 rows (32,32) 44, (16,16) 58; 128 rows (16,32) 22,
//    (8,16) 28; 512 rows (32,32) 109, (32,16) 135 (512^3: 345, 405); 384 rows
//    (32,32) 90, (24,16) 81.  FP64 lines never do here, though 32 columns were
//    faster at some lengths (768 x 512 x 96 (16,32) 121, (8,16) 142; 320 x 224 x
//    200 (32,32) 55, (20,16) 60): where was not mapped, tuned plans find it;
//  * fewer workgroups than four per CU are all resident at once, so a line's
//    chain of rows is what counts: 8 columns and short partitions, but only as
//    long as twice as many workgroups are resident too, which ends the earlier
//    the longer the line (and for FP32, whose 8 columns are a quarter of a
//    128-byte row); the lines below lie there.  32 x 32, 64 x 64, 64 x 80 and
//    120 x 120 lines (64, 256, 320, 960 workgroups):
//      66 rows (8,8) 7.4 8.6 - 12.4, (16,16) 8.7 9.1 - 13.2;
//      256 rows (8,8) 8.3 10.4 10.6 22.7, (16,16) 9.4 11.1 11.4 16.4;
//      300 rows (8,8) 9.5 11.6 13.1 27.8, (20,16) 9.9 11.8 12.2 19.7;
//      512 rows (16,8) 10.2 13.8 15.4 42.0, (32,16) 12.6 15.2 16.0 30.2;
//      768 rows (24,8) 12.4 16.9 24.0 63.7, (24,16) 15.2 18.0 20.8 42.6;
//      1024 rows (32,8) 14.8 20.1 31.0 84.1, (32,16) 18.0 21.4 34.1 72.7;
//      FP32 of 768 rows (24,8) 11.6 18.3 21.3 75.1, (24,16) 13.6 15.1 19.2 36.0;
//      of 1024 rows (32,8) 13.6 25.8 33.7 105, (32,16) 15.7 18.1 29.2 65;
//  * 1025..2048 rows 8 columns (a 16-column workgroup exceeds 512 threads or
//    its registers) and K = 32: 128 x 128 lines of 2048 rows 201, K=48 220.
//    K = 48 is faster up to 1536 rows (128, 164) but puts up to three times
//    the rounding on the nearly singular lines (16 x 96 x 1536, all periodic:
//    1.5e-11, 5.4e-12), so neither this rule nor, for FP64, the tuner takes it;
//  * longer lines one thread a line (k_zthomas, where the reason stands).
template <typename T>
int z_default(int n3m, int nwg16) {
    if (n3m > 2048) return 6;
    if (n3m > 1024) return 4;
    constexpr bool F32 = sizeof(T) == 4;
    const int cus = num_cus();
    if (nwg16 < 4 * cus) {
        const bool few = 2 * nwg16 <= 3 * cus, fewer = nwg16 <= (F32 ? cus / 2 : cus);
        if (n3m <= 256) return nwg16 <= (n3m <= 128 ? 4 : n3m <= 192 ? 3 : 2) * cus ? 5 : 1;
        if (n3m <= 320) return fewer ? 5 : 7;
        if (n3m <= 512 && few) return 2;
        if (n3m > 512 && (F32 ? fewer : few)) return n3m <= 768 ? 13 : 4;
    } else {
        if (n3m <= 24) return 11;
        if (F32 && n3m <= 256) return n3m <= 128 ? 16 : 15;
        if (F32 && n3m > 416 && n3m <= 512) return 15;
    }
    if (n3m <= 64) return 1;
    if (n3m <= 128) return 11;
    if (n3m <= 320) return 7;
    if (n3m <= 384) return 12;
    if (n3m <= 448) return 17;
    if (n3m <= 512) return 3;
    return n3m <= 768 ? 12 : 3;
}
}  // namespace

template <typename T>
int launch_z(ppf_plan *p, T *W, hipStream_t s) {
    // the kernels read the z row table that pass 1 of this solve filled
    ZArgs z;
    z.Lx = p->Lx;
    z.Lxs = p->Lxs;
    z.Ly = p->Ly;
    z.n3m = p->d.n3m;
    z.jlo = p->zjlo;
    z.njr = p->znjr;
    z.lamx = p->lamx;
    z.lamy = p->lamy;
    z.zx = p->zx;
    z.zy = p->zy;
    z.mean_kx = p->mean_kx;
    z.mean_jp = p->mean_jp;
    z.mean_scale = p->mean_scale;
    z.zper = p->d.pbc3 != 0;
    z.gate = p->gate;
    const int n3m = p->d.n3m;
    // partitioned register-resident Thomas, shape (K rows per thread, S
    // columns per workgroup); launched only when S*P <= NTMAX and the LDS
    // footprint stays within 64 KB
    bool done = false;
    auto part = [&](auto kk, auto ss, auto nt, auto wpe) {
        constexpr int K = decltype(kk)::value, S = decltype(ss)::value;
        constexpr int NTMAX = decltype(nt)::value, WPE = decltype(wpe)::value;
        const int P = (n3m + K - 1) / K;
        const size_t shm = zp_lds_bytes<K, S>(P);
        if (P < 1 || S * P > NTMAX || shm > 65536) return;
        const int tiles = (p->Lx + S - 1) / S;
        const int ntiles = tiles * p->znjr;
        // FP64 arithmetic for FP32 storage too: FP32 arithmetic measured no
        // faster at 512^3 (0.509 vs 0.515 ms) and costs the refinement a sweep
        hipLaunchKernelGGL((k_zpart<T, K, S, NTMAX, WPE>), dim3((unsigned)ntiles), dim3(S * P), shm, s, W, z,
                           p->zcoef, p->zcoef + n3m, p->mean, P);
        done = true;
    };
    using std::integral_constant;
#define PPF_Z(K, S, NT, WPE) integral_constant<int, K>{}, integral_constant<int, S>{}, integral_constant<int, NT>{}, integral_constant<int, WPE>{}
    int v = p->zvariant ? p->zvariant : z_default<T>(n3m, (p->Lx + 15) / 16 * p->znjr);
    if (n3m > z_id_rows(v)) {
        if (!z.zper) return PPF_ERR_UNSUPPORTED;
        v = n3m <= 1024 ? 3 : 4;
    }
    switch (v) {
        case 1: part(PPF_Z(16, 16, 512, 4)); break;
        case 2: part(PPF_Z(16, 8, 512, 4)); break;
        case 3: case 10: part(PPF_Z(32, 16, 512, 3)); break;
        case 4: case 9: part(PPF_Z(32, 8, 512, 3)); break;
        case 5: part(PPF_Z(8, 8, 512, 4)); break;
        case 7: part(PPF_Z(20, 16, 512, 4)); break;
        case 8: part(PPF_Z(12, 16, 704, 4)); break;
        case 11: part(PPF_Z(8, 16, 512, 4)); break;
        case 12: part(PPF_Z(24, 16, 512, 4)); break;
        case 13: part(PPF_Z(24, 8, 512, 3)); break;
        case 14: part(PPF_Z(48, 8, 512, 2)); break;
        // 32 columns: 128-byte row segments for FP32 workspaces
        case 15: part(PPF_Z(32, 32, 512, 3)); break;
        case 16: part(PPF_Z(16, 32, 512, 4)); break;
        case 17: part(PPF_Z(28, 16, 512, 3)); break;
        default: break;
    }
#undef PPF_Z
    // a shape that does not fit the extent is reported
    if (!done && v != 6) return PPF_ERR_UNSUPPORTED;
    if (!done) {
        const long ncol = (long)p->Lx * p->znjr;
        // the one-thread-per-line kernel keeps its forward multipliers in cs
        if (p->cs_elems < (size_t)ncol * (size_t)n3m) return PPF_ERR_UNSUPPORTED;
        constexpr int wt = w_tile<T>(), rj = 32 / wt;
        const unsigned blocks = (unsigned)((p->Lx + wt - 1) / wt) * (unsigned)((p->znjr + rj - 1) / rj);
        hipLaunchKernelGGL((k_zthomas<T>), dim3(blocks), dim3(64), 0, s, W, reinterpret_cast<T *>(p->cs), z, p->zcoef,
                           p->zcoef + n3m, p->mean);
    }
    return PPF_OK;
}

template int launch_z<double>(ppf_plan *, double *, hipStream_t);
template int launch_z<float>(ppf_plan *, float *, hipStream_t);

}  // namespace ppf
