// Jacobi sweeps (gfx950), out of place: u = J(v) on a box (mgp_jacobi_*;
// include/jacobi.h:39-82).  Bound by memory: 3 values moved per point.
//
// A wave owns R = 4 rows x 124 columns, two columns per lane (16-byte loads and
// stores in FP64; lanes 0 and 63 only feed their neighbours), and marches along
// x with the three planes of v it needs in registers, so a point of v is loaded
// once per tile and not five times through the caches as by one thread per
// point.  Four waves, one above the other, share a workgroup and so the cache
// lines of their edge rows.  Short marches (2 planes at least, about 65536
// waves) keep the waves that share rows close together in time: 1025 x 1025 x
// 513 FP64 3.44 / 3.35 ms with 32768 / 65536 waves, 3.63 with 8192.
//
// Measured against one thread per point (1: k_jacobi), with the ghost refresh:
// 385 x 353 x 321 FP64 0.234 / 0.315 ms (1.05 GB moved, 4.6 TB/s), FP32 0.129 /
// 0.184; 1025 x 1025 x 513 3.35 / 3.52 and 1.64 / 2.11; 801 x 609 x 417 1.24 /
// 1.52 and 0.62 / 0.90; 257 x 257 x 129 41 / 72 and 30 / 41 us.  Small boxes and
// those that fill little of the tiles' 16 rows x 124 columns are left to one
// thread per point (march_pays).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mgp.h"
#include "mgp_device.h"
#include "mgp_point.h"
#include "mgp_sweep.h"
#include "mgp_wave.h"

namespace mgp {

int64_t g_jacobi_kernel = 0;  // 1: one thread per point, 2: wave tiles marching along x, 0: by the box

namespace {

template <class T>
struct JacobiArgs {
    View<T> u, v, f;
    int32_t bx0, bx1, by0, by1, bz0, bz1;
    T one_omega, omega_sixth, hsq;
    int32_t ytiles, ztiles, ntiles, ntiles_pad, xchunk;
    uint32_t ubytes, vbytes, fbytes;  // a plane from row by0 (v: by0 - 1) on
};

template <class T, int MODE, int R, int NW, bool EDGE>
__device__ __forceinline__ void jacobi_march(const JacobiArgs<T>& A, int tl) {
    constexpr int NR = R + 2, W = 124;  // columns a wave writes: those of lanes 1 .. 62
    const int tz = tl % A.ztiles, ty = (tl / A.ztiles) % A.ytiles, xc = tl / (A.ztiles * A.ytiles);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int y0 = A.by0 + (ty * NW + w) * R, z = A.bz0 - 2 + tz * W + 2 * lane;
    const int xa = A.bx0 + xc * A.xchunk, xb = min(A.bx1, xa + A.xchunk);
    // columns bz0 - 1 .. bz1 of v and bz0 .. bz1 - 1 of f exist.  A pair that
    // reaches past them is taken where it does not and its one column that
    // counts moved into place (lane 0: the second, the lane at the end: the first).
    const int zv = min(max(z, A.bz0 - 1), A.bz1 - 1), zf = min(max(z, A.bz0), A.bz1 - 2);
    const bool vlo = EDGE && z < zv, vhi = EDGE && z > zv, fhi = EDGE && z > zf;
    const uint32_t vo = (uint32_t)((zv - (A.bz0 - 1)) * (int)sizeof(T)), fo = (uint32_t)((zf - A.bz0) * (int)sizeof(T));
    uint32_t vr[NR], fr[R], ur[R];
#pragma unroll
    for (int t = 0; t < NR; t++)
        vr[t] = (uint32_t)(min(y0 - 1 + t, A.by1) - (A.by0 - 1)) * (uint32_t)A.v.s1 * (uint32_t)sizeof(T);
#pragma unroll
    for (int t = 0; t < R; t++) {
        const uint32_t y = (uint32_t)(min(y0 + t, A.by1 - 1) - A.by0);
        fr[t] = y * (uint32_t)A.f.s1 * (uint32_t)sizeof(T);
        ur[t] = y * (uint32_t)A.u.s1 * (uint32_t)sizeof(T);
    }
    auto load_v = [&](int i, T (&V)[NR][2]) {
        const __amdgpu_buffer_rsrc_t rs = plane_rsrc(
            A.v.p + (int64_t)min(i, A.bx1) * A.v.s0 + (int64_t)(A.by0 - 1) * A.v.s1 + (A.bz0 - 1), A.vbytes);
#pragma unroll
        for (int t = 0; t < NR; t++) bload2<T>(rs, vo, vr[t], V[t][0], V[t][1]);
    };
    auto load_f = [&](int i, T (&F)[R][2]) {
        const __amdgpu_buffer_rsrc_t rs = plane_rsrc(
            A.f.p + (int64_t)min(i, A.bx1 - 1) * A.f.s0 + (int64_t)A.by0 * A.f.s1 + A.bz0, A.fbytes);
#pragma unroll
        for (int t = 0; t < R; t++) bload2<T>(rs, fo, fr[t], F[t][0], F[t][1]);
    };
    const uint32_t uz = (uint32_t)((z - A.bz0) * (int)sizeof(T));
    const bool own = lane >= 1 && lane <= 62;
    const uint32_t ua = own && z + 1 < A.bz1 ? uz : BUF_OOB;   // both columns
    const uint32_t u1 = own && z + 1 == A.bz1 ? uz : BUF_OOB;  // the box's last column alone
    T Vm[NR][2], V0[NR][2], Vp[NR][2], VL[NR][2], F0[R][2], FL[R][2];
    load_v(xa - 1, Vm);
    load_v(xa, V0);
    load_v(xa + 1, Vp);
    load_f(xa, F0);
    for (int i = xa; i < xb; i++) {
        load_v(i + 2, VL);
        load_f(i + 1, FL);
        const __amdgpu_buffer_rsrc_t ro =
            plane_rsrc(A.u.p + (int64_t)i * A.u.s0 + (int64_t)A.by0 * A.u.s1 + A.bz0, A.ubytes);
#pragma unroll
        for (int t = 0; t < R; t++) {
            const T(&c)[2] = V0[t + 1];
            const bool in = y0 + t < A.by1;
            // (vhi lanes and lane 0 feed their neighbours only)
            const T zl = lane_prev(vlo ? c[0] : c[1]), zh = lane_next(vhi ? c[1] : c[0]);
            const T f0 = fhi ? F0[t][1] : F0[t][0];
            const T o0 = relax_point<T, MODE>(c[0], Vm[t + 1][0], Vp[t + 1][0], V0[t][0], V0[t + 2][0], zl, c[1],
                                              f0, A.one_omega, A.omega_sixth, A.hsq);
            const T o1 = relax_point<T, MODE>(c[1], Vm[t + 1][1], Vp[t + 1][1], V0[t][1], V0[t + 2][1], c[0], zh,
                                              F0[t][1], A.one_omega, A.omega_sixth, A.hsq);
            bstore2(o0, o1, ro, in ? ua : BUF_OOB, ur[t]);
            if (EDGE) bstore(o0, ro, in ? u1 : BUF_OOB, ur[t]);
        }
#pragma unroll
        for (int t = 0; t < NR; t++)
#pragma unroll
            for (int k = 0; k < 2; k++) Vm[t][k] = V0[t][k], V0[t][k] = Vp[t][k], Vp[t][k] = VL[t][k];
#pragma unroll
        for (int t = 0; t < R; t++)
#pragma unroll
            for (int k = 0; k < 2; k++) F0[t][k] = FL[t][k];
    }
}

template <class T, int MODE, int R, int NW>
__global__ void __launch_bounds__(64 * NW) k_jacobi_march(JacobiArgs<T> A) {
    const int per_xcd = A.ntiles_pad / 8;
    const int tl = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (tl >= A.ntiles) return;
    const int tz = tl % A.ztiles;
    if (tz == 0 || tz == A.ztiles - 1) jacobi_march<T, MODE, R, NW, true>(A, tl);
    else jacobi_march<T, MODE, R, NW, false>(A, tl);
}

// Where the march is the faster one.  Below 2^20 (FP64) or 2^21 (FP32) box points
// either kernel is a few us, most of it the launch and one trip to memory, and
// the march adds its chain of planes: per point / march, us, without the ghost
// refresh, 33 x 33 x 33 FP64 4.2 / 4.9, 65 x 65 x 33 FP32 4.2 / 5.0, 128 x 128 x
// 65 FP32 4.9 / 7.0.  Lanes and rows of a tile outside the box cost as much as
// those inside.  FP32: the box has to fill half of its tiles (707 x 707 x 33
// 69.7 / 80.6, 2^22 points by 17 columns 33 / 46; 2^21 points by 129 columns 10.3 /
// 9.0, 2^22 by 65 17.0 / 14.9).  FP64, twice the bytes for the same lanes: a third
// of them below 2^21 points (1025 x 33 x 33 9.9 / 13.3, 128 x 128 x 65 8.0 / 7.4),
// any box above (2^21 points by 9 columns 51.0 / 48.9, 707 x 707 x 33 176 / 144).
// Of 1541 random boxes of up to 1100 points a side the rule sends 533 to the
// march, which gains 33 % (FP64) and 54 % (FP32) on average there; 7 of them, FP64,
// take 3 to 15 % longer.  The others would on average have taken 14 and 17 % longer.
template <class T>
static bool march_pays(int64_t nx, int64_t ny, int64_t nz) {
    const int64_t points = nx * ny * nz, area = ny * nz;
    const int64_t tiles = (ny + 15) / 16 * 16 * ((nz + 123) / 124 * 124);
    if (sizeof(T) == 8) return points >= (int64_t)1 << (3 * area >= tiles ? 20 : 21);
    return points >= (int64_t)1 << 21 && 2 * area >= tiles;
}

}  // namespace

template <class T>
int march_jacobi(int mode, const mgp_array* u, const mgp_array* v, const mgp_array* f, const int64_t b[6],
                 double omega, double h, void* stream) {
    constexpr int R = 4, NW = 4;
    const int64_t nx = b[1] - b[0], ny = b[3] - b[2], nz = b[5] - b[4];
    if (nx < 1 || ny < 1 || nz < 2) return MGP_ERR_ARG;
    if (g_jacobi_kernel == 0 && !march_pays<T>(nx, ny, nz)) return MGP_ERR_ARG;
    if (u->data == v->data) return MGP_ERR_ARG;  // (a march reads planes ahead of what it writes)
    JacobiArgs<T> A;
    const mgp_array* a[3] = {u, v, f};
    uint32_t bytes[3];
    for (int q = 0; q < 3; q++) {
        const int64_t ring = a[q] == v ? 2 : 0;
        const int64_t n = ((ny - 1 + ring) * a[q]->stride[1] + nz + ring) * (int64_t)sizeof(T);
        if (n >= (int64_t)BUF_OOB) return MGP_ERR_ARG;
        bytes[q] = (uint32_t)n;
    }
    A.ubytes = bytes[0], A.vbytes = bytes[1], A.fbytes = bytes[2];
    A.u = view_of<T>(*u);
    A.v = view_of<T>(*v);
    A.f = view_of<T>(*f);
    A.bx0 = (int32_t)b[0], A.bx1 = (int32_t)b[1], A.by0 = (int32_t)b[2], A.by1 = (int32_t)b[3];
    A.bz0 = (int32_t)b[4], A.bz1 = (int32_t)b[5];
    const RelaxConsts<T> c(omega, h);
    A.one_omega = c.one_omega, A.omega_sixth = c.omega_sixth, A.hsq = c.hsq;
    A.ytiles = (int32_t)((ny + R * NW - 1) / (R * NW));
    A.ztiles = (int32_t)((nz + 123) / 124);
    const int64_t tiles = (int64_t)A.ytiles * A.ztiles;
    int64_t chunks = std::max<int64_t>(1, 65536 / (tiles * NW));
    chunks = std::min<int64_t>(chunks, std::max<int64_t>(1, nx / 2));
    A.xchunk = (int32_t)((nx + chunks - 1) / chunks);
    const int64_t ntiles = tiles * ((nx + A.xchunk - 1) / A.xchunk);
    if (ntiles > INT32_MAX - 8) return MGP_ERR_ARG;
    A.ntiles = (int32_t)ntiles;
    A.ntiles_pad = (A.ntiles + 7) / 8 * 8;
    const dim3 g(A.ntiles_pad), blk(64 * NW);
    const hipStream_t st = (hipStream_t)stream;
    if (mode == MGP_MODE_REFERENCE)
        hipLaunchKernelGGL((k_jacobi_march<T, MGP_MODE_REFERENCE, R, NW>), g, blk, 0, st, A);
    else
        hipLaunchKernelGGL((k_jacobi_march<T, MGP_MODE_CONSISTENT, R, NW>), g, blk, 0, st, A);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MGP_OK : (int)e;
}
template int march_jacobi<double>(int, const mgp_array*, const mgp_array*, const mgp_array*, const int64_t[6], double,
                                  double, void*);
template int march_jacobi<float>(int, const mgp_array*, const mgp_array*, const mgp_array*, const int64_t[6], double,
                                 double, void*);

}  // namespace mgp
