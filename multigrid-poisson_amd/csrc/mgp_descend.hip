// Residual and full-weighting restriction in one pass (gfx950): coarse f = FW(f
// - L u), consistent mode (mgp_residual_restrict_fw_*; include/residual.h:58-79,
// include/fullweighting.h:59-121), of small levels on blocks and of larger ones
// by a march.
//
// A march along x (mgp_sweep.hip) takes its planes one after the other, 20 us
// and more however small the level.  Here a workgroup of 8 waves owns 4 x 4 x 32
// coarse points and takes the 9 x 9 x 65 fine residuals under them at once:
// each wave computes every eighth of the 81 rows into LDS (lane = fine column,
// the z neighbours from global memory like the others; the 65th column by one
// lane per row), then each thread forms two coarse points from LDS.  r outside
// the box is read as stored, and a neighbour outside the shape is the clamped
// one, as in the march.  The sums run in the order of the 27 terms; weights are
// powers of two, so a weight and its sum round together (fma) as they do apart,
// and the middle plane's doubled terms are twice the sum of the others' form.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mgp.h"
#include "mgp_device.h"
#include "mgp_point.h"
#include "mgp_sweep.h"
#include "mgp_wave.h"

namespace mgp {

int64_t g_fw_block_points = 1 << 21;  // largest fine level taken

namespace {

constexpr int DC = 4, DK = 32;             // coarse points per block: DC x DC x DK
constexpr int DF = 2 * DC + 1, DZ = 2 * DK + 1;  // fine residuals under them
constexpr int DW = 8;                      // waves

template <class T>
struct DescendArgs {
    View<T> u, f, r, c;
    int32_t bx0, bx1, by0, by1, bz0, bz1;
    T inv_h2;
    int32_t ytiles, ztiles;
};

template <class T>
__global__ void __launch_bounds__(64 * DW) k_resid_fw_block(DescendArgs<T> A) {
    __shared__ T sr[DF][DF][DZ + 1];
    const int tz = blockIdx.x % A.ztiles, ty = (blockIdx.x / A.ztiles) % A.ytiles,
              tx = blockIdx.x / (A.ztiles * A.ytiles);
    const int I0 = tx * DC, J0 = ty * DC, K0 = tz * DK;
    const int n0 = (int)A.u.n0, n1 = (int)A.u.n1, n2 = (int)A.u.n2;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // r at fine (x, y, z), each clamped into the shape
    auto residual = [&](int x, int y, int z) -> T {
        const int64_t o = (int64_t)x * A.u.s0 + (int64_t)y * A.u.s1 + z;
        if (x < A.bx0 || x >= A.bx1 || y < A.by0 || y >= A.by1 || z < A.bz0 || z >= A.bz1) return A.r.p[o];
        return residual_point<T, MGP_MODE_CONSISTENT>(A.u, o, A.f.p[o], (T)0, A.inv_h2);
    };
#pragma unroll 2
    for (int p = w; p < DF * DF; p += DW) {
        const int i = p / DF, j = p % DF;
        const int x = min(max(2 * I0 - 1 + i, 0), n0 - 1), y = min(max(2 * J0 - 1 + j, 0), n1 - 1);
        sr[i][j][lane] = residual(x, y, min(max(2 * K0 - 1 + lane, 0), n2 - 1));
    }
    for (int p = threadIdx.x; p < DF * DF; p += 64 * DW) {
        const int i = p / DF, j = p % DF;
        const int x = min(max(2 * I0 - 1 + i, 0), n0 - 1), y = min(max(2 * J0 - 1 + j, 0), n1 - 1);
        sr[i][j][DZ - 1] = residual(x, y, min(2 * K0 - 2 + DZ, n2 - 1));
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < DC * DC * DK / (64 * DW); m++) {
        const int t = threadIdx.x + m * 64 * DW;
        const int k = t % DK, j = (t / DK) % DC, i = t / (DK * DC);
        const int I = I0 + i, J = J0 + j, K = K0 + k;
        if (I >= A.c.n0 || J >= A.c.n1 || K >= A.c.n2) continue;
        // the 9 terms of one fine column in the reference's order, weights 1 2
        // 1 2 4 2 1 2 1 (in double, as its literals make them for either type)
        auto column = [&](int z) -> double {
            double v = sr[2 * i][2 * j][z];
            v = fma(2.0, (double)sr[2 * i][2 * j + 1][z], v);
            v = v + sr[2 * i][2 * j + 2][z];
            v = fma(2.0, (double)sr[2 * i + 1][2 * j][z], v);
            v = fma(4.0, (double)sr[2 * i + 1][2 * j + 1][z], v);
            v = fma(2.0, (double)sr[2 * i + 1][2 * j + 2][z], v);
            v = v + sr[2 * i + 2][2 * j][z];
            v = fma(2.0, (double)sr[2 * i + 2][2 * j + 1][z], v);
            v = v + sr[2 * i + 2][2 * j + 2][z];
            return v;
        };
        T v = (T)column(2 * k);
        v = (T)fma(2.0, column(2 * k + 1), (double)v);
        v = (T)((double)v + column(2 * k + 2));
        A.c.at(I, J, K) = (T)(v / 64.0);
    }
}

// ---------------------------------------------------------------------------
// The same for larger levels: one wave per tile of RJ coarse rows x 30 coarse
// columns marching along x (lane l = fine column 2 K0 - 2 + l, coarse column K
// on lane 2 (K - K0) + 2).  The 27-term sum is taken as its planes arrive: one
// running sum per coarse row and fine column instead of three planes of r, the
// three columns joined by two lane shifts per output, so three waves fit a SIMD
// where the march of mgp_sweep.hip runs two.  Measured against it, us: 257 x
// 257 x 129 FP64 54 / 65, FP32 33 / 41; 513 x 513 x 257 348 / 356, 184 / 200;
// 1025 x 1025 x 513 FP32 1363 / 1423.  There both are bound by the memory
// traffic of the shared rows: short marches (many waves close together in x)
// beat fewer warm-up planes; waves of a workgroup kept in step by a barrier
// per plane were slower (2.73-3.39 ms at 1025 x 1025 x 513 FP64).
template <class T>
struct MarchDescendArgs : DescendArgs<T> {
    int32_t ylo, yhi, zlo, zhi, xlo, xhi;  // allocated index ranges of the fine arrays
    int32_t ntiles, ntiles_pad, ichunk;    // coarse planes per wave
};

constexpr int MK = 30;  // coarse columns per wave

template <class T, int RJ, bool EDGE>
__device__ __forceinline__ void descend_march(const MarchDescendArgs<T>& A, int tl) {
    constexpr int NU = 2 * RJ + 3, NS = 2 * RJ + 1;
    const int lane = threadIdx.x;
    const int tz = tl % A.ztiles, ty = (tl / A.ztiles) % A.ytiles, tx = tl / (A.ztiles * A.ytiles);
    const int n0 = (int)A.u.n0, n1 = (int)A.u.n1, n2 = (int)A.u.n2;
    const int c0 = (int)A.c.n0, c1 = (int)A.c.n1, c2 = (int)A.c.n2;
    const int J0 = ty * RJ, K0 = tz * MK;
    const int Ia = tx * A.ichunk, Ib = min(c0, Ia + A.ichunk);
    const int64_t s0 = A.u.s0, s1 = A.u.s1;
    const uint32_t plane_bytes =
        (uint32_t)(((int64_t)(A.yhi - A.ylo) * s1 + (A.zhi - A.zlo) + 1) * (int64_t)sizeof(T));
    const int64_t corner = (int64_t)A.ylo * s1 + A.zlo;
    const int z = 2 * K0 - 2 + lane;
    const uint32_t zoff = (uint32_t)((min(max(z, A.zlo), A.zhi) - A.zlo) * (int)sizeof(T));
    const bool z_box = z >= A.bz0 && z < A.bz1;
    uint32_t roff[NU];
#pragma unroll
    for (int t = 0; t < NU; t++)
        roff[t] = (uint32_t)((int64_t)(min(max(2 * J0 - 2 + t, A.ylo), A.yhi) - A.ylo) * s1 * (int64_t)sizeof(T));
    auto rsrc = [&](const T* p, int i) {
        return plane_rsrc(p + (int64_t)min(max(i, A.xlo), A.xhi) * s0 + corner, plane_bytes);
    };
    auto load_u = [&](int i, T (&U)[NU]) {
        const __amdgpu_buffer_rsrc_t rs = rsrc(A.u.p, i);
#pragma unroll
        for (int t = 0; t < NU; t++) U[t] = bload<T>(rs, zoff, roff[t]);
    };
    auto load_f = [&](int i, T (&F)[NS]) {
        const __amdgpu_buffer_rsrc_t rs = rsrc(A.f.p, i);
#pragma unroll
        for (int t = 0; t < NS; t++) F[t] = bload<T>(rs, zoff, roff[t + 1]);
    };
    T Um[NU], U0[NU], Up[NU], UL[NU], F0[NS], FL[NS], R[NS];
    double acc[RJ];
    // r of fine plane i at rows 2 J0 - 1 + t: computed on the box, as stored
    // elsewhere in the shape, the clamped row's and lane's value outside it
    auto residual_plane = [&](int i) {
#pragma unroll
        for (int t = 0; t < NS; t++) {
            const T c = U0[t + 1];
            const T sum = ((Um[t + 1] - c) + (Up[t + 1] - c)) + ((U0[t] - c) + (U0[t + 2] - c)) +
                          ((lane_prev(c) - c) + (lane_next(c) - c));
            R[t] = fma(-A.inv_h2, sum, F0[t]);
        }
        if constexpr (EDGE) {
            const bool x_box = i >= A.bx0 && i < A.bx1;
            const __amdgpu_buffer_rsrc_t rs = rsrc(A.r.p, i);
#pragma unroll
            for (int t = 0; t < NS; t++) {
                const int y = 2 * J0 - 1 + t;
                const T st = bload<T>(rs, zoff, roff[t + 1]);
                R[t] = x_box && z_box && y >= A.by0 && y < A.by1 ? R[t] : st;
            }
#pragma unroll
            for (int t = 0; t < NS; t++) {
                const int y = 2 * J0 - 1 + t;
                if (y < 0 && t + 1 < NS) R[t] = R[t + 1];
                if (y >= n1 && t > 0) R[t] = R[t - 1];
                const T nx = lane_next(R[t]), pv = lane_prev(R[t]);
                R[t] = z == -1 ? nx : (z == n2 ? pv : R[t]);
            }
        }
    };
    // the terms of one plane, in order: weights 1 2 1 (a neighbouring plane) or
    // 2 4 2 (the middle one), in double as the reference's literals make them
    // (products with powers of two are exact)
    auto side = [&](bool first) {
#pragma unroll
        for (int j = 0; j < RJ; j++) {
            const double v = first ? (double)R[2 * j] : acc[j] + (double)R[2 * j];
            acc[j] = fma(2.0, (double)R[2 * j + 1], v) + (double)R[2 * j + 2];
        }
    };
    auto middle = [&]() {
#pragma unroll
        for (int j = 0; j < RJ; j++)
            acc[j] = fma(2.0, (double)R[2 * j + 2], fma(4.0, (double)R[2 * j + 1], fma(2.0, (double)R[2 * j], acc[j])));
    };
    const uint32_t cplane = (uint32_t)(((int64_t)(c1 - 1) * A.c.s1 + c2) * (int64_t)sizeof(T));
    const int K = K0 + (lane - 2) / 2;
    const bool k_out = lane >= 2 && lane <= 60 && (lane & 1) == 0 && K < c2;
    const uint32_t koff = k_out ? (uint32_t)(K * (int)sizeof(T)) : BUF_OOB;
    auto emit = [&](int I) {
        const __amdgpu_buffer_rsrc_t co = plane_rsrc(A.c.p + (int64_t)I * A.c.s0, cplane);
#pragma unroll
        for (int j = 0; j < RJ; j++) {
            T v = (T)lane_prev(acc[j]);
            v = (T)fma(2.0, acc[j], (double)v);
            v = (T)((double)v + lane_next(acc[j]));
            bstore((T)(v / 64.0), co, J0 + j < c1 ? koff : BUF_OOB,
                   (uint32_t)((int64_t)min(J0 + j, c1 - 1) * A.c.s1 * (int64_t)sizeof(T)));
        }
    };
    const int i0 = 2 * Ia - 1;  // first fine plane whose r is needed
    load_u(i0 - 1, Um);
    load_u(i0, U0);
    load_u(i0 + 1, Up);
    load_f(i0, F0);
#pragma unroll
    for (int j = 0; j < RJ; j++) acc[j] = 0.0;
    auto step = [&](int i) {
        load_u(i + 2, UL);
        load_f(i + 1, FL);
        residual_plane(i);
        if (i & 1) {
            if (i > i0) {  // the last plane of coarse plane (i - 1) / 2
                if (i < n0) side(false);
                if (i < n0) emit((i - 1) >> 1);
            }
            side(true);
        } else {
            if (i == 0) side(true);  // plane -1 is clamped to plane 0
            middle();
            if (i + 1 >= n0) {  // plane n0 is clamped to plane n0 - 1
                side(false);
                emit(i >> 1);
            }
        }
#pragma unroll
        for (int t = 0; t < NU; t++) Um[t] = U0[t], U0[t] = Up[t], Up[t] = UL[t];
#pragma unroll
        for (int t = 0; t < NS; t++) F0[t] = FL[t];
    };
    for (int i = i0; i <= 2 * Ib - 1; i++) step(i);
}

template <class T, int RJ>
__global__ void __launch_bounds__(64) k_resid_fw_march(MarchDescendArgs<T> A) {
    const int per_xcd = A.ntiles_pad / 8;
    const int tl = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (tl >= A.ntiles) return;
    const int tz = tl % A.ztiles, ty = (tl / A.ztiles) % A.ytiles, tx = tl / (A.ztiles * A.ytiles);
    const int J0 = ty * RJ, J1 = J0 + RJ, K0 = tz * MK, K1 = K0 + MK;
    const int Ia = tx * A.ichunk, Ib = min((int)A.c.n0, Ia + A.ichunk);
    const bool inner = 2 * J0 - 1 >= A.by0 && 2 * J1 - 1 < A.by1 && 2 * K0 - 1 >= A.bz0 && 2 * K1 - 1 < A.bz1 &&
                       2 * Ia - 1 >= A.bx0 && 2 * Ib - 1 < A.bx1 && J1 <= A.c.n1 && K1 <= A.c.n2;
    if (inner) descend_march<T, RJ, false>(A, tl);
    else descend_march<T, RJ, true>(A, tl);
}

template <class T>
static int march_descend(const DescendArgs<T>& D, const mgp_array* u, const mgp_array* cf, void* stream) {
    MarchDescendArgs<T> A;
    static_cast<DescendArgs<T>&>(A) = D;
    A.xlo = (int32_t)-u->halo[MGP_WEST], A.xhi = (int32_t)(u->shape[0] - 1 + u->halo[MGP_EAST]);
    A.ylo = (int32_t)-u->halo[MGP_SOUTH], A.yhi = (int32_t)(u->shape[1] - 1 + u->halo[MGP_NORTH]);
    A.zlo = (int32_t)-u->halo[MGP_BOTTOM], A.zhi = (int32_t)(u->shape[2] - 1 + u->halo[MGP_TOP]);
    const int64_t plane_bytes = ((int64_t)(A.yhi - A.ylo) * u->stride[1] + (A.zhi - A.zlo) + 1) * (int64_t)sizeof(T);
    const int64_t cplane = ((cf->shape[1] - 1) * cf->stride[1] + cf->shape[2]) * (int64_t)sizeof(T);
    if (plane_bytes >= (int64_t)BUF_OOB || cplane >= (int64_t)BUF_OOB) return MGP_ERR_ARG;
    constexpr int RJ = 4;
    const int64_t c0 = cf->shape[0];
    A.ytiles = (int32_t)((cf->shape[1] + RJ - 1) / RJ);
    A.ztiles = (int32_t)((cf->shape[2] + MK - 1) / MK);
    const int64_t tiles = (int64_t)A.ytiles * A.ztiles;
    // (the march of mgp_sweep.hip aims for half as many)
    int64_t chunks = std::max<int64_t>(1, 2 * target_wgs(g_fw_target) / std::max<int64_t>(tiles, 1));
    chunks = std::min<int64_t>(chunks, std::max<int64_t>(1, c0 / 2));
    A.ichunk = (int32_t)((c0 + chunks - 1) / chunks);
    A.ntiles = (int32_t)(tiles * ((c0 + A.ichunk - 1) / A.ichunk));
    A.ntiles_pad = (A.ntiles + 7) / 8 * 8;
    hipLaunchKernelGGL((k_resid_fw_march<T, RJ>), dim3(A.ntiles_pad), dim3(64), 0, (hipStream_t)stream, A);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MGP_OK : (int)e;
}

}  // namespace

template <class T>
int block_residual_fw(const mgp_array* u, const mgp_array* f, const mgp_array* r, const mgp_array* cf,
                      const int64_t b[6], double h, void* stream) {
    for (int d = 0; d < 3; d++)
        if (u->stride[d] != f->stride[d] || u->stride[d] != r->stride[d]) return MGP_ERR_ARG;
    DescendArgs<T> A;
    A.u = view_of<T>(*u);
    A.f = view_of<T>(*f);
    A.r = view_of<T>(*r);
    A.c = view_of<T>(*cf);
    A.bx0 = (int32_t)b[0], A.bx1 = (int32_t)b[1], A.by0 = (int32_t)b[2], A.by1 = (int32_t)b[3];
    A.bz0 = (int32_t)b[4], A.bz1 = (int32_t)b[5];
    A.inv_h2 = (T)(1.0 / (h * h));
    const int64_t pts = u->shape[0] * u->shape[1] * u->shape[2];
    // Large FP64 levels keep the taller tiles of mgp_sweep.hip, which re-read fewer
    // rows.  Running sums / taller tiles, us, over 70 random sizes from 2.5e7 points
    // on: below 5 * 2^24 points 1.5 % more to 11 % less (683 x 265 x 181 221 / 245, 513 x
    // 513 x 257 348 / 355), above from 2 % less to 11 % more (195 x 613 x 893 683 /
    // 616, 483 x 525 x 407 537 / 505, 1025 x 1025 x 513 2631 / 2598)
    if (sizeof(T) == 8 && pts >= (int64_t)5 << 24) return MGP_ERR_ARG;
    const int64_t xt = (cf->shape[0] + DC - 1) / DC;
    A.ytiles = (int32_t)((cf->shape[1] + DC - 1) / DC);
    A.ztiles = (int32_t)((cf->shape[2] + DK - 1) / DK);
    // FP64 blocks of which at most half the lanes have a coarse column, on levels that
    // take more than two of them per CU: march / blocks, us, 233 x 303 x 11 19.2 /
    // 27.3, 895 x 89 x 25 23.2 / 33.3, 443 x 89 x 17 14.8 / 18.1, 301 x 301 x 17 24.6 /
    // 33.4 (filled ones, 129 x 129 x 125: 20.4 / 19.0)
    const bool narrow = sizeof(T) == 8 && cf->shape[2] <= DK / 2 && xt * A.ytiles > 512;
    if (pts > g_fw_block_points || narrow) return march_descend<T>(A, u, cf, stream);
    hipLaunchKernelGGL(k_resid_fw_block<T>, dim3((unsigned)(xt * A.ytiles * A.ztiles)), dim3(64 * DW), 0,
                       (hipStream_t)stream, A);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MGP_OK : (int)e;
}
template int block_residual_fw<double>(const mgp_array*, const mgp_array*, const mgp_array*, const mgp_array*,
                                       const int64_t[6], double, void*);
template int block_residual_fw<float>(const mgp_array*, const mgp_array*, const mgp_array*, const mgp_array*,
                                      const int64_t[6], double, void*);

}  // namespace mgp
