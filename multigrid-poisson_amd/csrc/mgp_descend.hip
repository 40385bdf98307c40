// Residual and full-weighting restriction of small levels in one pass, on
// blocks (gfx950): coarse f = FW(f - L u), consistent mode
// (mgp_residual_restrict_fw_*; include/residual.h:58-79,
// include/fullweighting.h:59-121).
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

}  // namespace

template <class T>
int block_residual_fw(const mgp_array* u, const mgp_array* f, const mgp_array* r, const mgp_array* cf,
                      const int64_t b[6], double h, void* stream) {
    if (u->shape[0] * u->shape[1] * u->shape[2] > g_fw_block_points) return MGP_ERR_ARG;
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
    const int64_t xt = (cf->shape[0] + DC - 1) / DC;
    A.ytiles = (int32_t)((cf->shape[1] + DC - 1) / DC);
    A.ztiles = (int32_t)((cf->shape[2] + DK - 1) / DK);
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
