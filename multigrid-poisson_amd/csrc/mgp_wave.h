// Device helpers shared by the marching kernels (mgp_sweep.hip, mgp_tile.hip):
// their argument block, the copy of the shape points outside the box, lane
// moves and buffer-resource access.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mgp.h"
#include "mgp_device.h"
#include "mgp_point.h"

namespace mgp {
namespace {

template <class T>
struct MarchArgs {
    View<T> ui, uo, f;
    View<T> c;  // coarse level whose prolongation the pass adds first (two-sweep pass only)
    const T* g[6];
    T two_h;
    int64_t bx0, bx1, by0, by1, bz0, bz1;
    int64_t lin0;
    T one_omega, omega_sixth, hsq;
    int ytiles, ztiles, ntiles, ntiles_pad;
    int64_t xchunk;
};

// The shape points outside the box, copied from ui to uo by extra blocks of a
// sweep launch (the blocks after the tiles): an out-of-place pass then leaves
// a complete image of what the in-place half-sweeps leave, whichever of the
// two buffers ends up current (the boundary points' own history of updates,
// signs of zero included, stays with the solution).  The halo is not copied:
// ghost values are formed again before every use.
constexpr int COPY_PER_THREAD = 8;

template <class T>
inline int64_t complement_points(const View<T>& u, const int64_t b[6]) {
    const int64_t BX = b[1] - b[0], BY = b[3] - b[2];
    return (b[0] + u.n0 - b[1]) * u.n1 * u.n2 + BX * (b[2] + u.n1 - b[3]) * u.n2 + BX * BY * (b[4] + u.n2 - b[5]);
}
template <class T>
inline int complement_blocks(const View<T>& u, const int64_t b[6], int threads) {
    const int64_t per = (int64_t)threads * COPY_PER_THREAD;
    return (int)((complement_points(u, b) + per - 1) / per);
}

// points [blk * blockDim * COPY_PER_THREAD, ...) of the complement, in the
// order: x outside the box (whole planes), then y outside (box planes), then
// z outside (box rows); consecutive threads take consecutive z where it runs.
// PRO: ui + P(coarse) instead of ui (the pass that adds the prolongation);
// ZERO: 0 (the pass whose input is zero and not read)
template <class T, bool PRO = false, bool ZERO = false>
__device__ __forceinline__ void copy_complement(const MarchArgs<T>& A, int blk) {
    const int64_t n0 = A.ui.n0, n1 = A.ui.n1, n2 = A.ui.n2;
    const int64_t BX = A.bx1 - A.bx0, BY = A.by1 - A.by0;
    const int64_t xo = A.bx0 + n0 - A.bx1, yo = A.by0 + n1 - A.by1, zo = A.bz0 + n2 - A.bz1;
    const int64_t c1 = xo * n1 * n2, c2 = BX * yo * n2, c3 = BX * BY * zo;
    const int64_t per = (int64_t)blockDim.x * COPY_PER_THREAD;
    const int64_t end = min(c1 + c2 + c3, (int64_t)(blk + 1) * per);
    for (int64_t t = (int64_t)blk * per + threadIdx.x; t < end; t += blockDim.x) {
        int64_t x, y, z;
        if (t < c1) {
            const int64_t a = t / (n1 * n2), r = t % (n1 * n2);
            x = a < A.bx0 ? a : A.bx1 + (a - A.bx0);
            y = r / n2;
            z = r % n2;
        } else if (t < c1 + c2) {
            const int64_t u = t - c1, a = u / (yo * n2), r = u % (yo * n2), c = r / n2;
            x = A.bx0 + a;
            y = c < A.by0 ? c : A.by1 + (c - A.by0);
            z = r % n2;
        } else {
            const int64_t u = t - c1 - c2, a = u / (BY * zo), r = u % (BY * zo), c = r % zo;
            x = A.bx0 + a;
            y = A.by0 + r / zo;
            z = c < A.bz0 ? c : A.bz1 + (c - A.bz0);
        }
        if (ZERO)
            A.uo.at(x, y, z) = (T)0;
        else if (PRO)
            A.uo.at(x, y, z) = A.ui.at(x, y, z) + trilinear<T>(A.c, x, y, z);
        else
            A.uo.at(x, y, z) = A.ui.at(x, y, z);
    }
}

// DPP lane move of a 32- or 64-bit value with bound_ctrl: a lane whose source
// lane lies outside the wave reads 0.  No old value is involved, so the
// compiler emits no initialising move before each DPP move.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    typedef int i32x2 __attribute__((ext_vector_type(2)));
    i32x2 w = __builtin_bit_cast(i32x2, v);
    w.x = __builtin_amdgcn_mov_dpp(w.x, CTRL, 0xf, 0xf, true);
    w.y = __builtin_amdgcn_mov_dpp(w.y, CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, w);
}
template <class T>
__device__ __forceinline__ T lane_prev(T v) {  // value of lane l-1 (z - 1); 0 on lane 0
    return dpp_move<0x138>(v);                 // wave_shr:1
}
template <class T>
__device__ __forceinline__ T lane_next(T v) {  // value of lane l+1 (z + 1); 0 on lane 63
    return dpp_move<0x130>(v);                 // wave_shl:1
}

// Buffer-resource access (SGPR descriptor + 32-bit lane offset + SGPR row
// offset): no per-lane address arithmetic.  A lane offset at or beyond the
// record count drops the store in hardware, which masks stores without
// branches; only the lane (VGPR) offset is used for that, since the range
// check does not cover the SGPR offset.  Loads always use in-range offsets.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t BUF_OOB = 0x40000000u;  // offset past any plane (planes < 1 GiB)
// cache-policy bits of the buffer loads and stores (gfx950: bit 0 sc0, bit 1
// nt, bit 4 sc1); a build-time choice, measured per kernel
#ifndef MGP_LOAD_POLICY
#define MGP_LOAD_POLICY 0
#endif
#ifndef MGP_STORE_POLICY
#define MGP_STORE_POLICY 0
#endif

__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}
template <class T>
__device__ __forceinline__ T bload(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff);
template <>
__device__ __forceinline__ double bload<double>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, MGP_LOAD_POLICY));
}
template <>
__device__ __forceinline__ float bload<float>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, MGP_LOAD_POLICY));
}
__device__ __forceinline__ void bstore(double v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, (int)voff, (int)soff, MGP_STORE_POLICY);
}
__device__ __forceinline__ void bstore(float v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, (int)voff, (int)soff,
                                          MGP_STORE_POLICY);
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// two adjacent values of a row (no alignment beyond the element's)
template <class T>
__device__ __forceinline__ void bload2(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, T& a, T& b) {
    if constexpr (sizeof(T) == 8) {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
        a = __builtin_bit_cast(double, (u32x2){v.x, v.y});
        b = __builtin_bit_cast(double, (u32x2){v.z, v.w});
    } else {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
        const unsigned int x = v.x, y = v.y;  // (a bit cast of the component itself reads v.x for both)
        a = __builtin_bit_cast(float, x);
        b = __builtin_bit_cast(float, y);
    }
}
__device__ __forceinline__ void bstore2(double a, double b, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    const u32x2 x = __builtin_bit_cast(u32x2, a), y = __builtin_bit_cast(u32x2, b);
    __builtin_amdgcn_raw_buffer_store_b128((u32x4){x.x, x.y, y.x, y.y}, r, (int)voff, (int)soff, 0);
}
__device__ __forceinline__ void bstore2(float a, float b, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b64(
        (u32x2){__builtin_bit_cast(unsigned int, a), __builtin_bit_cast(unsigned int, b)}, r, (int)voff, (int)soff, 0);
}

}  // namespace
}  // namespace mgp
