// Two red-black Gauss-Seidel sweeps of a small level in one launch, on blocks
// (gfx950), out of place (mgp_rbgs_sweep2_*, mgp_rbgs_sweep2_prolong_*,
// mgp_rbgs_sweep2_from_zero_*).
//
// A level of a few hundred thousand points is bound by latency: a march along
// x (mgp_tile.hip) takes its warm-up planes one after the other.  Here a
// workgroup of 16 waves takes a block of 16 planes x 12 (FP64) or 16 (FP32)
// rows x 64 columns at once: wave w plane x = xs + w, lane l column z = zs + l,
// the rows in registers, so that
// the whole block is loaded in one go and a half-sweep is one barrier.  A
// thread keeps its points by colour: with s the parity that makes (x, 2 q + s,
// z) red, R[q] is that point and B[q] the other one of rows 2 q and 2 q + 1;
// the z neighbours of a point are then the other colour's [q] of the adjacent
// lanes (lane shifts), its x neighbours the other colour's [q] of the adjacent
// waves (LDS, an array per colour, published after each half-sweep), its y
// neighbours two of the thread's own.  Each half-sweep is valid one point
// further inside the block than the one before; the ring of 4 points is
// recomputed by the neighbouring blocks, except at the box's own faces, where fixed points are in the block and Neumann ghosts,
// sign*2h*g + mirror (include/neumann.h:112-130), are formed where they are
// used.  Operands and their order are those of the half-sweeps
// (include/gaussseidel.h:28-94), so the result is the same bits.
//
// Measured against the tiles' march, us (two sweeps / with the correction):
// 65 x 65 x 33 with Neumann x and y faces FP64 24 -> 15 / 32 -> 20, FP32 21 -> 12
// / 25 -> 14; 33^3 FP64 23 -> 11 / 32 -> 17.  A block inside the level holds 12288
// (FP64) or 16384 (FP32) points to write 8 x 4 x 56 = 1792 or 8 x 8 x 56 = 3584, its
// rings 5.9 or 3.6 times that, so a launch takes this form while one block per CU
// covers the level: 129 x 129 x 65 (992 blocks in FP64) takes 61 / 91 us, the march
// 39 / 47.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "mgp.h"
#include "mgp_device.h"
#include "mgp_point.h"
#include "mgp_sweep.h"
#include "mgp_wave.h"

namespace mgp {

int64_t g_block_count = 256;  // most blocks of a launch: one per compute unit

namespace {

constexpr int BL = 16, BZL = 64;  // planes and columns of a block
// row pairs per thread: 16 rows of FP64 do not fit the 128 registers (two sweeps
// of 65 x 65 x 33, Neumann x and y faces: 26.5 us with 16 rows, 15.2 us with 12)
template <class T>
constexpr int BQ = sizeof(T) == 8 ? 6 : 8;

template <class T>
struct BlockArgs : MarchArgs<T> {
    int32_t xfirst, yfirst, zfirst;  // first planes, rows and columns of the first blocks
    int32_t xtiles;
};

constexpr int HS = 4;  // half-sweeps

template <class T, int MODE, bool PRO, bool ZIN, bool NEU>
__device__ __forceinline__ void block_sweeps(const BlockArgs<T>& A, T (&sh)[2][BL][BQ<T>][64], T (&sz)[2][BL][2 * BQ<T>],
                                             int tx, int ty, int tz) {
    constexpr int BQ = mgp::BQ<T>, BY = 2 * BQ;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n0 = (int)A.ui.n0, n1 = (int)A.ui.n1, n2 = (int)A.ui.n2;
    const T two_h = A.two_h;
    const int xs = A.xfirst + tx * (BL - 2 * HS), ys = A.yfirst + ty * (BY - 2 * HS),
              zs = A.zfirst + tz * (BZL - 2 * HS);
    const int x = xs + w, z = zs + lane;
    // the points updated (not the block's outermost ones, unless they are the
    // box's) and those written
    const bool x0 = tx == 0, x1 = tx == A.xtiles - 1, y0 = ty == 0, y1 = ty == A.ytiles - 1, z0 = tz == 0,
               z1 = tz == A.ztiles - 1;
    const bool xu = x >= (x0 ? (int)A.bx0 : xs + 1) && x < (x1 ? (int)A.bx1 : xs + BL - 1);
    const bool zu = z >= (z0 ? (int)A.bz0 : zs + 1) && z < (z1 ? (int)A.bz1 : zs + BZL - 1);
    const int yu0 = (y0 ? (int)A.by0 : ys + 1) - ys, yu1 = (y1 ? (int)A.by1 : ys + BY - 1) - ys;
    const bool xw = x >= (x0 ? (int)A.bx0 : xs + HS) && x < (x1 ? (int)A.bx1 : xs + BL - HS);
    const bool zw = z >= (z0 ? (int)A.bz0 : zs + HS) && z < (z1 ? (int)A.bz1 : zs + BZL - HS);
    const int yw0 = (y0 ? (int)A.by0 : ys + HS) - ys, yw1 = (y1 ? (int)A.by1 : ys + BY - HS) - ys;

    const int lin = MODE == MGP_MODE_REFERENCE ? (int)(A.lin0 & 1) : 0;
    const int s = (x + ys + z + lin) & 1;  // rows 2 q + s are red
    const int xc = min(x, n0 - 1), zc = min(z, n2 - 1);
    // byte offsets within the arrays (from their first to their last point less
    // than BUF_OOB, checked by the launch): row y of the block, clamped into the
    // shape
    const uint32_t rowb = (uint32_t)(A.ui.s1 * (int64_t)sizeof(T));
    const uint32_t col = (uint32_t)(((int64_t)xc * A.ui.s0 + zc) * (int64_t)sizeof(T));
    const uint32_t row0 = col + (uint32_t)min(ys, n1 - 1) * rowb, rowl = col + (uint32_t)(n1 - 1) * rowb;
    const uint32_t bytes = (uint32_t)(((n0 - 1) * A.ui.s0 + (n1 - 1) * A.ui.s1 + n2) * (int64_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t ru = plane_rsrc(A.ui.p, bytes), rf = plane_rsrc(A.f.p, bytes);
    auto row = [&](int y) -> uint32_t { return min(row0 + (uint32_t)y * rowb, rowl); };

    T U[2][BQ], F[2][BQ];
#pragma unroll
    for (int q = 0; q < BQ; q++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const uint32_t o = row(2 * q + (s ^ c));
            U[c][q] = ZIN ? (T)0 : bload<T>(ru, o, 0);
            F[c][q] = bload<T>(rf, o, 0);
        }
    if constexpr (NEU) {
        // sign*2h*g of the z faces in the block's planes and rows (face (nx, ny, 1))
        for (int t = threadIdx.x; t < 2 * BL * BY; t += 64 * BL) {
            const int side = t / (BL * BY), i = (t / BY) % BL, j = t % BY;
            const T* g = A.g[side ? MGP_TOP : MGP_BOTTOM];
            if (g)
                sz[side][i][j] = (side ? (T)1.0 : (T)-1.0) * two_h *
                                 g[(int64_t)min(xs + i, n0 - 1) * n1 + min(ys + j, n1 - 1)];
        }
    }
    if constexpr (PRO) {
        // U += P(coarse): x-, then y-, then z-midpoints (include/
        // trilinearinterpolation.h:50-133); row b of the thread's coarse
        // column pair, y = ys + t between rows (t + py) >> 1 and the next
        constexpr int CR = BQ + 1;
        const int c1 = (int)A.c.n1, c2 = (int)A.c.n2;
        const int a0 = xc >> 1, a1 = min(a0 + 1, (int)A.c.n0 - 1);
        const uint32_t k0 = (uint32_t)((zc >> 1) * (int)sizeof(T)),
                       k1 = (uint32_t)(min((zc >> 1) + 1, c2 - 1) * (int)sizeof(T));
        const uint32_t crow = (uint32_t)(A.c.s1 * (int64_t)sizeof(T)), cplane = (uint32_t)(c1 - 1) * crow + c2 * sizeof(T);
        const __amdgpu_buffer_rsrc_t ra = plane_rsrc(A.c.p + (int64_t)a0 * A.c.s0, cplane),
                                     rb = plane_rsrc(A.c.p + (int64_t)a1 * A.c.s0, cplane);
        T v[CR][2];
#pragma unroll
        for (int b = 0; b < CR; b++) {
            const uint32_t j = (uint32_t)min((ys >> 1) + b, c1 - 1) * crow;
            v[b][0] = bload<T>(ra, k0, j), v[b][1] = bload<T>(ra, k1, j);
            if (xc & 1) {
                v[b][0] = half_sum<T>(v[b][0], bload<T>(rb, k0, j));
                v[b][1] = half_sum<T>(v[b][1], bload<T>(rb, k1, j));
            }
        }
        auto add = [&](auto pyc) {
            constexpr int PY = decltype(pyc)::value;
#pragma unroll
            for (int q = 0; q < BQ; q++) {
                T P[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int t = 2 * q + h, b = (t + PY) >> 1, e = b + 1 < CR ? b + 1 : b;
                    T l = v[b][0], r = v[b][1];
                    if ((t + PY) & 1) l = half_sum<T>(l, v[e][0]), r = half_sum<T>(r, v[e][1]);
                    P[h] = zc & 1 ? half_sum<T>(l, r) : l;
                }
                U[0][q] = U[0][q] + (s ? P[1] : P[0]);
                U[1][q] = U[1][q] + (s ? P[0] : P[1]);
            }
        };
        if (ys & 1) add(std::integral_constant<int, 1>{});
        else add(std::integral_constant<int, 0>{});
    }
    // Neumann faces next to this thread's points
    const T *gW = A.g[MGP_WEST], *gE = A.g[MGP_EAST];
    const bool wW = NEU && x == 0 && gW, wE = NEU && x == n0 - 1 && gE;
    const uint32_t n2b = (uint32_t)(n2 * (int)sizeof(T));
    const __amdgpu_buffer_rsrc_t rx = plane_rsrc(wW ? gW : gE, (uint32_t)n1 * n2b);
    const bool zf = NEU && ((z0 && A.g[MGP_BOTTOM]) || (z1 && A.g[MGP_TOP]));
    const bool yf = NEU && ((y0 && A.g[MGP_SOUTH]) || (y1 && A.g[MGP_NORTH]));
    const bool lB = NEU && z == 0 && A.g[MGP_BOTTOM], lT = NEU && z == n2 - 1 && A.g[MGP_TOP];
    T gS = (T)0, gN = (T)0;
    const int rS = NEU && A.g[MGP_SOUTH] ? -ys : -1, rN = NEU && A.g[MGP_NORTH] ? n1 - 1 - ys : -1;
    if (NEU && rS == 0) gS = (T)-1.0 * two_h * A.g[MGP_SOUTH][(int64_t)xc * n2 + zc];
    if (NEU && rN >= 0 && rN < BY) gN = (T)1.0 * two_h * A.g[MGP_NORTH][(int64_t)xc * n2 + zc];
    const int wm = max(w - 1, 0), wp = min(w + 1, BL - 1);

#pragma unroll
    for (int q = 0; q < BQ; q++) sh[1][w][q][lane] = U[1][q];
    __syncthreads();
    auto half_sweep = [&](auto Xc) {
        constexpr int X = decltype(Xc)::value, Y = X ^ 1;
        const bool odd = s ^ X;  // the updated points' rows are 2 q + odd
        // row 2 q + odd is updated where 2 q + yr < len.  What depends on the
        // row is formed again in each half-sweep: hidden from the optimiser,
        // which would keep it for every row, in more registers than there are
        const uint32_t len = zu ? (uint32_t)max(yu1 - yu0, 0) : 0u;
        int yo = odd;
        uint32_t go = (uint32_t)((zc + (ys + (int)odd) * n2) * (int)sizeof(T));  // x faces (1, ny, nz)
        asm volatile("" : "+v"(yo));
        if (NEU) asm volatile("" : "+v"(go));
        const uint32_t yr = (uint32_t)(yo - yu0);
        const T* zt = &sz[0][w][yo];  // z faces: [side][plane][row]
        if (xu) {
#pragma unroll
            for (int q = 0; q < BQ; q++) {
                const T below = q > 0 ? U[Y][q - 1] : (T)0, above = q + 1 < BQ ? U[Y][q + 1] : (T)0;
                T vW = sh[Y][wm][q][lane], vE = sh[Y][wp][q][lane];
                T vS = odd ? U[Y][q] : below, vN = odd ? above : U[Y][q];
                T vB = lane_prev(U[Y][q]), vT = lane_next(U[Y][q]);
                if constexpr (NEU) {
                    if (wE) vE = (T)1.0 * two_h * bload<T>(rx, go + (uint32_t)q * 2 * n2b, 0) + vW;
                    if (wW) vW = (T)-1.0 * two_h * bload<T>(rx, go + (uint32_t)q * 2 * n2b, 0) + vE;
                    if (yf) {
                        vN = 2 * q + yo == rN ? gN + vS : vN;
                        if (q == 0) vS = yo == rS ? gS + vN : vS;
                    }
                    if (zf) {
                        const T zT = zt[BL * BY + 2 * q], zB = zt[2 * q];
                        vT = lT ? zT + vB : vT;
                        vB = lB ? zB + vT : vB;
                    }
                }
                const T v = relax_point<T, MODE>(U[X][q], vW, vE, vS, vN, vB, vT, F[X][q], A.one_omega, A.omega_sixth,
                                                 A.hsq);
                U[X][q] = 2 * q + yr < len ? v : U[X][q];
                if (q & 1) __builtin_amdgcn_sched_barrier(0);  // (else all rows' operands are fetched at once, and spill)
            }
        }
    };
#pragma unroll 1
    for (int S = 0; S < HS; S += 2) {
        half_sweep(std::integral_constant<int, 0>{});
#pragma unroll
        for (int q = 0; q < BQ; q++) sh[0][w][q][lane] = U[0][q];
        __syncthreads();
        half_sweep(std::integral_constant<int, 1>{});
#pragma unroll
        for (int q = 0; q < BQ; q++) sh[1][w][q][lane] = U[1][q];
        __syncthreads();
    }
    if (xw && zw) {
        const __amdgpu_buffer_rsrc_t ro = plane_rsrc(A.uo.p, bytes);
        uint32_t r0 = row0;
        asm volatile("" : "+v"(r0));
#pragma unroll
        for (int q = 0; q < BQ; q++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int y = 2 * q + (s ^ c);
                bstore(U[c][q], ro, y >= yw0 && y < yw1 ? r0 + (uint32_t)y * rowb : BUF_OOB, 0);
            }
    }
}

template <class T, int MODE, bool PRO, bool ZIN>
__global__ void __launch_bounds__(64 * BL) k_rbgs_block(BlockArgs<T> A) {
    if ((int)blockIdx.x >= A.ntiles) {
        copy_complement<T, PRO, ZIN>(A, (int)blockIdx.x - A.ntiles);
        return;
    }
    __shared__ T sh[2][BL][BQ<T>][64];
    __shared__ T sz[2][BL][2 * BQ<T>];
    const int tl = (int)blockIdx.x;
    const int tz = tl % A.ztiles, ty = (tl / A.ztiles) % A.ytiles, tx = tl / (A.ztiles * A.ytiles);
    const bool neu = (tx == 0 && A.g[MGP_WEST]) || (tx == A.xtiles - 1 && A.g[MGP_EAST]) ||
                     (ty == 0 && A.g[MGP_SOUTH]) || (ty == A.ytiles - 1 && A.g[MGP_NORTH]) ||
                     (tz == 0 && A.g[MGP_BOTTOM]) || (tz == A.ztiles - 1 && A.g[MGP_TOP]);
    if (neu) block_sweeps<T, MODE, PRO, ZIN, true>(A, sh, sz, tx, ty, tz);
    else block_sweeps<T, MODE, PRO, ZIN, false>(A, sh, sz, tx, ty, tz);
}

}  // namespace

template <class T>
int block_sweep(int mode, const mgp_array* ui, const mgp_array* uo, const mgp_array* f, const mgp_faces* faces,
                const int64_t b[6], double omega, void* stream, const mgp_array* coarse, bool zero_in) {
    if (ui->data == uo->data && !zero_in) return MGP_ERR_ARG;
    if ((coarse || zero_in) && mode != MGP_MODE_CONSISTENT) return MGP_ERR_ARG;
    BlockArgs<T> A;
    A.ui = view_of<T>(*ui);
    A.uo = view_of<T>(*uo);
    A.f = view_of<T>(*f);
    A.c = coarse ? view_of<T>(*coarse) : A.ui;
    for (int d = 0; d < 3; d++)
        if (f->stride[d] != ui->stride[d] || uo->stride[d] != ui->stride[d]) return MGP_ERR_ARG;
    const int64_t n[3] = {A.ui.n0, A.ui.n1, A.ui.n2};
    if (n[0] < 3 || n[1] < 2 || n[2] < 2 || n[0] * n[1] * n[2] > (int64_t)1 << 24) return MGP_ERR_ARG;
    // u, f and the output are each addressed through one descriptor with 32-bit
    // offsets, whose masked stores need BUF_OOB to lie past the array: a window
    // into a larger array (strides wider than its shape) can span more.  The
    // coarse level is addressed plane by plane
    auto plane = [](const View<T>& v) { return ((v.n1 - 1) * v.s1 + v.n2) * (int64_t)sizeof(T); };
    if ((n[0] - 1) * A.ui.s0 * (int64_t)sizeof(T) + plane(A.ui) >= (int64_t)BUF_OOB) return MGP_ERR_ARG;
    if (coarse && plane(A.c) >= (int64_t)BUF_OOB) return MGP_ERR_ARG;
    for (int q = 0; q < 6; q++) {
        A.g[q] = faces->type[q] == MGP_NEUMANN ? static_cast<const T*>(faces->g[q]) : nullptr;
        if (faces->type[q] == MGP_NEUMANN && !A.g[q]) return MGP_ERR_ARG;
    }
    A.two_h = (T)(2.0 * faces->h);  // include/neumann.h:108
    A.bx0 = b[0], A.bx1 = b[1], A.by0 = b[2], A.by1 = b[3], A.bz0 = b[4], A.bz1 = b[5];
    A.lin0 = ui->halo[MGP_WEST] * ui->stride[0] + ui->halo[MGP_SOUTH] * ui->stride[1] + ui->halo[MGP_BOTTOM];
    const RelaxConsts<T> k(omega, faces->h);
    A.one_omega = k.one_omega, A.omega_sixth = k.omega_sixth, A.hsq = k.hsq;
    // blocks along an axis: the box and the fixed points next to it
    int32_t first[3], tiles[3];
    for (int d = 0; d < 3; d++) {
        const int64_t len = d == 2 ? BZL : d == 1 ? 2 * BQ<T> : BL;
        first[d] = (int32_t)(b[2 * d] - (b[2 * d] > 0));
        const int64_t ext = b[2 * d + 1] + (b[2 * d + 1] < n[d]) - first[d];
        tiles[d] = (int32_t)(ext <= len ? 1 : 1 + (ext - len + len - 2 * HS - 1) / (len - 2 * HS));
    }
    if ((int64_t)tiles[0] * tiles[1] * tiles[2] > g_block_count) return MGP_ERR_ARG;
    A.xfirst = first[0], A.yfirst = first[1], A.zfirst = first[2];
    A.xtiles = tiles[0], A.ytiles = tiles[1], A.ztiles = tiles[2];
    A.ntiles = A.ntiles_pad = tiles[0] * tiles[1] * tiles[2];
    A.xchunk = BL;
    const dim3 g(A.ntiles + complement_blocks(A.ui, b, 64 * BL)), blk(64 * BL);
    const hipStream_t st = (hipStream_t)stream;
    const bool ref = mode == MGP_MODE_REFERENCE;
    constexpr int C = MGP_MODE_CONSISTENT, E = MGP_MODE_REFERENCE;
    if (coarse) hipLaunchKernelGGL((k_rbgs_block<T, C, true, false>), g, blk, 0, st, A);
    else if (zero_in) hipLaunchKernelGGL((k_rbgs_block<T, C, false, true>), g, blk, 0, st, A);
    else if (ref) hipLaunchKernelGGL((k_rbgs_block<T, E, false, false>), g, blk, 0, st, A);
    else hipLaunchKernelGGL((k_rbgs_block<T, C, false, false>), g, blk, 0, st, A);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MGP_OK : (int)e;
}
template int block_sweep<double>(int, const mgp_array*, const mgp_array*, const mgp_array*, const mgp_faces*,
                                 const int64_t[6], double, void*, const mgp_array*, bool);
template int block_sweep<float>(int, const mgp_array*, const mgp_array*, const mgp_array*, const mgp_faces*,
                                const int64_t[6], double, void*, const mgp_array*, bool);



}  // namespace mgp
