// Red-black Gauss-Seidel sweeps on workgroup tiles (gfx950): one or two sweeps
// per pass over memory, out of place (mgp_rbgs_sweep_*, mgp_rbgs_sweep2_*,
// mgp_rbgs_sweep2_prolong_*, mgp_rbgs_sweep2_from_zero_*).
//
// A workgroup of NW waves owns a (y, z) tile of NW * R rows x 128 columns and
// marches along x.  Wave w holds rows w R .. w R + R - 1; lane l holds the two
// columns z = zb + 2 l and zb + 2 l + 1 of each row, kept not by column but by
// colour: for every plane in flight one register array of the red points and
// one of the black points, one value per lane and row.  With
// p + y + z even for red, the points of one colour in rows t and t + 1 sit in
// different columns, so the colour-c values of a row are exactly the y
// neighbours, and those of a plane the x neighbours, of the other colour's
// points in the adjacent row or plane: a half-sweep reads and writes whole
// registers, without selects, and its only lane movement is one shift of the
// other colour's row for one of the two z neighbours.  The column a step
// updates in row t depends on the parity of the plane step alone, so the march
// is unrolled by two and the column is known at compile time.
//
// HS = 2 (one sweep) or 4 (two sweeps) half-sweep stages are in flight: at
// plane step i stage S updates plane i - S, S = 0 .. HS - 1 in that order
// (even S red, odd S black), then plane i - HS + 1 is written.  A stage reads
// the neighbouring planes after the stage before it and its own plane after
// the stage before it, which ran one step earlier: so what the waves need of
// each other's edge rows was final at the end of the previous step, and one
// barrier per plane step (edge rows published to LDS, two buffers) is all they
// share.  In y and z the tile loses one row and column per stage on each side
// (ring HS, recomputed by the neighbouring tiles); not at the box's own faces:
// the fixed points next to a Dirichlet face are in the tile and keep their
// values, and a Neumann ghost, sign*2h*g + mirror, is formed where a point next
// to it is updated, its mirror being the neighbour on the other side of that
// point (include/neumann.h:112-130; the refresh before each half-sweep,
// include/relaxation.h:25-90, sees that neighbour's current value).  Per point
// the operands and their order are those of the half-sweeps
// (include/gaussseidel.h:28-94), so the result is the same bits.
//
// Measured against the wave marches (mgp_sweep.hip), which recompute a ring
// around every wave's 8 rows and select lanes by colour: two sweeps at 1025 x
// 1025 x 513 FP64 3.50 against 4.52 ms (14.3 GB moved, 4.1 TB/s: bound by
// memory, where a plain 2-read-1-write stream over these arrays reaches 4.7
// TB/s), FP32 1.79 against 2.29 ms; with the correction 3.69 against 5.16 and
// 1.90 against 2.45 ms; 513 x 513 x 257 FP64 0.50 against 0.71 ms, 257 x 257 x
// 129 84 against 183 us (bound by instruction issue and the steps of a march);
// FP32 with Neumann z faces, 801 x 609 x 417, 0.80 against 2.45 ms.
//
// PRO: the trilinear prolongation of a coarse level is added to every plane as
// it arrives (include/vcycle.h:81-94, include/trilinearinterpolation.h:50-133):
// u + P(coarse) is what the sweeps start from.  ZIN: the input is zero and not
// read.
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

int64_t g_tile = 3;  // bit 0: one sweep, bit 1: two sweeps through the workgroup tiles

namespace {

constexpr int TZC = 128;  // columns per tile: two per lane
constexpr int PARTS = 4;  // most y tiles a narrow tile holds
constexpr int CUS = 256;  // compute units: one workgroup each at these register counts

template <class T>
struct TileArgs : MarchArgs<T> {
    int32_t parts;           // y tiles side by side in a tile of the last, narrow z column (1, 2 or 4)
    int32_t tiles;           // tiles of one x chunk
    int32_t yfirst, zfirst;  // first row and column of the first tiles: the box's, or the fixed ones before it
    uint32_t plane_bytes;
};

template <class T, int HS, int R, int NW, bool PRO>
struct TileShared {
    static constexpr int CR = R / 2 + 1;       // coarse rows under a wave's rows
    T x[2][NW][2][HS][64];                     // edge rows (first, last) for each stage of the next step
    T fz[2][4][PARTS * NW * R];                // sign*2h*g of the z faces per row of planes p & 3
    T fy[2][4][2][64];                         // of the y faces per column
    T c[PRO ? NW : 1][2][CR][2][PRO ? 64 : 1];  // the two coarse planes of each wave
};

// EDGE (what a tile has to take care of): 1: fixed columns next to the box's z
// faces; 2: Neumann z faces; 4: y faces; 8: several y tiles side by side
template <class T, int MODE, int HS, int R, int NW, bool PRO, bool ZIN, int EDGE, class SH>
__device__ __forceinline__ void tile_march(const TileArgs<T>& A, SH& sh, int xc, int ty, int tz, int parts) {
    constexpr int NR = R * NW;
    constexpr bool ZF = EDGE & 1, ZN = EDGE & 2, YF = EDGE & 4, PK = EDGE & 8;
    static_assert(R % 2 == 0, "the column of a row's colour alternates from row to row and wave to wave alike");
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n0 = (int)A.ui.n0, n1 = (int)A.ui.n1, n2 = (int)A.ui.n2;
    const int64_t s0 = A.ui.s0, s1 = A.ui.s1;
    const int bx0 = (int)A.bx0, bx1 = (int)A.bx1;
    // PK: lane l belongs to the y tile ty + l / (64 / parts); else there is one y
    // tile, and what depends on the row is uniform
    const int lp = 64 / parts;
    const int ll = PK ? lane & (lp - 1) : lane;
    const int part = PK ? lane / lp : 0;
    const int tyl = PK ? min(ty + part, A.ytiles - 1) : ty;
    const int yt = A.yfirst + tyl * (NR - 2 * HS);  // tile's first row
    const int yb = yt + w * R;                      // wave's first row
    const int zb = A.zfirst + tz * (TZC - 2 * HS);  // tile's first column
    const int xa = bx0 + xc * (int)A.xchunk, xb = min(bx1, xa + (int)A.xchunk);
    const T two_h = A.two_h;
    const int z = zb + 2 * ll;
    const uint32_t zoff = (uint32_t)(min(z, n2 - 2) * (int)sizeof(T));
    // the shape's last column as the first of its lane: loaded as the second
    // of the pair before it
    const bool zshift = ZF && z == n2 - 1;
    // byte offsets of row t: uniform (roff, the loads' and stores' scalar
    // offset), or per lane (PK, added to the lane's)
    const uint32_t rowb = (uint32_t)(s1 * (int64_t)sizeof(T));
    uint32_t roff[R];
#pragma unroll
    for (int t = 0; t < R; t++) roff[t] = PK ? 0u : (uint32_t)min(yb + t, n1 - 1) * rowb;
    const uint32_t row0 = PK ? (uint32_t)min(yb, n1 - 1) * rowb : 0u, rowl = (uint32_t)(n1 - 1) * rowb;
    auto voff = [&](int t) -> uint32_t { return PK ? zoff + min(row0 + (uint32_t)t * rowb, rowl) : zoff; };
    // rows and columns this tile writes
    const int ro0 = (tyl == 0 ? (int)A.by0 : yt + HS) - yb;
    const int ro1 = PK && ty + part >= A.ytiles ? ro0
                                                       : (tyl == A.ytiles - 1 ? (int)A.by1 : yt + NR - HS) - yb;
    const int co0 = tz == 0 ? (int)A.bz0 : zb + HS, co1 = tz == A.ztiles - 1 ? (int)A.bz1 : zb + TZC - HS;
    const uint32_t zst = z >= co0 && z + 1 < co1 ? zoff : BUF_OOB;  // both columns
    // one column only: the second (the first is fixed) or the first (the last of the box)
    const uint32_t zst0 = z < co0 && z + 1 >= co0 && z + 1 < co1 ? (uint32_t)((z + 1) * (int)sizeof(T)) : BUF_OOB;
    const uint32_t zst1 = z >= co0 && z + 1 == co1 ? (uint32_t)(z * (int)sizeof(T)) : BUF_OOB;

    // points outside the box keep their values; columns:
    const bool zin[2] = {z >= (int)A.bz0 && z < (int)A.bz1, z + 1 >= (int)A.bz0 && z + 1 < (int)A.bz1};
    // Neumann faces of the box in this tile: their ghosts are formed where a
    // point next to them is updated
    const int rhi = YF && A.by1 == n1 ? n1 - 1 - yb : -1;  // row of the high y face
    const bool has_ylo = YF && A.by0 == 0 && yb == 0;      // row 0
    const bool has_yhi = rhi >= 0 && rhi < R;
    const bool has_zlo = ZN && A.bz0 == 0 && tz == 0;      // column 0 of lane 0
    const bool has_zhi = ZN && A.bz1 == n2 && tz == A.ztiles - 1;
    const bool zl = has_zlo && ll == 0;
    const bool zh[2] = {has_zhi && z == n2 - 1, has_zhi && z + 1 == n2 - 1};
    bool yin[R];
#pragma unroll
    for (int t = 0; t < R; t++) yin[t] = yb + t >= (int)A.by0 && yb + t < (int)A.by1;
    const int wl = max(w - 1, 0), wh = min(w + 1, NW - 1);  // the waves below and above
    T gz[2], gy[2][2];
    auto load_faces = [&](int j) {  // face data of plane j (clamped into the shape)
        if constexpr (ZN || YF) {
            const int q = min(max(j, 0), n0 - 1);
            const uint32_t yo = (uint32_t)(min(yb + ll % R, n1 - 1) * (int)sizeof(T));
            const uint32_t zbytes = (uint32_t)(n1 * (int)sizeof(T)), ybytes = (uint32_t)(n2 * (int)sizeof(T));
            if (has_zlo) gz[0] = bload<T>(plane_rsrc(A.g[MGP_BOTTOM] + (int64_t)q * n1, zbytes), yo, 0);
            if (has_zhi) gz[1] = bload<T>(plane_rsrc(A.g[MGP_TOP] + (int64_t)q * n1, zbytes), yo, 0);
#pragma unroll
            for (int c = 0; c < (YF ? 2 : 0); c++) {
                const uint32_t zo = (uint32_t)(min(z + c, n2 - 1) * (int)sizeof(T));
                if (has_ylo) gy[0][c] = bload<T>(plane_rsrc(A.g[MGP_SOUTH] + (int64_t)q * n2, ybytes), zo, 0);
                if (has_yhi) gy[1][c] = bload<T>(plane_rsrc(A.g[MGP_NORTH] + (int64_t)q * n2, ybytes), zo, 0);
            }
        }
    };
    auto keep_faces = [&](int j) {  // sign*2h*g into plane j's slot
        if constexpr (ZN || YF) {
            if (ll < R) {
                if (has_zlo) sh.fz[0][j & 3][part * NR + w * R + ll] = (T)-1.0 * two_h * gz[0];
                if (has_zhi) sh.fz[1][j & 3][part * NR + w * R + ll] = (T)1.0 * two_h * gz[1];
            }
#pragma unroll
            for (int c = 0; c < (YF ? 2 : 0); c++) {
                if (has_ylo) sh.fy[0][j & 3][c][lane] = (T)-1.0 * two_h * gy[0][c];
                if (has_yhi) sh.fy[1][j & 3][c][lane] = (T)1.0 * two_h * gy[1][c];
            }
        }
    };

    // plane j into red (X[0]) and black (X[1]); par = parity of j + yb + zb (+
    // lin0 in reference mode): the red column of row t is par ^ (t & 1)
    auto load_u = [&](auto par, int j, T (&X)[2][R]) {
        if constexpr (ZIN) {
#pragma unroll
            for (int t = 0; t < R; t++) X[0][t] = X[1][t] = (T)0;
        } else {
            const __amdgpu_buffer_rsrc_t r = plane_rsrc(A.ui.p + (int64_t)min(max(j, 0), n0 - 1) * s0, A.plane_bytes);
#pragma unroll
            for (int t = 0; t < R; t++) {
                constexpr int P = decltype(par)::value;
                bload2<T>(r, voff(t), roff[t], X[P ^ (t & 1)][t], X[1 ^ P ^ (t & 1)][t]);
            }
        }
    };
    auto load_f = [&](auto par, int j, T (&X)[2][R]) {
        const __amdgpu_buffer_rsrc_t r = plane_rsrc(A.f.p + (int64_t)min(max(j, 0), n0 - 1) * s0, A.plane_bytes);
#pragma unroll
        for (int t = 0; t < R; t++) {
            constexpr int P = decltype(par)::value;
            bload2<T>(r, voff(t), roff[t], X[P ^ (t & 1)][t], X[1 ^ P ^ (t & 1)][t]);
        }
    };

    auto shift_columns = [&](auto par, T (&X)[2][R]) {
        if constexpr (ZF) {
            constexpr int P = decltype(par)::value;
#pragma unroll
            for (int t = 0; t < R; t++)
                X[P ^ (t & 1)][t] = zshift ? X[1 ^ P ^ (t & 1)][t] : X[P ^ (t & 1)][t];
        }
    };

    // PRO: coarse rows (yb >> 1) + b at the two coarse columns around the
    // lane's pair; the parities of yb and zb are those of by0 and bz0 (tiles
    // step by even counts).  Plane a lives in the wave's LDS slot a & 1; rows
    // outside the coarse shape read values that no update reads
    constexpr int CR = R / 2 + 1;
    T ct[CR][2];
    uint32_t coff[CR], cplane = 0;
    bool cshift = false;  // the first of the two is the coarse level's last column
    if constexpr (PRO) {
        const int q = min(z >> 1, (int)A.c.n2 - 2);
        cshift = ZF && (z >> 1) > q;
        cplane = (uint32_t)(((A.c.n1 - 1) * A.c.s1 + A.c.n2) * (int64_t)sizeof(T));
#pragma unroll
        for (int b = 0; b < CR; b++)
            coff[b] = (uint32_t)(((int64_t)min((yb >> 1) + b, (int)A.c.n1 - 1) * A.c.s1 + q) * (int64_t)sizeof(T));
    }
    auto load_coarse = [&](int a) {
        const __amdgpu_buffer_rsrc_t r =
            plane_rsrc(A.c.p + (int64_t)min(max(a, 0), (int)A.c.n0 - 1) * A.c.s0, cplane);
#pragma unroll
        for (int b = 0; b < CR; b++) bload2<T>(r, coff[b], 0, ct[b][0], ct[b][1]);
    };
    auto keep_coarse = [&](int a) {
#pragma unroll
        for (int b = 0; b < CR; b++) {
            sh.c[w][a & 1][b][0][lane] = cshift ? ct[b][1] : ct[b][0];
            sh.c[w][a & 1][b][1][lane] = ct[b][1];
        }
    };
    // X += P(coarse) on plane j: x-, then y-, then z-midpoints
    const bool py = yb & 1, pz = zb & 1;
    auto add_coarse = [&](auto par, int j, T (&X)[2][R]) {
        constexpr int P = decltype(par)::value;
        T v[CR][2];
#pragma unroll
        for (int b = 0; b < CR; b++)
#pragma unroll
            for (int c = 0; c < 2; c++) v[b][c] = sh.c[w][(j >> 1) & 1][b][c][lane];
        if (j & 1) {
#pragma unroll
            for (int b = 0; b < CR; b++)
#pragma unroll
                for (int c = 0; c < 2; c++)
                    v[b][c] = half_sum<T>(v[b][c], sh.c[w][((j >> 1) + 1) & 1][b][c][lane]);
        }
        auto rows = [&](auto pyc) {
            constexpr int PY = decltype(pyc)::value;
#pragma unroll
            for (int t = 0; t < R; t++) {
                const int b = (t + PY) >> 1;
                T y0 = v[b][0], y1 = v[b][1];
                if ((t + PY) & 1) {
                    y0 = half_sum<T>(y0, v[b + 1 < CR ? b + 1 : b][0]);
                    y1 = half_sum<T>(y1, v[b + 1 < CR ? b + 1 : b][1]);
                }
                const T m = half_sum<T>(y0, y1);
                X[P ^ (t & 1)][t] = X[P ^ (t & 1)][t] + (pz ? m : y0);          // first column
                X[1 ^ P ^ (t & 1)][t] = X[1 ^ P ^ (t & 1)][t] + (pz ? y1 : m);  // second column
            }
        };
        if (py) rows(std::integral_constant<int, 1>{});
        else rows(std::integral_constant<int, 0>{});
    };

    // U[k][colour]: plane i + 1 - k of step i; F[k][colour]: f of plane i - k
    T U[HS + 2][2][R], N[2][R], F[HS][2][R], FN[2][R];

    // edge rows of the stages of step i + 1 (off 0: planes counted for step i,
    // 1: for step i + 1)
    auto publish = [&](auto offc, int i) {
        constexpr int off = decltype(offc)::value;
#pragma unroll
        for (int S = 0; S < HS; S++) {
            const int Y = (S & 1) ^ 1;
            sh.x[i & 1][w][0][S][lane] = U[S + off][Y][0];
            sh.x[i & 1][w][1][S][lane] = U[S + off][Y][R - 1];
        }
    };
    // stage S of step i (par = parity of step i) with the other colour's rows
    // below and above the wave's; FAST: not at an x face of the box
    auto stage = [&](auto par, auto fast, auto Sc, int i) {
        constexpr int P = decltype(par)::value;
        constexpr bool FAST = decltype(fast)::value;
        constexpr int S = decltype(Sc)::value;
        constexpr int X = S & 1, Y = X ^ 1, K = S + 1;
        const int p = i - S;
        if constexpr (!FAST) {
            // from the first plane the chunk's output depends on
            if (p < max(bx0, xa - (HS - 1 - S)) || p >= bx1) return;
            // x-ghost planes: sign*2h*g + the plane on the other side (face (1, ny, nz))
            auto ghost = [&](const T* g, T sign, T (&to)[2][R], T (&from)[2][R]) {
                const __amdgpu_buffer_rsrc_t r = plane_rsrc(g, (uint32_t)(n1 * n2 * (int)sizeof(T)));
#pragma unroll
                for (int t = 0; t < R; t++) {
                    const uint32_t o = (uint32_t)(min(yb + t, n1 - 1) * n2 * (int)sizeof(T));
                    const uint32_t zo = (uint32_t)(min(z + (P ^ (t & 1)), n2 - 1) * (int)sizeof(T));
                    const T g = PK ? bload<T>(r, zo + o, 0) : bload<T>(r, zo, o);
                    to[Y][t] = sign * two_h * g + from[Y][t];
                }
            };
            if (p == 0 && A.g[MGP_WEST]) ghost(A.g[MGP_WEST], (T)-1.0, U[K + 1], U[K - 1]);
            if (p == n0 - 1 && A.g[MGP_EAST]) ghost(A.g[MGP_EAST], (T)1.0, U[K - 1], U[K + 1]);
        }
        const T lo = sh.x[(i - 1) & 1][wl][1][S][lane], hi = sh.x[(i - 1) & 1][wh][0][S][lane];
        T gzh[R], gzl[R], gyl = (T)0, gyh[2] = {(T)0, (T)0};
        if constexpr (ZN || YF) {
#pragma unroll
            for (int t = 0; t < R; t++) {
                gzh[t] = sh.fz[1][p & 3][part * NR + w * R + t];
                gzl[t] = sh.fz[0][p & 3][part * NR + w * R + t];
            }
        }
        if constexpr (YF) {
            gyl = sh.fy[0][p & 3][P][lane];  // row 0
            gyh[0] = sh.fy[1][p & 3][0][lane], gyh[1] = sh.fy[1][p & 3][1][lane];
        }
#pragma unroll
        for (int t = 0; t < R; t++) {
            const int c = P ^ (t & 1);  // column of the updated points
            const T vc = U[K][X][t], y = U[K][Y][t];
            T vB = c ? y : lane_prev(y), vT = c ? lane_next(y) : y;
            T vS = t > 0 ? U[K][Y][t - 1] : lo, vN = t < R - 1 ? U[K][Y][t + 1] : hi;
            if constexpr (ZN || YF) {
                vT = zh[c] ? gzh[t] + vB : vT;
                if (c == 0) vB = zl ? gzl[t] + vT : vB;
            }
            if constexpr (YF) {
                vN = t == rhi ? gyh[c] + vS : vN;
                if (t == 0) vS = has_ylo ? gyl + vN : vS;
            }
            const T v = relax_point<T, MODE>(vc, U[K + 1][Y][t], U[K - 1][Y][t], vS, vN, vB, vT, F[S][X][t],
                                             A.one_omega, A.omega_sixth, A.hsq);
            if (!ZF && !YF) U[K][X][t] = v;
            else if (!YF) U[K][X][t] = zin[c] ? v : vc;
            else U[K][X][t] = zin[c] && yin[t] ? v : vc;
        }
    };
    using Z = std::integral_constant<int, 0>;
    using O = std::integral_constant<int, 1>;
    auto step = [&](auto par, auto fast, int i) {
        constexpr bool FAST = decltype(fast)::value;
        constexpr int P = decltype(par)::value;
        using Q = std::integral_constant<int, 1 ^ P>;
        // what arrived during the step before, then the next loads: those the
        // next step keeps first come first (loads return in order)
        keep_faces(i);
        load_faces(i + 1);
        if constexpr (PRO) {
            if (i & 1) load_coarse(((i + 1) >> 1) + 1);
            else keep_coarse((i >> 1) + 1);
        }
        if constexpr (PRO) {
            // before the loads: their destinations and the correction's
            // values do not fit the registers together
            shift_columns(Q{}, U[0]);
            add_coarse(Q{}, i + 1, U[0]);
            __builtin_amdgcn_sched_barrier(0);
        }
        load_u(par, i + 2, N);
        load_f(Q{}, i + 1, FN);
        if constexpr (!ZIN && !PRO) shift_columns(Q{}, U[0]);
        shift_columns(par, F[0]);
        stage(par, fast, Z{}, i);
        if constexpr (HS == 4) {
            stage(par, fast, O{}, i);
            stage(par, fast, std::integral_constant<int, 2>{}, i);
        }
        publish(Z{}, i);
        stage(par, fast, std::integral_constant<int, HS - 1>{}, i);
        const int p = i - (HS - 1);
        if (FAST || (p >= xa && p < xb)) {
            const __amdgpu_buffer_rsrc_t ro = plane_rsrc(A.uo.p + (int64_t)p * s0, A.plane_bytes);
            auto put = [&](int t) {
                const int r = 1 ^ P ^ (t & 1);  // red column of row t on plane p (HS - 1 odd)
                const T a = U[HS][r ? 1 : 0][t], c = U[HS][r ? 0 : 1][t];
                const bool ok = !PK || (t >= ro0 && t < ro1);
                const uint32_t row = PK ? row0 + (uint32_t)t * rowb : 0u;
                bstore2(a, c, ro, ok ? zst + row : BUF_OOB, roff[t]);
                if constexpr (ZF) {
                    if (tz == 0) bstore(c, ro, ok ? zst0 + row : BUF_OOB, roff[t]);
                    if (tz == A.ztiles - 1) bstore(a, ro, ok ? zst1 + row : BUF_OOB, roff[t]);
                }
            };
            if (PK || (ro0 <= 0 && ro1 >= R)) {
#pragma unroll
                for (int t = 0; t < R; t++) put(t);
            } else if (ro1 > 0 && ro0 < R) {
#pragma unroll
                for (int t = 0; t < R; t++)
                    if (t >= ro0 && t < ro1) put(t);
            }
        }
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int t = 0; t < R; t++) {
#pragma unroll
                for (int k = HS + 1; k > 0; k--) U[k][c][t] = U[k - 1][c][t];
                U[0][c][t] = N[c][t];
#pragma unroll
                for (int k = HS - 1; k > 0; k--) F[k][c][t] = F[k - 1][c][t];
                F[0][c][t] = FN[c][t];
            }
        __syncthreads();
    };

    // first step: of even parity, at or before the first plane stage 0 is needed on
    const int base = A.yfirst + zb + (MODE == MGP_MODE_REFERENCE ? (int)(A.lin0 & 1) : 0);
    int i0 = xa - (HS - 1);
    i0 -= (i0 + base) & 1;
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int t = 0; t < R; t++) {
#pragma unroll
            for (int k = 3; k < HS + 2; k++) U[k][c][t] = (T)0;
#pragma unroll
            for (int k = 1; k < HS; k++) F[k][c][t] = (T)0;
        }
    load_u(O{}, i0 - 1, U[2]);
    load_u(Z{}, i0, U[1]);
    load_u(O{}, i0 + 1, U[0]);
    load_f(Z{}, i0, F[0]);
    load_faces(i0);
    if constexpr (!ZIN) {
        shift_columns(O{}, U[2]);
        shift_columns(Z{}, U[1]);
    }
    if constexpr (PRO) {
        // planes i0 - 1 and i0; plane i0 + 1 in the first step (whose even
        // case keeps the plane loaded last here)
        load_coarse((i0 - 1) >> 1);
        keep_coarse((i0 - 1) >> 1);
        load_coarse(((i0 - 1) >> 1) + 1);
        keep_coarse(((i0 - 1) >> 1) + 1);
        add_coarse(O{}, i0 - 1, U[2]);
        add_coarse(Z{}, i0, U[1]);
        if (!(i0 & 1)) load_coarse((i0 >> 1) + 1);
    }
    publish(O{}, i0 - 1);
    __syncthreads();
    // FP32: the steps whose stages are all inside the box, away from its x
    // faces, and write a plane run without the checks for either (1025 x 1025 x
    // 513, with the correction: 1.91 against 2.45 ms; in FP64 the copy without
    // checks spills and is slower, 3.89 against 3.69 ms)
    using Fast = std::integral_constant<bool, true>;
    using Full = std::integral_constant<bool, false>;
    [[maybe_unused]] const int f0 = max(xa, bx0 + 1) + HS - 1, f1 = min(bx1 - 2, xb + HS - 2);
    const int last = xb + HS - 2;
    int i = i0;
    if constexpr (sizeof(T) == 4) {
        for (; i <= last && i < f0; i += 2) step(Z{}, Full{}, i), step(O{}, Full{}, i + 1);
        for (; i + 1 <= f1; i += 2) step(Z{}, Fast{}, i), step(O{}, Fast{}, i + 1);
    }
    for (; i <= last; i += 2) step(Z{}, Full{}, i), step(O{}, Full{}, i + 1);
}

template <class T, int MODE, int HS, int R, int NW, bool PRO, bool ZIN>
__global__ void __launch_bounds__(64 * NW) k_rbgs_tile(TileArgs<T> A) {
    if ((int)blockIdx.x >= A.ntiles_pad) {
        copy_complement<T, PRO, ZIN>(A, (int)blockIdx.x - A.ntiles_pad);
        return;
    }
    // contiguous runs of tiles per XCD: neighbours share ring rows in one L2
    const int per_xcd = A.ntiles_pad / 8;
    const int tl = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (tl >= A.ntiles) return;
    __shared__ TileShared<T, HS, R, NW, PRO> sh;
    const int xc = tl / A.tiles, r = tl % A.tiles;
    // with several parts the last z column's tiles come first, then the others,
    // z fastest
    const int zw = A.parts > 1 ? A.ztiles - 1 : A.ztiles, packed = A.tiles - zw * A.ytiles;
    constexpr int ZFIX = 1, ZANY = 3, ANY = 7, PACK = 8;
    if (r < packed) {
        const int ty = r * A.parts, tz = A.ztiles - 1;
        if (ty == 0 || ty + A.parts >= A.ytiles || A.bz1 == A.ui.n2 || (tz == 0 && A.bz0 == 0))
            tile_march<T, MODE, HS, R, NW, PRO, ZIN, ANY | PACK>(A, sh, xc, ty, tz, A.parts);
        else
            tile_march<T, MODE, HS, R, NW, PRO, ZIN, ZFIX | PACK>(A, sh, xc, ty, tz, A.parts);
        return;
    }
    const int tz = (r - packed) % zw, ty = (r - packed) / zw;
    if (ty == 0 || ty == A.ytiles - 1) tile_march<T, MODE, HS, R, NW, PRO, ZIN, ANY>(A, sh, xc, ty, tz, 1);
    else if ((tz == 0 && A.bz0 == 0) || (tz == A.ztiles - 1 && A.bz1 == A.ui.n2))
        tile_march<T, MODE, HS, R, NW, PRO, ZIN, ZANY>(A, sh, xc, ty, tz, 1);
    else if (tz == 0 || tz == A.ztiles - 1) tile_march<T, MODE, HS, R, NW, PRO, ZIN, ZFIX>(A, sh, xc, ty, tz, 1);
    else tile_march<T, MODE, HS, R, NW, PRO, ZIN, 0>(A, sh, xc, ty, tz, 1);
}

}  // namespace

// x chunks per tile column: a chunk of n planes costs n + 2 (HS - 1) + 1 steps,
// and one workgroup runs per CU, so the count with the fewest steps over the
// rounds of CUS workgroups a launch takes
static int64_t tile_xchunk(int64_t tiles, int64_t nx, int hs) {
    int64_t best = nx, cost = INT64_MAX;
    for (int64_t c = 1; c <= nx && (c == 1 || tiles * c <= 16 * CUS); c++) {
        const int64_t len = (nx + c - 1) / c, n = tiles * ((nx + len - 1) / len);
        const int64_t t = (n + CUS - 1) / CUS * (len + 2 * (hs - 1) + 1);
        if (t < cost) cost = t, best = len;
    }
    return best;
}

// rows per wave and waves per workgroup: 4 x 8 leaves two waves per SIMD (two
// sweeps: FP64 256 registers, FP32 172).  Measured, two sweeps at 1025 x 1025 x
// 513: FP32 with 8 x 8 2.06 ms, with 4 x 16 1.94 ms, with 4 x 8 1.79 ms; FP64
// with 4 x 4 5.6 ms, with 4 x 8 3.5 ms (8 rows per wave spill)
constexpr int TR = 4, TW = 8;

// tiles of a launch of HS / 2 sweeps; pack: a narrow last z column's tiles hold
// several y tiles
template <class T, int HS>
static void tile_geometry(TileArgs<T>& A, const int64_t b[6], bool pack) {
    constexpr int NR = TR * TW;
    auto tiles_of = [&](int64_t n, int64_t cap) {
        return (int)(n <= cap ? 1 : 1 + (n - cap + cap - 2 * HS - 1) / (cap - 2 * HS));
    };
    A.ytiles = tiles_of(b[3] + (b[3] < A.ui.n1) - A.yfirst, NR);
    A.ztiles = tiles_of(b[5] + (b[5] < A.ui.n2) - A.zfirst, TZC);
    const int64_t cols = b[5] + (b[5] < A.ui.n2) - (A.zfirst + (int64_t)(A.ztiles - 1) * (TZC - 2 * HS));
    A.parts = 1;
    while (pack && A.parts < PARTS && cols * 2 * A.parts <= TZC && A.parts < A.ytiles) A.parts *= 2;
    A.tiles = A.parts > 1 ? (A.ztiles - 1) * A.ytiles + (A.ytiles + A.parts - 1) / A.parts : A.ztiles * A.ytiles;
    const int64_t nx = b[1] - b[0];
    A.xchunk = tile_xchunk(A.tiles, nx, HS);
    A.ntiles = (int)(A.tiles * ((nx + A.xchunk - 1) / A.xchunk));
    A.ntiles_pad = (A.ntiles + 7) / 8 * 8;
}

template <class T>
int tile_sweep(int mode, const mgp_array* ui, const mgp_array* uo, const mgp_array* f, const mgp_faces* faces,
               const int64_t b[6], double omega, int sweeps, void* stream, const mgp_array* coarse, bool zero_in) {
    if (!(g_tile & sweeps) || (ui->data == uo->data && !zero_in)) return MGP_ERR_ARG;
    if ((coarse || zero_in) && (mode != MGP_MODE_CONSISTENT || sweeps != 2)) return MGP_ERR_ARG;
    // a single sweep of a small level without Neumann faces: the wave march,
    // whose code is shorter to fetch (65^3: a solve of ten V-cycles 2.51 against
    // 2.59 ms; with Neumann faces the march takes 17 us, the tiles 11 us)
    const int64_t pts = (b[1] - b[0]) * (b[3] - b[2]) * (b[5] - b[4]);
    bool neumann = false;
    for (int q = 0; q < 6; q++) neumann = neumann || faces->type[q] == MGP_NEUMANN;
    if (sweeps == 1 && !neumann && pts < (int64_t)1 << 19) return MGP_ERR_ARG;
    // two FP32 sweeps of a flat level without Neumann faces, whose rows leave half of
    // the 32 of a tile empty (with the correction a quarter): the wave march, 8 rows to
    // a tile.  Tiles / march, us: 558 x 12 x 391 43 / 32, 593 x 9 x 191 35 / 27, from zero
    // 278 x 10 x 416 28 / 22, with the correction 457 x 9 x 503 60 / 34, 1059 x 15 x 149
    // 60 / 40, 345 x 23 x 207 43 / 33.  (FP64 levels as flat gain from tiles on average,
    // 5 to 24 %, though single ones lose; Neumann faces cost the march more.)
    if (sizeof(T) == 4 && sweeps == 2 && !neumann && b[3] - b[2] <= (coarse ? 24 : 16)) return MGP_ERR_ARG;
    TileArgs<T> A;
    A.ui = view_of<T>(*ui);
    A.uo = view_of<T>(*uo);
    A.f = view_of<T>(*f);
    A.c = coarse ? view_of<T>(*coarse) : A.ui;
    const int64_t n0 = A.ui.n0, n1 = A.ui.n1, n2 = A.ui.n2;
    for (int d = 0; d < 3; d++)
        if (f->stride[d] != ui->stride[d] || uo->stride[d] != ui->stride[d]) return MGP_ERR_ARG;
    if (n0 < 3 || n1 < 2 || n2 < 3 || n0 > (1 << 24) || n1 > (1 << 24) || n2 > (1 << 24)) return MGP_ERR_ARG;
    for (int q = 0; q < 6; q++) {
        A.g[q] = faces->type[q] == MGP_NEUMANN ? static_cast<const T*>(faces->g[q]) : nullptr;
        if (faces->type[q] == MGP_NEUMANN && !A.g[q]) return MGP_ERR_ARG;
    }
    A.yfirst = (int32_t)(b[2] - (b[2] > 0)), A.zfirst = (int32_t)(b[4] - (b[4] > 0));
    const int64_t bytes = ((n1 - 1) * A.ui.s1 + n2) * (int64_t)sizeof(T);
    if (bytes >= (int64_t)BUF_OOB) return MGP_ERR_ARG;
    A.plane_bytes = (uint32_t)bytes;
    if (coarse && (A.c.n2 < 2 || ((A.c.n1 - 1) * A.c.s1 + A.c.n2) * (int64_t)sizeof(T) >= (int64_t)BUF_OOB))
        return MGP_ERR_ARG;
    A.two_h = (T)(2.0 * faces->h);  // include/neumann.h:108
    A.bx0 = b[0], A.bx1 = b[1], A.by0 = b[2], A.by1 = b[3], A.bz0 = b[4], A.bz1 = b[5];
    A.lin0 = ui->halo[MGP_WEST] * ui->stride[0] + ui->halo[MGP_SOUTH] * ui->stride[1] + ui->halo[MGP_BOTTOM];
    const RelaxConsts<T> k(omega, faces->h);
    A.one_omega = k.one_omega, A.omega_sixth = k.omega_sixth, A.hsq = k.hsq;
    // Packing a narrow last z column (2^k + 1 points leave one of 9 to 33
    // columns) saves workgroups, but a packed one takes longer (its rows'
    // offsets are per lane), and in a large level, where memory and not the
    // steps per workgroup is the limit, it ends last.  Packed against not, us:
    // FP64 pair 257 x 257 x 129 84 / 121, 513 x 513 x 257 496 / 563, 1025 x 1025
    // x 513 3500 / 3504; FP64 with the correction 123 / 141, 746 / 627, 3987 /
    // 3695; FP32 pair 56 / 81, 294 / 327, 2043 / 1785; FP64 single sweep 52 /
    // 67, 417 / 443, 3102 / 3238
    const bool pack = sizeof(T) == 8 && sweeps == 1 ? true : pts < (int64_t)1 << (sizeof(T) == 8 && coarse ? 25 : 27);
    if (sweeps == 2) tile_geometry<T, 4>(A, b, pack);
    else tile_geometry<T, 2>(A, b, pack);
    constexpr int R = TR, NW = TW;
    const dim3 g(A.ntiles_pad + complement_blocks(A.ui, b, 64 * NW)), blk(64 * NW);
    const hipStream_t st = (hipStream_t)stream;
    const bool ref = mode == MGP_MODE_REFERENCE;
    constexpr int C = MGP_MODE_CONSISTENT, E = MGP_MODE_REFERENCE;
    if (coarse) hipLaunchKernelGGL((k_rbgs_tile<T, C, 4, R, NW, true, false>), g, blk, 0, st, A);
    else if (zero_in) hipLaunchKernelGGL((k_rbgs_tile<T, C, 4, R, NW, false, true>), g, blk, 0, st, A);
    else if (sweeps == 2 && ref) hipLaunchKernelGGL((k_rbgs_tile<T, E, 4, R, NW, false, false>), g, blk, 0, st, A);
    else if (sweeps == 2) hipLaunchKernelGGL((k_rbgs_tile<T, C, 4, R, NW, false, false>), g, blk, 0, st, A);
    else if (ref) hipLaunchKernelGGL((k_rbgs_tile<T, E, 2, R, NW, false, false>), g, blk, 0, st, A);
    else hipLaunchKernelGGL((k_rbgs_tile<T, C, 2, R, NW, false, false>), g, blk, 0, st, A);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MGP_OK : (int)e;
}
template int tile_sweep<double>(int, const mgp_array*, const mgp_array*, const mgp_array*, const mgp_faces*,
                                const int64_t[6], double, int, void*, const mgp_array*, bool);
template int tile_sweep<float>(int, const mgp_array*, const mgp_array*, const mgp_array*, const mgp_faces*,
                               const int64_t[6], double, int, void*, const mgp_array*, bool);

}  // namespace mgp
