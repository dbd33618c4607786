// Two GSRB sweeps of a small 3-D tile in one pass, for levels that live in
// cache and are bound by latency, not bandwidth: the tile and a halo wide
// enough for both sweeps are staged in LDS at once (one memory round trip), the
// four colour passes shrink over the halo (halo cells are recomputed, with the
// values the neighbouring tiles compute for them), and the tile is written out.
// A z-marching sweep of the same level takes two launches, each a serial chain
// of plane loads and barriers.  FP32, 64^3 and 32^3 levels in 32^3 boxes: sweep,
// sweep and restriction 8.5 + 10.1 + 7.5 us in three launches -> 10.7 us in one;
// the two post-smoothing sweeps 15.2 + 10.1 -> 9.9 us.  Shared by the level kernels (boxes of a layout,
// pm_block.hip) and the solve server (one periodic box a request,
// pm_serve.hip).
//
// The arithmetic, order and colouring are k_gsrb's; the input forms, the
// accumulated output and the residual restriction are those of k_gsrb_fused and
// k_residual_nb, so every value has the bits of the passes it replaces.
#pragma once

#include "pm_internal.hpp"

namespace pm {

// Tiles of at most 16 x 8 x 8 cells; 512 threads (two waves a SIMD) hide the
// LDS latency of a colour pass.  LDS: 8424 + 6144 values, 57 KB in FP32 (two
// workgroups a CU), 114 KB in FP64 (one).
constexpr int kBlkThreads = 512, kBlkX = 16, kBlkY = 8, kBlkZ = 8, kBlkHalo = 5;
constexpr int kBlkPhi = (kBlkX + 2 * kBlkHalo) * (kBlkY + 2 * kBlkHalo) * (kBlkZ + 2 * kBlkHalo);
constexpr int kBlkRhs = (kBlkX + 2 * kBlkHalo - 2) * (kBlkY + 2 * kBlkHalo - 2) * (kBlkZ + 2 * kBlkHalo - 2);

template<typename T>
struct BlockTile {
    int n[3];                   // cells of the box, even, at least 6 a side
    int t0[3], t[3];            // the tile: box-local low corner (even), size (even)
    int par;                    // parity of the box's low corner
    const T* in;                // staged input (IN 0, 2); element of cell (x, y, z) of neighbour box k:
    int ix, ixy;                //   s_in[k] + x + ix y + ixy z, likewise rhs and (IN 2) the coarse level
    const T* rhs;
    int rx, rxy;
    const T* crs;
    int cx, cxy;
    T* out;                     // cell (0, 0, 0) of the box
    double* acc;                // OUT 1: the same element of the FP64 solution
    int ox, oxy;
    T* crhs;                    // RES: the coarse cell under cell (0, 0, 0) of the box
    int qx, qxy;
    T c0, c1, lam;              // centre / neighbour coefficients, GSRB weight
    T r0, r1, avg;              // RES: residual coefficients, average weight
};

// Offsets of the 27 neighbouring boxes' cells (0, 0, 0), k = (ox + 1) + 3 (oy + 1)
// + 9 (oz + 1) with 13 the tile's own box.
struct BlockBases {
    int in[27], rhs[27], crs[27];
};

// IN 0: `in`; 1: the zero guess (not read); 2: `in` + the constant prolongation
// of crs.  OUT 1: add the result to acc instead of storing it.  RES: also write
// the residual restricted to the coarse right-hand side.
template<typename T, int IN, int OUT, int RES>
__device__ __forceinline__ void block_two_sweeps(const BlockTile<T>& B, const BlockBases& s, T* u, T* f)
{
    constexpr int H = RES ? 5 : 4, HR = H - 1;  // halo of phi; of rhs
    const int tid = threadIdx.x;
    const int W = B.t[0] + 2 * H, HY = B.t[1] + 2 * H, HZ = B.t[2] + 2 * H, P = W * HY;
    const int WR = W - 2, RY = HY - 2, RZ = HZ - 2, PR = WR * RY;
    // staging: 32 lanes a row, rows (y, z) 16 at a time, two sets of U rows in
    // flight a lane (the next set is loaded before a set is stored)
    const int col = tid & 31, rg = tid >> 5;
    constexpr int G = kBlkThreads / 32, U = 8;
    auto side = [](int v, int n) { return v < 0 ? 0 : (v >= n ? 2 : 1); };
    auto stage = [&](auto&& load, T* dst, int h, int w, int hy, int hz) {
        const int x = B.t0[0] - h + min(col, w - 1), kx = side(x, B.n[0]), xl = x - (kx - 1) * B.n[0];
        const int dq = small_div(G, hy), dm = G - dq * hy, rows = hy * hz;
        int zz = small_div(rg, hy), yy = rg - zz * hy;
        T v[2][U];
        auto fetch = [&](T (&d)[U]) {
#pragma unroll
            for (int i = 0; i < U; i++) {
                // rows past the end repeat the last plane, unstored
                const int y = B.t0[1] - h + yy, z = B.t0[2] - h + min(zz, hz - 1);
                const int ky = side(y, B.n[1]), kz = side(z, B.n[2]);
                d[i] = load(kx + 3 * ky + 9 * kz, xl, y - (ky - 1) * B.n[1], z - (kz - 1) * B.n[2]);
                yy += dm;
                zz += dq;
                if (yy >= hy) {
                    yy -= hy;
                    zz++;
                }
            }
        };
        auto store = [&](const T (&d)[U], int r0) {
            // row r of the staged block starts at w r
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int r = r0 + G * i;
                if (r < rows && col < w) { dst[col + __mul24(w, r)] = d[i]; }
            }
        };
        fetch(v[0]);
        for (int r0 = rg;;) {
            if (r0 + G * U < rows) { fetch(v[1]); }
            store(v[0], r0);
            r0 += G * U;
            if (r0 >= rows) { break; }
            if (r0 + G * U < rows) { fetch(v[0]); }
            store(v[1], r0);
            r0 += G * U;
            if (r0 >= rows) { break; }
        }
    };
    if constexpr (IN == 1) {
        for (int i = tid; i < P * HZ; i += kBlkThreads) { u[i] = 0; }
    } else {
        stage(
            [&](int k, int x, int y, int z) -> T {
                const T v = B.in[s.in[k] + x + __mul24(B.ix, y) + __mul24(B.ixy, z)];
                if constexpr (IN == 2) {
                    const T zero = 0;
                    return v + (zero + B.crs[s.crs[k] + (x >> 1) + __mul24(B.cx, y >> 1) + __mul24(B.cxy, z >> 1)]);
                } else {
                    return v;
                }
            },
            u, H, W, HY, HZ);
    }
    stage([&](int k, int x, int y, int z) -> T { return B.rhs[s.rhs[k] + x + __mul24(B.rx, y) + __mul24(B.rxy, z)]; }, f, HR, WR, RY, RZ);
    // the tile's cells this lane writes (16 lanes a row, 32 rows at a time)
    const int lx = tid & 15, lr = tid >> 4;
    constexpr int NO = (kBlkY * kBlkZ * 16 + kBlkThreads - 1) / kBlkThreads;
    double a64[NO];
    if constexpr (OUT == 1) {
#pragma unroll
        for (int i = 0; i < NO; i++) {
            const int r = lr + 32 * i, z = small_div(r, B.t[1]), y = r - z * B.t[1];
            a64[i] = 0;
            if (z < B.t[2] && lx < B.t[0]) {
                a64[i] = B.acc[(B.t0[0] + lx) + B.ox * (B.t0[1] + y) + B.oxy * (B.t0[2] + z)];
            }
        }
    }
    // one colour over the tile grown by e cells
    auto pass = [&](int e, int colour) {
        __syncthreads();
        const int hy = B.t[1] + 2 * e, rows = hy * (B.t[2] + 2 * e), pairs = (B.t[0] + 2 * e) >> 1;
        if (lx >= pairs) { return; }
        // row (yy, zz) of the grown tile, 32 rows on per turn: its elements of u and f
        const int dq = small_div(32, hy), dm = 32 - dq * hy;
        int zz = small_div(lr, hy), yy = lr - zz * hy;
        const int ustep = __mul24(dm, W) + __mul24(dq, P), uwrap = P - __mul24(hy, W);
        const int fstep = __mul24(dm, WR) + __mul24(dq, PR), fwrap = PR - __mul24(hy, WR);
        int ur = (2 * lx + H - e) + __mul24(W, yy + H - e) + __mul24(P, zz + H - e);
        int fr = (2 * lx + HR - e) + __mul24(WR, yy + HR - e) + __mul24(PR, zz + HR - e);
        const int p0 = B.par + B.t0[0] + B.t0[1] + B.t0[2] - 3 * e + colour;
        for (int r = lr; r < rows; r += 32) {
            const int d = (p0 + yy + zz) & 1, li = ur + d;
            T sv = 0;
            sv = sv + B.c0 * u[li];
            sv = sv + B.c1 * u[li + 1];
            sv = sv + B.c1 * u[li - 1];
            sv = sv + B.c1 * u[li + W];
            sv = sv + B.c1 * u[li - W];
            sv = sv + B.c1 * u[li + P];
            sv = sv + B.c1 * u[li - P];
            sv = sv + f[fr + d];
            u[li] = u[li] + B.lam * sv;
            yy += dm;
            zz += dq;
            ur += ustep;
            fr += fstep;
            if (yy >= hy) {
                yy -= hy;
                zz++;
                ur += uwrap;
                fr += fwrap;
            }
        }
    };
    pass(H - 1, 0);
    pass(H - 2, 1);
    pass(H - 3, 0);
    pass(H - 4, 1);
    __syncthreads();
    // the tile out, and its residual over its right-hand side
#pragma unroll
    for (int i = 0; i < NO; i++) {
        const int r = lr + 32 * i, z = small_div(r, B.t[1]), y = r - z * B.t[1];
        if (z < B.t[2] && lx < B.t[0]) {
            const int li = (lx + H) + W * (y + H) + P * (z + H);
            const int o = (B.t0[0] + lx) + B.ox * (B.t0[1] + y) + B.oxy * (B.t0[2] + z);
            if constexpr (OUT == 1) {
                B.acc[o] = a64[i] + (double)u[li];
            } else {
                B.out[o] = u[li];
            }
            if constexpr (RES) {
                const int fi = (lx + HR) + WR * (y + HR) + PR * (z + HR);
                T sv = 0;
                sv = sv + f[fi];
                sv = sv + B.r0 * u[li];
                sv = sv + B.r1 * u[li + 1];
                sv = sv + B.r1 * u[li - 1];
                sv = sv + B.r1 * u[li + W];
                sv = sv + B.r1 * u[li - W];
                sv = sv + B.r1 * u[li + P];
                sv = sv + B.r1 * u[li - P];
                f[fi] = sv;
            }
        }
    }
    if constexpr (RES) {
        __syncthreads();
        const int hx = B.t[0] >> 1, hy = B.t[1] >> 1, hz = B.t[2] >> 1;
        const int X = tid & 7, r = tid >> 3, Z = small_div(r, hy), Y = r - Z * hy;  // at most 8 x 4 x 4 coarse cells
        if (X < hx && Z < hz) {
            T a = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                a = a + B.avg * f[(2 * X + (k & 1) + HR) + WR * (2 * Y + ((k >> 1) & 1) + HR) + PR * (2 * Z + (k >> 2) + HR)];
            }
            B.crhs[((B.t0[0] >> 1) + X) + B.qx * ((B.t0[1] >> 1) + Y) + B.qxy * ((B.t0[2] >> 1) + Z)] = a;
        }
    }
}

// Tile sizes for boxes of n cells a side, `boxes` of them in the launch: even
// splits of at most 16 x 8 x 8 cells, thinner ones (which recompute more halo)
// while the launch would hold fewer than 128 tiles, one for every other CU.
inline void block_tiles(const int n[3], long boxes, int nt[3], int t[3])
{
    const int shapes[3][3] = {{kBlkX, kBlkY, kBlkZ}, {kBlkX, kBlkY, 4}, {kBlkX, 4, 4}};
    for (const auto& s : shapes) {
        long tiles = boxes;
        for (int d = 0; d < 3; d++) {
            nt[d] = (n[d] + s[d] - 1) / s[d];
            t[d] = ((n[d] + nt[d] - 1) / nt[d] + 1) & ~1;
            nt[d] = (n[d] + t[d] - 1) / t[d];
            tiles *= nt[d];
        }
        if (tiles >= 128) { return; }
    }
}

// ---------------------------------------------------------------- bottom
// The bottom of a V-cycle in one workgroup: the levels from a one-box periodic
// level of at most kBotCells cells down to the coarsest, phi and rhs of all of
// them in LDS (75 KB in FP64).  Bound by the LDS latency of its 28 colour passes
// (V(2,2) with 10 bottom sweeps from 16^3): FP32 18.2 us with 1024 threads, 21.3
// with 512, 30 with 256; as launches of their own these levels took 65 us (17 + 4
// + 4 + 17 + 22) and four more launch gaps.
constexpr int kBotThreads = 1024, kBotCells = 4096, kBotLevels = 4;
constexpr int kBotStore = kBotCells + kBotCells / 8 + kBotCells / 64 + kBotCells / 512;

template<typename T>
struct BottomLevel {
    int n[3];          // even
    T c0, c1, lam;     // sweeps
    T r0, r1;          // residual (all but the coarsest)
};

template<typename T>
struct BottomArgs {
    int nl, par;       // levels; parity of the top box's low corner (the coarser ones start at 0)
    int pre, post, bottom;
    BottomLevel<T> lv[kBotLevels];
    T avg;
};

// u, f: kBotStore values of LDS, level 0 of u and f loaded by the caller (u not
// where zero_in); on return u holds the cycle's result.  Every thread of the
// workgroup calls it.
template<typename T>
__device__ __forceinline__ void bottom_cycle(const BottomArgs<T>& A, T* u, T* f, bool zero_in)
{
    const int tid = threadIdx.x;
    constexpr int NP = kBotCells / 2 / kBotThreads;  // pairs of a thread
    auto relax = [&](const BottomLevel<T>& L, T* v, const T* q, int par, int nsw) {
        const int nx = L.n[0], ny = L.n[1], nz = L.n[2], hx = nx >> 1, np = hx * ny * nz;
        int xk[NP], row[NP], ym[NP], yp[NP], zm[NP], zp[NP], pr[NP];
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int p = min(tid + kBotThreads * i, np - 1), r = small_div(p, hx), z = small_div(r, ny), y = r - z * ny;
            xk[i] = 2 * (p - r * hx);
            row[i] = nx * (y + ny * z);
            ym[i] = nx * ((y == 0 ? ny - 1 : y - 1) + ny * z);
            yp[i] = nx * ((y == ny - 1 ? 0 : y + 1) + ny * z);
            zm[i] = nx * (y + ny * (z == 0 ? nz - 1 : z - 1));
            zp[i] = nx * (y + ny * (z == nz - 1 ? 0 : z + 1));
            pr[i] = par + y + z;
        }
        for (int h = 0; h < 2 * nsw; h++) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NP; i++) {
                if (tid + kBotThreads * i >= np) { continue; }
                const int x = xk[i] + ((pr[i] + h) & 1);
                const int xm = x == 0 ? nx - 1 : x - 1, xp = x == nx - 1 ? 0 : x + 1;
                const T cur = v[x + row[i]];
                T s = 0;
                s = s + L.c0 * cur;
                s = s + L.c1 * v[xp + row[i]];
                s = s + L.c1 * v[xm + row[i]];
                s = s + L.c1 * v[x + yp[i]];
                s = s + L.c1 * v[x + ym[i]];
                s = s + L.c1 * v[x + zp[i]];
                s = s + L.c1 * v[x + zm[i]];
                s = s + q[x + row[i]];
                v[x + row[i]] = cur + L.lam * s;
            }
        }
        __syncthreads();
    };
    int off = 0, par = A.par;
    for (int l = 0; l < A.nl; l++) {
        const BottomLevel<T>& L = A.lv[l];
        const int N = L.n[0] * L.n[1] * L.n[2];
        if (l > 0 || zero_in) {
            for (int i = tid; i < N; i += kBotThreads) { u[off + i] = 0; }
        }
        const bool last = l == A.nl - 1;
        relax(L, u + off, f + off, par, last ? A.bottom : A.pre);
        if (last) { break; }
        const int nx = L.n[0], ny = L.n[1], nz = L.n[2], hx = nx >> 1, hy = ny >> 1;
        const T* v = u + off;
        const T* q = f + off;
        for (int t = tid; t < N / 8; t += kBotThreads) {
            const int r = small_div(t, hx), Z = small_div(r, hy), X = t - r * hx, Y = r - Z * hy;
            const int nxy = nx * ny, xl = 2 * X, yr = nx * (2 * Y), zr = nxy * (2 * Z);
            // child coordinates -1, 0, 1, 2 of the 2 x 2 x 2 block, images folded in
            const int xs[4] = {xl == 0 ? nx - 1 : xl - 1, xl, xl + 1, xl + 2 == nx ? 0 : xl + 2};
            const int ys[4] = {yr == 0 ? nxy - nx : yr - nx, yr, yr + nx, yr + 2 * nx == nxy ? 0 : yr + 2 * nx};
            const int zs[4] = {zr == 0 ? nxy * (nz - 1) : zr - nxy, zr, zr + nxy, zr + 2 * nxy == nxy * nz ? 0 : zr + 2 * nxy};
            T a = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int i = 1 + (k & 1), j = 1 + ((k >> 1) & 1), m = 1 + (k >> 2);
                T s = 0;
                s = s + q[xs[i] + ys[j] + zs[m]];
                s = s + L.r0 * v[xs[i] + ys[j] + zs[m]];
                s = s + L.r1 * v[xs[i + 1] + ys[j] + zs[m]];
                s = s + L.r1 * v[xs[i - 1] + ys[j] + zs[m]];
                s = s + L.r1 * v[xs[i] + ys[j + 1] + zs[m]];
                s = s + L.r1 * v[xs[i] + ys[j - 1] + zs[m]];
                s = s + L.r1 * v[xs[i] + ys[j] + zs[m + 1]];
                s = s + L.r1 * v[xs[i] + ys[j] + zs[m - 1]];
                a = a + A.avg * s;
            }
            f[off + N + t] = a;
        }
        off += N;
        par = 0;
    }
    for (int l = A.nl - 2; l >= 0; l--) {
        const BottomLevel<T>& L = A.lv[l];
        const int nx = L.n[0], ny = L.n[1], N = nx * ny * L.n[2], hx = nx >> 1, hy = ny >> 1;
        const T* cu = u + off;
        off -= N;
        for (int i = tid; i < N; i += kBotThreads) {
            const int r = small_div(i, nx), z = small_div(r, ny), x = i - r * nx, y = r - z * ny;
            const T zero = 0;
            u[off + i] = u[off + i] + (zero + cu[(x >> 1) + hx * ((y >> 1) + hy * (z >> 1))]);
        }
        relax(L, u + off, f + off, l == 0 ? A.par : 0, A.post);
    }
}

}  // namespace pm
