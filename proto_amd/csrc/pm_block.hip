// Levels of the multigrid driver that live in cache: two sweeps with the
// residual restriction (or the prolongation) in one pass per level, and every
// level of at most 4096 cells in one launch (pm_block.hpp).
#include <algorithm>
#include <cmath>

#include "pm_block.hpp"
#include "pm_layout.hpp"

namespace pm {

// Shared of both passes: the level's geometry and the 27 neighbour bases.
template<typename T, int IN, int OUT, int RES>
__global__ __launch_bounds__(kBlkThreads) void k_level_block(LayoutDev L, G3 gi, G3 gr, G3 go, const T* __restrict__ in,
                                                            const T* __restrict__ rhs, T* __restrict__ out,
                                                            double* __restrict__ acc, LayoutDev C, G3 gc,
                                                            const T* __restrict__ crs, G3 gq, T* __restrict__ crhs,
                                                            BlockTile<T> B, int ntx, int nty, int ntz)
{
    __shared__ T u[kBlkPhi], f[kBlkRhs];
    __shared__ BlockBases s;
    // box by its position in the grid, so that every neighbour's index is one load
    const int tiles = ntx * nty * ntz;
    const int at_box = blockIdx.x / tiles, t = blockIdx.x - at_box * tiles;
    const int px = at_box % L.nb[0], pr = at_box / L.nb[0], py = pr % L.nb[1], pz = pr / L.nb[1];
    auto wrap = [](int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); };
    // box of C holding the coarse cell under fine box (x, y, z)'s low corner, and that cell's element
    auto under = [&](const G3& g, int x, int y, int z) {
        const int q[3] = {(x * L.bs[0]) >> 1, (y * L.bs[1]) >> 1, (z * L.bs[2]) >> 1};
        const int c[3] = {small_div(q[0], C.bs[0]), small_div(q[1], C.bs[1]), small_div(q[2], C.bs[2])};
        const int o = C.table[c[0] + C.nb[0] * (c[1] + C.nb[1] * c[2])];
        return o * gvol(C, g) + rel_index(C, g, q[0] - c[0] * C.bs[0], q[1] - c[1] * C.bs[1], q[2] - c[2] * C.bs[2]);
    };
    if (threadIdx.x < 27) {
        const int k = threadIdx.x;
        const int x = wrap(px + k % 3 - 1, L.nb[0]), y = wrap(py + (k / 3) % 3 - 1, L.nb[1]), z = wrap(pz + k / 9 - 1, L.nb[2]);
        const int o = L.table[x + L.nb[0] * (y + L.nb[1] * z)];
        if (IN != 1) { s.in[k] = (int)(o * gvol(L, gi) + rel_index(L, gi, 0, 0, 0)); }
        s.rhs[k] = (int)(o * gvol(L, gr) + rel_index(L, gr, 0, 0, 0));
        if (IN == 2) { s.crs[k] = (int)under(gc, x, y, z); }
    }
    const int b = L.table[at_box];
    const int tx = t % ntx, r = t / ntx, ty = r % nty, tz = r / nty;
    const int at[3] = {tx, ty, tz};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        B.n[d] = L.bs[d];
        B.t0[d] = at[d] * B.t[d];
        B.t[d] = min(B.t[d], L.bs[d] - B.t0[d]);
    }
    B.par = px * L.bs[0] + py * L.bs[1] + pz * L.bs[2];
    B.in = in;
    B.rhs = rhs;
    B.crs = crs;
    const long ob = b * gvol(L, go) + rel_index(L, go, 0, 0, 0);
    B.out = out + ob;
    B.acc = acc + ob;
    if (RES) {
        B.crhs = crhs + under(gq, px, py, pz);
    }
    __syncthreads();
    block_two_sweeps<T, IN, OUT, RES>(B, s, u, f);
}

// One periodic box: loads the top level, runs the cycle, writes the top level.
template<typename T>
__global__ __launch_bounds__(kBotThreads) void k_level_bottom(BottomArgs<T> A, G3 gp, T* __restrict__ phi,
                                                             const T* __restrict__ rhs, int zero_in)
{
    __shared__ T u[kBotStore], f[kBotStore];
    const int nx = A.lv[0].n[0], ny = A.lv[0].n[1], nz = A.lv[0].n[2], N = nx * ny * nz;
    const int X = nx + 2 * gp.g[0], Y = ny + 2 * gp.g[1];
    auto at = [&](int i) {
        const int r = small_div(i, nx), z = small_div(r, ny), x = i - r * nx, y = r - z * ny;
        return (x + gp.g[0]) + X * ((y + gp.g[1]) + Y * (z + gp.g[2]));
    };
    for (int i = threadIdx.x; i < N; i += kBotThreads) {
        f[i] = rhs[i];
        if (!zero_in) { u[i] = phi[at(i)]; }
    }
    bottom_cycle<T>(A, u, f, zero_in);
    for (int i = threadIdx.x; i < N; i += kBotThreads) { phi[at(i)] = u[i]; }
}

// coefficients as the sweeps' and the restriction's launches round them
template<typename T>
static void level_coefs(double dx, T* c0, T* c1, T* lam, T* r0, T* r1)
{
    double l = -(dx * dx) / (4.0 * 3);
    l *= 2.0;
    const double m = -1.0 / (dx * dx), hs = 1. / (dx * dx);
    if (sizeof(T) == 8) {
        *c0 = (T)(-6.0 * m);
        *c1 = (T)(1.0 * m);
    } else {
        *c0 = (T)-6.0 * (T)m;
        *c1 = (T)1.0 * (T)m;
    }
    *lam = (T)(1.0 * l);
    *r0 = (T)-6.0 * (T)(-hs);
    *r1 = (T)1.0 * (T)(-hs);
}

static bool covers_periodic(const pm_layout* L)
{
    return L->dim == 3 && L->nboxes == L->nb[0] * L->nb[1] * L->nb[2] && L->periodic[0] && L->periodic[1] &&
           L->periodic[2];
}

// Largest level: on 16 x 8 x 8 tiles the pass down does 3.7 times the updates, the one
// up 2.4 times (more on thinner tiles), and FP64 tiles leave one workgroup a CU, so
// they pay while launches and latency dominate.
// us of one V-cycle solve (10 cycles) with every level of up to 64^3 / 96^3 /
// 128^3 cells swept this way: FP32 cycles, 32^3 boxes, 128^3 cells: 2660 / 2667
// / 2413; 64^3 boxes (whose sweeps run the row-register kernels) 1752 / 1773 /
// 2408; FP64 cycles, 32^3 boxes 2882 / 2888 / 3455, 48^3 boxes, 96^3 cells:
// 1986 / 2215 / -.
bool level_block_ok(const pm_layout* L, const pm_layout* C, int dtype)
{
    if (!covers_periodic(L) || !levels_box_aligned(L, C)) { return false; }
    long cells = 1;
    for (int d = 0; d < 3; d++) {
        if (L->bs[d] < 6 || L->bs[d] % 2 || C->domain[d] * 2 != L->domain[d]) { return false; }
        cells *= L->domain[d];
    }
    const long side = dtype == PM_F32 && L->bs[0] != 64 ? 128 : 80;
    return cells <= side * side * side;
}

template<typename T>
static int block_launch(const pm_layout* L, const pm_layout* C, bool down, int in_mode, const void* in, const void* rhs,
                        void* out, double* acc, const void* crs, void* crhs, double dx, hipStream_t stream)
{
    const int g1[3] = {1, 1, 1};
    const G3 one = g3(g1), none = g3(nullptr);
    const G3 gi = down ? one : none, go = down ? none : one;
    BlockTile<T> B;
    int nt[3];
    block_tiles(L->bs, L->nboxes, nt, B.t);
    auto strides = [](const pm_layout* l, const G3& g, int* x, int* xy) {
        *x = l->bs[0] + 2 * g.g[0];
        *xy = *x * (l->bs[1] + 2 * g.g[1]);
    };
    strides(L, gi, &B.ix, &B.ixy);
    strides(L, none, &B.rx, &B.rxy);
    strides(C, one, &B.cx, &B.cxy);
    strides(L, go, &B.ox, &B.oxy);
    strides(C, none, &B.qx, &B.qxy);
    level_coefs<T>(dx, &B.c0, &B.c1, &B.lam, &B.r0, &B.r1);
    B.avg = (T)(1.0 / 8);
    const LayoutDev D = ldev(L), DC = ldev(C);
    const unsigned blocks = (unsigned)(nt[0] * nt[1] * nt[2] * L->nboxes);
    auto go_ = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kBlkThreads), 0, stream, D, gi, none, go, (const T*)in, (const T*)rhs,
                           (T*)out, acc, DC, one, (const T*)crs, none, (T*)crhs, B, nt[0], nt[1], nt[2]);
    };
    if (down) {
        if (in_mode == 1) { go_(k_level_block<T, 1, 0, 1>); } else { go_(k_level_block<T, 0, 0, 1>); }
    } else if (acc) {
        if constexpr (sizeof(T) == 4) { go_(k_level_block<T, 2, 1, 0>); }
    } else {
        go_(k_level_block<T, 2, 0, 0>);
    }
    PM_CHECK_LAUNCH();
    return PM_OK;
}

int level_block_down(const pm_layout* L, const pm_layout* C, int dtype, const void* phi, int zero_in, void* tmp,
                     const void* rhs, double dx, void* crhs, hipStream_t stream)
{
    return dtype == PM_F64 ? block_launch<double>(L, C, true, zero_in, phi, rhs, tmp, nullptr, nullptr, crhs, dx, stream)
                           : block_launch<float>(L, C, true, zero_in, phi, rhs, tmp, nullptr, nullptr, crhs, dx, stream);
}

int level_block_up(const pm_layout* L, const pm_layout* C, int dtype, const void* tmp, const void* cphi, void* phi,
                   double* acc, const void* rhs, double dx, hipStream_t stream)
{
    PM_REQUIRE(!acc || dtype == PM_F32, "multigrid: the FP64 accumulation is for FP32 sweeps");
    return dtype == PM_F64 ? block_launch<double>(L, C, false, 2, tmp, rhs, phi, nullptr, cphi, nullptr, dx, stream)
                           : block_launch<float>(L, C, false, 2, tmp, rhs, phi, acc, cphi, nullptr, dx, stream);
}

template<typename T>
static int bottom_launch(const std::vector<const pm_layout*>& lv, const std::vector<double>& dx, int pre, int post,
                         int bottom, void* phi, const void* rhs, bool zero_in, hipStream_t stream)
{
    BottomArgs<T> A;
    A.nl = (int)lv.size();
    A.par = lv[0]->lows[0] + lv[0]->lows[1] + lv[0]->lows[2];
    A.pre = pre;
    A.post = post;
    A.bottom = bottom;
    A.avg = (T)(1.0 / 8);
    for (int l = 0; l < A.nl; l++) {
        BottomLevel<T>& B = A.lv[l];
        for (int d = 0; d < 3; d++) { B.n[d] = lv[l]->bs[d]; }
        level_coefs<T>(dx[l], &B.c0, &B.c1, &B.lam, &B.r0, &B.r1);
    }
    const int g1[3] = {1, 1, 1};
    hipLaunchKernelGGL(k_level_bottom<T>, dim3(1), dim3(kBotThreads), 0, stream, A, g3(g1), (T*)phi, (const T*)rhs,
                       zero_in ? 1 : 0);
    PM_CHECK_LAUNCH();
    return PM_OK;
}

int level_bottom(const std::vector<const pm_layout*>& lv, const std::vector<double>& dx, int dtype, int pre, int post,
                 int bottom, void* phi, const void* rhs, bool zero_in, hipStream_t stream)
{
    bool ok = !lv.empty() && lv.size() <= (size_t)kBotLevels;
    for (size_t l = 0; l < lv.size() && ok; l++) {
        const pm_layout* L = lv[l];
        ok = covers_periodic(L) && L->nboxes == 1 && (long)L->bs[0] * L->bs[1] * L->bs[2] <= (kBotCells >> (3 * l));
        for (int d = 0; d < 3 && ok; d++) {
            ok = L->bs[d] % 2 == 0 && (l == 0 || L->bs[d] * 2 == lv[l - 1]->bs[d]);
        }
    }
    if (!ok) { return PM_ERR_UNSUPPORTED; }
    return dtype == PM_F64 ? bottom_launch<double>(lv, dx, pre, post, bottom, phi, rhs, zero_in, stream)
                           : bottom_launch<float>(lv, dx, pre, post, bottom, phi, rhs, zero_in, stream);
}

}  // namespace pm
