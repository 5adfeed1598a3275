// d2q9_adjoint.hip -- channel step with a partial bounce-back obstacle
// (per-node solid fraction s in [0,1]) and its hand-written discrete adjoint.
//
// Forward iteration t (t >= 1), node x, in deviations h = f - w:
//   h   = pull(H_{t-1}) with the Zou-He plan of the channel apps
//         (turek.py:112-125: velocity walls bottom/top at rest, velocity
//         inlet u = a_{t-1} * profile on the left, pressure outlet on the
//         right, the four corners; nb.py:121-344)
//   c   = TRT collision of h (nb.py:7-35, written on deviations)
//   H_t = (1 - s) c + s h_bar          (partial bounce-back: h_bar_q = h_{ns[q]})
//   D_t = sum_x s sum_q c_qx (c_q - h_bar_q)   (momentum taken from the fluid)
// Iteration 0 starts from rest (h = 0, so H_0 = 0 for every s).
// Loss L = mean of D_t over the last `window` iterations.
//
// Adjoint iteration t, given lam_t = dL/dH_t, recomputes h, c at every node
// from H_{t-1} and forms
//   cbar = (1-s) lam + W s cx,   hbar = s lam_bar + W s cx,
//   sbar += lam . (h_bar - c) + W cx . (c - h_bar),
//   hbar += cbar - Om cbar + rhobar + c . jbar     (TRT + equilibrium VJP),
// then pushes hbar back along -c_q (the transpose of the pull); boundary
// nodes first apply the transpose of their (affine) Zou-He map, columns
// evaluated exactly, and the inlet nodes accumulate dL/da.
#include "d2q9_tile.h"

#include <algorithm>
#include <memory>
#include <vector>

namespace lbm {
namespace {

struct PbbParams {
    int nx, ny, N;
    double om_p, om_m, rho_out;
    const double *prof;     // [2][ny] inlet profile of unit amplitude
    const void *s;          // solid fraction [N]
};

// A launch advances n = K - lev0 iterations (entry j of the arrays: its j-th)
// on the tiles of a plan (d2q9_plan.h).
struct PbbFwd {
    PbbParams p;
    const void *src;        // state before the first iteration
    char *dst;              // state after the last one ...
    size_t stride;          // ... or, if not 0, after each, `stride` bytes apart
    double *drag_part;      // [n][gridDim.x] drag sums of the tiles, or null
    double amp[TILE_MAX_LEVELS];    // inlet amplitude a_{t-1}
    int K, lev0;
};
struct PbbAdj {
    PbbParams p;
    const void *h[TILE_MAX_LEVELS];     // H_{t-1}, t descending
    const void *lam_in;     // lam_t of the first
    void *lam_out;          // lam_{t-1} of the last
    double *s_bar;          // [N]
    double *a_bar;          // [ny]
    double amp[TILE_MAX_LEVELS];
    double ramp[TILE_MAX_LEVELS];       // da/du_max of the iteration's inlet
    double W[TILE_MAX_LEVELS];          // its drag weight
    int K, lev0;
};

template <typename T> __device__ __forceinline__ T rcp(T v) { return T(1) / v; }
template <> __device__ __forceinline__ float rcp<float>(float v) { return __builtin_amdgcn_rcpf(v); }

// a b + c: one instruction in double; two roundings in float
__device__ __forceinline__ double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float mad(float a, float b, float c) { return a * b + c; }

// A plane element: uniform base, 32-bit byte offset of the node.
template <typename T> __device__ __forceinline__ T plane(const void *b, const PbbParams &p, int q, int cell)
{
    return ld_off<T>(static_cast<const T *>(b) + (size_t)q * p.N, (uint32_t)cell * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void put(void *b, const PbbParams &p, int q, int cell, T v)
{
    st_off(sbase(static_cast<T *>(b) + (size_t)q * p.N), (uint32_t)cell * (uint32_t)sizeof(T), v);
}

// v, not known to be the same in the next iteration: what is formed from it
// stays inside the loop instead of taking registers throughout.
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ double opaque(double v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Boundary step (turek.py:112-125 at rest, pressure outlet) of a perimeter
// node's pulled deviations v, in place.  (ux, uy): inlet velocity of a left
// node; fn: a corner's neighbour, its populations 0, 1, 2 and the three that
// leave through its wall.  Entries of v without a source hold any value: the
// routines set them without reading them.
template <typename T>
__device__ __forceinline__ void pbb_wall(const PbbParams &p, int type, bool left, bool low, T ux,
                                         T uy, const T *fn, T *v)
{
    T f[9], r = T(0), u = T(0);
#pragma unroll
    for (int q = 0; q < 9; ++q) f[q] = weight<T>(q) + v[q];
    if (type == NODE_CORNER) {
        T h[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) h[k] = weight<T>(k < 3 ? k : 2 * k - 3) + fn[k];
        zh_corner_beside(f, left, low, h, T(0), T(0));
    } else if (type == NODE_BOTTOM) {
        zh_bottom(f, T(0), T(0), r);
    } else if (type == NODE_TOP) {
        zh_top(f, T(0), T(0), r);
    } else if (type == NODE_LEFT) {
        zh_left(f, ux, uy, r);
    } else {
        zh_right_pres(f, T(opaque(p.rho_out)), T(0), u);
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) v[q] = f[q] - weight<T>(q);
}

// TRT collision on deviations; also returns rho and u.
template <typename T>
__device__ __forceinline__ void collide_dev(T om_p, T om_m, const T *h, T *c, T &rho, T &ux,
                                            T &uy)
{
    const T drho = ((h[0] + h[1]) + (h[2] + h[3])) + ((h[4] + h[5]) + (h[6] + h[7])) + h[8];
    const T jx = (h[1] - h[2]) + (h[5] - h[6]) + (h[8] - h[7]);
    const T jy = (h[3] - h[4]) + (h[5] - h[6]) + (h[7] - h[8]);
    rho = T(1) + drho;
    const T inv = rcp(rho);
    ux = jx * inv;
    uy = jy * inv;
    const T usq = T(1.5) * mad(ux, ux, uy * uy);
    const T base = mad(-rho, usq, drho);
    c[0] = mad(-om_p, mad(-weight<T>(0), base, h[0]), h[0]);
    const T hp = T(0.5) * om_p, hm = T(0.5) * om_m;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int q = 2 * j + 1, qb = q + 1;
        const T w = weight<T>(q);
        const T cu = j == 0 ? ux : (j == 1 ? uy : (j == 2 ? ux + uy : uy - ux));
        const T ep = w * mad(T(4.5) * rho * cu, cu, base);
        const T em = T(3) * w * rho * cu;
        const T dp = hp * mad(T(-2), ep, h[q] + h[qb]);
        const T dm = hm * mad(T(-2), em, h[q] - h[qb]);
        c[q] = h[q] - dp - dm;
        c[qb] = h[qb] - dp + dm;
    }
}

// v + c a, c = -1, 0 or 1
template <typename T> __device__ __forceinline__ T add_c(T v, int c, T a)
{
    return c > 0 ? v + a : (c < 0 ? v - a : v);
}

// Adjoint of the collision + partial bounce-back + drag at one node:
// lam (adjoint of H at the node) -> hbar (adjoint of the post-boundary h),
// and the node's contribution to dL/ds.  Terms with a zero component of c are
// left out by hand: the compiler has to keep 0 x (x may be infinite).
template <typename T>
__device__ __forceinline__ void node_adjoint(const PbbParams &p, double w, const T *h, T sv,
                                             const T *lam, T *hbar, double &sbar)
{
    const T om_p = T(p.om_p), om_m = T(p.om_m), W = T(w);
    T c[9], rho, ux, uy;
    collide_dev<T>(om_p, om_m, h, c, rho, ux, uy);
    T cb[9];
    double sb = 0.0;
    const T fs = T(1) - sv, ws = W * sv;
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const int qb = NS[q];
        cb[q] = CX[q] ? mad(fs, lam[q], CX[q] > 0 ? ws : -ws) : fs * lam[q];
        hbar[q] = CX[q] ? mad(sv, lam[qb], CX[q] > 0 ? ws : -ws) : sv * lam[qb];
        const T d = h[qb] - c[q];
        sb += (double)(CX[q] ? mad(lam[q], d, CX[q] > 0 ? -(W * d) : W * d) : lam[q] * d);
    }
    sbar = sb;
    // Ebar = Om cbar (TRT relaxation operator, symmetric)
    T eb[9];
    eb[0] = om_p * cb[0];
#pragma unroll
    for (int q = 1; q < 9; q += 2) {
        const T sp = T(0.5) * (cb[q] + cb[q + 1]), sm = T(0.5) * (cb[q] - cb[q + 1]);
        const T em = om_m * sm;
        eb[q] = mad(om_p, sp, em);
        eb[q + 1] = mad(om_p, sp, -em);
    }
    // E_q = w (drho + 3 c.j + (4.5 (c.j)^2 - 1.5 j.j) / rho); cu of q + 1 is
    // that of q with the other sign, 9 cu c the same
    const T u2 = T(1.5) * mad(ux, ux, uy * uy), tx = T(3) * ux, ty = T(3) * uy;
    const T k0 = eb[0] * weight<T>(0);
    T rb = k0 * (T(1) + u2), jbx = k0 * -tx, jby = k0 * -ty;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int q = 2 * j + 1, cx = CX[q], cy = CY[q];
        const T w = weight<T>(q);
        const T cu = j == 0 ? ux : (j == 1 ? uy : (j == 2 ? ux + uy : uy - ux));
        const T nine = T(9) * cu, r = mad(T(-4.5) * cu, cu, T(1)) + u2;
        const T k = eb[q] * w, kb = eb[q + 1] * w;
        rb = mad(kb, r, mad(k, r, rb));
        const T gx = cx ? T(cx) * nine : T(0), gy = cy ? T(cy) * nine : T(0);
        jbx = mad(kb, (T(-3 * cx) + gx) - tx, mad(k, (T(3 * cx) + gx) - tx, jbx));
        jby = mad(kb, (T(-3 * cy) + gy) - ty, mad(k, (T(3 * cy) + gy) - ty, jby));
    }
#pragma unroll
    for (int q = 0; q < 9; ++q)
        hbar[q] += add_c(add_c(cb[q] - eb[q] + rb, CX[q], jbx), CY[q], jby);
}

// Sum over a wave, in work-item 63: rows of 16 by shifts, then across rows.
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_add(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double wave_sum(double v)
{
    v = dpp_add<0x111, 0xf>(v);     // row_shr 1, 2, 4, 8
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);     // lane 15 of rows 0, 2 -> rows 1, 3
    return dpp_add<0x143, 0xc>(v);  // lane 31 -> rows 2, 3
}

// This work-item's node m of region r (slots of tile_perim: perimeter nodes
// first, a wave of one kind each, then the inner ones); false on padding.
__device__ __forceinline__ bool tile_node(const TileRect &r, const TilePerim &P, uint32_t inv, int n,
                                          int &x, int &y, int &type)
{
    type = NODE_INNER;
    if (n < P.slots) return tile_perim_node(r, P, n, x, y, type);
    n -= P.slots;
    const int hi = r.h - P.tb - P.tt;
    const int xx = hi == 1 ? n : (int)__umulhi((uint32_t)n, inv);
    x = r.x + P.tl + xx;
    y = r.y + P.tb + n - xx * hi;
    return n < P.inner;
}

// K less the node's distance from the owned rectangle, or by the rectangles.
__device__ __forceinline__ int last_level(const TileDesc &D, int K, int lev0, int x, int y)
{
    if (D.regular) {
        const TileRect r = D.r[K];
        return K - max(max(max(r.x - x, x - r.x - r.w + 1), max(r.y - y, y - r.y - r.h + 1)), 0);
    }
    int lm = lev0;
#pragma unroll
    for (int l = 1; l <= TILE_MAX_LEVELS; ++l) {
        const TileRect r = D.r[l];
        const bool in = (unsigned)(x - r.x) < (unsigned)r.w && (unsigned)(y - r.y) < (unsigned)r.h;
        if (l > lev0 && l <= K && in) lm = l;
    }
    return lm;
}

// The nine pulls of LDS node c (columns h0 nodes apart).
template <int CAP, typename T> __device__ __forceinline__ void lds_pull(const T *lds, int c, int h0, T *f)
{
    const int e = c - h0, w = c + h0;
    f[0] = lds[0 * CAP + c];
    f[1] = lds[1 * CAP + e];
    f[2] = lds[2 * CAP + w];
    f[3] = lds[3 * CAP + c - 1];
    f[4] = lds[4 * CAP + c + 1];
    f[5] = lds[5 * CAP + e - 1];
    f[6] = lds[6 * CAP + w + 1];
    f[7] = lds[7 * CAP + w - 1];
    f[8] = lds[8 * CAP + e + 1];
}

// ------------------------------------------------------------- forward --
// Several iterations per launch in LDS, as d2q9_tile.hip (the same planes,
// nodes and barriers).  The recomputation before an adjoint segment stores the
// owned nodes of every iteration, the forward run only the last.  Drag: the
// owned nodes' terms in double, summed per wave and tile (fixed order).
template <typename T, int NT, int M>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_pbb_fwd(
    PbbFwd a, const TileDesc *__restrict__ tiles)
{
    constexpr int CAP = NT * M, WAVES = NT / 64;
    extern __shared__ __align__(16) char smem[];
    T *const lds = reinterpret_cast<T *>(smem);
    double *const s_drag = reinterpret_cast<double *>(lds + 9 * CAP);     // [level][wave]
    const PbbParams &p = a.p;
    const int tile = xcd_tile(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const TileDesc &D = tiles[tile];
    const int K = a.K, lev0 = a.lev0, nx = p.nx, ny = p.ny;
    const TileRect r0 = D.r[lev0], r1 = D.r[lev0 + 1];
    const int a0 = r0.w * r0.h, h0 = r0.h;
    T v[M][9];
    const uint32_t inv0 = D.mh[lev0];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int n = tid + m * NT;
        const int x = (int)__umulhi((uint32_t)n, inv0), cell = (r0.x + x) * ny + r0.y + n - x * h0;
        if (n < a0) {
#pragma unroll
            for (int q = 0; q < 9; ++q) v[m][q] = plane<T>(a.src, p, q, cell);
        }
    }
    const TilePerim P = tile_perim(r1, nx, ny);
    const uint32_t inv = D.mi[lev0 + 1];
    int li[M], cell[M], lm[M], type = NODE_INNER;
    bool left = false, low = false;
    T sv[M];
    double px = 0.0, py = 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        li[m] = cell[m] = lm[m] = 0;
        sv[m] = T(0);
        int x = 0, y = 0, t;
        if (!tile_node(r1, P, inv, tid + m * NT, x, y, t)) continue;
        if (m == 0) {
            type = t;
            left = x == 0;
            low = y == 0;
            if (t == NODE_LEFT) {
                px = p.prof[y];
                py = p.prof[ny + y];
            }
        }
        li[m] = (x - r0.x) * h0 + (y - r0.y);
        cell[m] = x * ny + y;
        lm[m] = last_level(D, K, lev0, x, y);
        sv[m] = static_cast<const T *>(p.s)[cell[m]];
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int n = tid + m * NT;
        if (n < a0) {
#pragma unroll
            for (int q = 0; q < 9; ++q) lds[q * CAP + n] = v[m][q];
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int l = lev0 + 1; l <= K; ++l) {
        const bool last = l == K;
        const int j = l - lev0 - 1;
        T f[M][9], fn[6];
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (l <= lm[m]) lds_pull<CAP>(lds, opaque(li[m]), h0, f[m]);
        if (type == NODE_CORNER && l <= lm[0]) {
            const int c = opaque(left ? li[0] + h0 : li[0] - h0), e = c - h0, w = c + h0;
            fn[0] = lds[c];
            fn[1] = lds[1 * CAP + e];
            fn[2] = lds[2 * CAP + w];
            fn[3] = lds[low ? 4 * CAP + c + 1 : 3 * CAP + c - 1];
            fn[4] = lds[low ? 6 * CAP + w + 1 : 5 * CAP + e - 1];
            fn[5] = lds[low ? 8 * CAP + e + 1 : 7 * CAP + w - 1];
        }
        __syncthreads();
        double drag = 0.0;
        char *const dst = a.dst + (size_t)j * a.stride;
        const bool out = last || a.stride;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (l > lm[m]) continue;
            if (m == 0 && type != NODE_INNER)
                pbb_wall<T>(p, type, left, low, T(a.amp[j] * px), T(a.amp[j] * py), fn, f[0]);
            T c[9], rho, ux, uy;
            collide_dev<T>(T(p.om_p), T(p.om_m), f[m], c, rho, ux, uy);
            double dd = 0.0;
#pragma unroll
            for (int q = 0; q < 9; ++q)
                if (CX[q]) dd += (double)(T(CX[q]) * (c[q] - f[m][NS[q]]));
#pragma unroll
            for (int q = 0; q < 9; ++q) c[q] = mad(T(1) - sv[m], c[q], sv[m] * f[m][NS[q]]);
            if (lm[m] == K) {
                drag += (double)sv[m] * dd;
                if (out) {
#pragma unroll
                    for (int q = 0; q < 9; ++q) put<T>(dst, p, q, cell[m], c[q]);
                }
            }
            if (!last) {
                const int n = opaque(li[m]);
#pragma unroll
                for (int q = 0; q < 9; ++q) lds[q * CAP + n] = c[q];
            }
        }
        if (a.drag_part) {
            // most waves see no solid: nothing to add (a NaN is not zero)
            const double t = __any(drag != 0.0) ? wave_sum(drag) : 0.0;
            if ((tid & 63) == 63) s_drag[j * WAVES + (tid >> 6)] = t;
        }
        __syncthreads();
    }
    if (a.drag_part && tid < K - lev0) {
        double t = 0.0;
        for (int w = 0; w < WAVES; ++w) t += s_drag[tid * WAVES + w];
        a.drag_part[(size_t)tid * gridDim.x + tile] = t;
    }
}

// Iteration 0, from rest: h = 0, so H_0 = (1 - s) 0 + s 0 and its drag terms
// s 0, formed as written for the sake of a non-finite s.
template <typename T>
__global__ __launch_bounds__(256) void k_pbb_start(PbbParams p, T *dst, double *drag_part)
{
    __shared__ double red[4];
    double d = 0.0;
    for (int cell = blockIdx.x * 256 + threadIdx.x; cell < p.N; cell += gridDim.x * 256) {
        const T sv = static_cast<const T *>(p.s)[cell];
        const T h = (T(1) - sv) * T(0) + sv * T(0);
#pragma unroll
        for (int q = 0; q < 9; ++q) dst[(size_t)q * p.N + cell] = h;
        d += (double)sv * 0.0;
    }
    d = wave_sum(d);
    if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = d;
    __syncthreads();
    if (threadIdx.x == 0) drag_part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// ------------------------------------------------------------- adjoint --
// Transpose of the (affine) boundary step of a perimeter node: h, the adjoint
// of its post-boundary populations, -> the adjoint of its pulled ones, in
// place.  Populations the step sets have none.  Each pulled population's
// entry is sum_q h_q d(out_q)/d(in), in the order of q, with the derivatives
// the step's own expressions give for a unit population (T arithmetic).
//   bottom/top (at rest): f_in = f_out, diagonals -+ K3 (f_1 - f_2)
//   left:  rho = S / (1 - ux), S = f0 + f3 + f4 + 2 (f2 + f6 + f7)
//   right: ux = M / rho - 1,   M = f0 + f3 + f4 + 2 (f1 + f5 + f8)
//   corner (at rest): f_in = f_out, f0 = rho - sum, rho the neighbour's
template <typename T>
__device__ __forceinline__ void wall_adjoint(int type, bool left, bool low, T ux, T uy, T rho, T *h)
{
    const T k1 = T(K1), k2 = T(K2), k3 = T(K3), z = T(0);
    if (type == NODE_BOTTOM) {
        h[1] = (h[1] + h[5] * -k3) + h[7] * k3;
        h[2] = (h[2] + h[5] * k3) + h[7] * -k3;
        h[4] = h[3] + h[4];
        h[6] = h[5] + h[6];
        h[8] = h[7] + h[8];
        h[3] = h[5] = h[7] = z;
    } else if (type == NODE_TOP) {
        h[1] = (h[1] + h[6] * k3) + h[8] * -k3;
        h[2] = (h[2] + h[6] * -k3) + h[8] * k3;
        h[3] = h[3] + h[4];
        h[5] = h[5] + h[6];
        h[7] = h[7] + h[8];
        h[4] = h[6] = h[8] = z;
    } else if (type == NODE_LEFT) {
        const T r1 = T(1) / (T(1) - ux), r2 = T(2) * r1;     // rho of S = 1, 2
        const T n1 = k1 * r1 * ux, n2 = k1 * r2 * ux;
        const T x1 = k2 * r1 * ux, x2 = k2 * r2 * ux, y1 = k3 * r1 * uy, y2 = k3 * r2 * uy;
        h[0] = ((h[0] + h[1] * n1) + h[5] * (x1 + y1)) + h[8] * (x1 - y1);
        h[3] = ((h[1] * n1 + h[3]) + h[5] * (-k3 + x1 + y1)) + h[8] * (k3 + x1 - y1);
        h[4] = ((h[1] * n1 + h[4]) + h[5] * (k3 + x1 + y1)) + h[8] * (-k3 + x1 - y1);
        h[2] = ((h[1] * (T(1) + n2) + h[2]) + h[5] * (x2 + y2)) + h[8] * (x2 - y2);
        h[6] = ((h[1] * n2 + h[5] * (T(1) + x2 + y2)) + h[6]) + h[8] * (x2 - y2);
        h[7] = ((h[1] * n2 + h[5] * (x2 + y2)) + h[7]) + h[8] * (T(1) + x2 - y2);
        h[1] = h[5] = h[8] = z;
    } else if (type == NODE_RIGHT) {
        const T a = k1 * rho, b = k2 * rho;                  // f2 = f1 - a ux, ... ux = M / rho - 1
        const T u1 = T(1) / rho - T(1), u2 = T(2) / rho - T(1);
        const T a0 = z - a * T(-1), b0 = z - b * T(-1);      // M = 0
        const T a1 = z - a * u1, b1 = z - b * u1, a2 = z - a * u2, b2 = z - b * u2;
        const T h2 = h[2], h6 = h[6], h7 = h[7];
        h[0] = ((h[0] + h2 * (a1 - a0)) + h6 * (b1 - b0)) + h7 * (b1 - b0);
        h[3] = ((h2 * (a1 - a0) + h[3]) + h6 * ((k3 - b * u1) - b0)) + h7 * ((-k3 - b * u1) - b0);
        h[4] = ((h2 * (a1 - a0) + h[4]) + h6 * ((-k3 - b * u1) - b0)) + h7 * ((k3 - b * u1) - b0);
        h[1] = ((h[1] + h2 * ((T(1) - a * u2) - a0)) + h6 * (b2 - b0)) + h7 * (b2 - b0);
        h[5] = ((h2 * (a2 - a0) + h[5]) + h6 * ((T(1) - b * u2) - b0)) + h7 * (b2 - b0);
        h[8] = ((h2 * (a2 - a0) + h6 * (b2 - b0)) + h7 * ((T(1) - b * u2) - b0)) + h[8];
        h[2] = h[6] = h[7] = z;
    } else {
        const T g = h[0] * T(-2);
        const T sx = (g + h[1]) + h[2], sy = (g + h[3]) + h[4];
        const bool main = left == low;          // bottom left and top right: diagonal 5, 6
        const T d0 = main ? +h[5] : +h[7], d1 = main ? +h[6] : +h[8];
        const T sd = (g + d0) + d1;
        h[0] = z;
        h[1] = left ? z : +sx;
        h[2] = left ? +sx : z;
        h[3] = low ? z : +sy;
        h[4] = low ? +sy : z;
        h[5] = main && !left ? +sd : z;
        h[6] = main && left ? +sd : z;
        h[7] = !main && left ? +sd : z;
        h[8] = !main && !left ? +sd : z;
    }
}

// d(boundary output)/d(ux, uy) . hbar on a left-wall node (zh_left with
// rho = S / (1 - ux), S of its pulled populations).
template <typename T>
__device__ __forceinline__ void left_velocity_adjoint(T S, T ux, T uy, const T *hbar, T &gx, T &gy)
{
    const T r = S / (T(1) - ux);
    const T dr = r / (T(1) - ux);          // d(rho ux)/dux = rho / (1 - ux)
    const T d1x = T(K1) * dr;
    const T d5x = T(K2) * dr + T(K3) * uy * (r / (T(1) - ux));
    const T d8x = T(K2) * dr - T(K3) * uy * (r / (T(1) - ux));
    gx = hbar[1] * d1x + hbar[5] * d5x + hbar[8] * d8x;
    gy = hbar[5] * (T(K3) * r) - hbar[8] * (T(K3) * r);
}

// Several adjoint iterations per launch.  lam lives in LDS: an iteration reads
// each node's nine adjoints, forms the adjoint of its pulled populations
// (node_adjoint, then the wall's transpose on the perimeter) and writes them
// to the nodes they were pulled from, x - c_q; level l computes r[l - 1] and
// writes into r[l].  Between the two stands a barrier, so the M nodes' results
// wait in registers; the states are fetched one node ahead, not M, which is
// what keeps a double node's ~100 live values within two waves per SIMD (with
// all M prefetched and the loop's invariants hoisted, 800 bytes of scratch a
// work-item: 90 us a launch of 3).  s_bar and a_bar are carried in registers,
// in the order of the iterations, so grouping does not change them.
//
// Bound by issue: ~300 FP64 (350 FP32) and ~90 other vector instructions a
// node, VALU busy 52 % in double, waits for the stack's reads 39 %.  1024x256:
// FP64 20.5 us per adjoint iteration (one per launch, its perimeter's maps
// evaluated column by column) -> 9.3; loss and gradient of 400 iterations
// FP64 17.5 -> 7.1 ms, FP32 14.5 -> 5.1 ms.
template <typename T, int NT, int M>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT / 256))) void k_pbb_adj(PbbAdj a, const TileDesc *__restrict__ tiles)
{
    constexpr int CAP = NT * M;
    extern __shared__ __align__(16) char smem[];
    T *const lds = reinterpret_cast<T *>(smem);
    T *const s_corner = lds + 9 * CAP;          // hb[0] of the corners BL, TL, BR, TR; one unread
    const PbbParams &p = a.p;
    const int tid = threadIdx.x;
    const TileDesc &D = tiles[xcd_tile(blockIdx.x, gridDim.x)];
    const int K = a.K, lev0 = a.lev0, nx = p.nx, ny = p.ny, lx = nx - 1, ly = ny - 1;
    const TileRect r0 = D.r[lev0];
    const int h0 = r0.h;
    const TilePerim P = tile_perim(r0, nx, ny);
    const uint32_t inv = D.mi[lev0];
    int li[M], lm[M], xs[M], ys[M], type = NODE_INNER;
    T sv[M], h[9], hb[M][9], fn[6];
    double sacc[M], px = 0.0, py = 0.0, aacc = 0.0;
    // pulls of node (x, y) from state b; sources beyond the lattice read some
    // other element of the state (index within [0, 9 N))
    auto pull = [&](const void *b, int x, int y, T *f) {
        const int cell = x * ny + y;
#pragma unroll
        for (int q = 0; q < 9; ++q) f[q] = plane<T>(static_cast<const T *>(b) - (CX[q] * ny + CY[q]), p, q, cell);
    };
    auto pull_corner = [&](const void *b, int x, int y) {
        const int cell = (x == 0 ? 1 : lx - 1) * ny + y;
        const bool low = y == 0;
        fn[0] = plane<T>(b, p, 0, cell);
        fn[1] = plane<T>(b, p, 1, cell - ny);
        fn[2] = plane<T>(b, p, 2, cell + ny);
        fn[3] = low ? plane<T>(b, p, 4, cell + 1) : plane<T>(b, p, 3, cell - 1);
        fn[4] = low ? plane<T>(b, p, 6, cell + ny + 1) : plane<T>(b, p, 5, cell - ny - 1);
        fn[5] = low ? plane<T>(b, p, 8, cell - ny + 1) : plane<T>(b, p, 7, cell + ny - 1);
    };
#pragma unroll
    for (int m = 0; m < M; ++m) {
        li[m] = xs[m] = ys[m] = 0;
        lm[m] = -1;
        sv[m] = T(0);
        sacc[m] = 0.0;
        int x = 0, y = 0, t;
        if (!tile_node(r0, P, inv, tid + m * NT, x, y, t)) continue;
        xs[m] = x;
        ys[m] = y;
        li[m] = (x - r0.x) * h0 + (y - r0.y);
        lm[m] = last_level(D, K, lev0, x, y);
        if (m == 0) pull(a.h[0], x, y, h);
        sv[m] = static_cast<const T *>(p.s)[x * ny + y];
        if (lm[m] == K) sacc[m] = a.s_bar[x * ny + y];
        if (m == 0) {
            type = t;
            if (t == NODE_CORNER) pull_corner(a.h[0], x, y);
            if (t == NODE_LEFT) {
                px = p.prof[y];
                py = p.prof[ny + y];
                if (lm[0] == K) aacc = a.a_bar[y];
            }
        }
    }
#pragma unroll 1
    for (int l = lev0 + 1; l <= K; ++l) {
        const bool last = l == K;
        const int j = l - lev0 - 1;
        const T ux = T(a.amp[j] * px), uy = T(a.amp[j] * py);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            T hn[9];                            // the node after this one
            if (m + 1 < M) {
                if (l - 1 <= lm[m + 1]) pull(a.h[j], opaque(xs[m + 1]), opaque(ys[m + 1]), hn);
            } else if (!last && l <= lm[0]) {
                pull(a.h[j + 1], opaque(xs[0]), opaque(ys[0]), hn);
            }
            if (l - 1 <= lm[m]) {
                const int x = opaque(xs[m]), y = opaque(ys[m]), cell = x * ny + y, c = opaque(li[m]);
                const bool edge = m == 0 && type != NODE_INNER, left = x == 0, low = y == 0;
                T lam[9], S = T(0);
                if (j == 0) {
#pragma unroll
                    for (int q = 0; q < 9; ++q) lam[q] = plane<T>(a.lam_in, p, q, cell);
                } else {
#pragma unroll
                    for (int q = 0; q < 9; ++q) lam[q] = lds[q * CAP + c];
                }
                if (edge) {
                    if (type == NODE_LEFT)
                        S = (weight<T>(0) + h[0]) + (weight<T>(3) + h[3]) + (weight<T>(4) + h[4]) +
                            T(2) * (weight<T>(2) + h[2]) + T(2) * (weight<T>(6) + h[6]) +
                            T(2) * (weight<T>(7) + h[7]);
                    pbb_wall<T>(p, type, left, low, ux, uy, fn, h);
                    if (!last && type == NODE_CORNER) pull_corner(a.h[j + 1], x, y);
                }
                double sb;
                node_adjoint<T>(p, a.W[j], h, sv[m], lam, hb[m], sb);
                if (lm[m] == K) sacc[m] += sb;
                if (edge) {
                    if (type == NODE_CORNER) s_corner[2 * !left + !low] = hb[0][0];
                    if (type == NODE_LEFT && lm[0] == K) {
                        T gx, gy;
                        left_velocity_adjoint<T>(S, ux, uy, hb[0], gx, gy);
                        aacc += a.ramp[j] * ((double)gx * px + (double)gy * py);
                    }
                    wall_adjoint<T>(type, left, low, ux, uy, T(opaque(p.rho_out)), hb[0]);
                }
            }
#pragma unroll
            for (int q = 0; q < 9; ++q) h[q] = hn[q];
        }
        __syncthreads();
        const TileRect R = D.r[l];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (l - 1 > lm[m]) continue;
            const int x = opaque(xs[m]), y = opaque(ys[m]), cell = x * ny + y, c0 = opaque(li[m]);
            if (m == 0 && (type == NODE_BOTTOM || type == NODE_TOP) && (x == 1 || x == lx - 1)) {
                // the corner beside takes this node's density
                const bool low = type == NODE_BOTTOM;
                const T g = s_corner[2 * (x != 1) + !low], up = low ? T(2) * g : T(0),
                        dn = low ? T(0) : T(2) * g;
                hb[0][0] += g;
                hb[0][1] += g;
                hb[0][2] += g;
                hb[0][4] += up;
                hb[0][6] += up;
                hb[0][8] += up;
                hb[0][3] += dn;
                hb[0][5] += dn;
                hb[0][7] += dn;
            }
            // targets x - c inside R, by component of c
            bool okx[3], oky[3];
#pragma unroll
            for (int c = -1; c <= 1; ++c) {
                okx[c + 1] = (unsigned)(x - c - R.x) < (unsigned)R.w;
                oky[c + 1] = (unsigned)(y - c - R.y) < (unsigned)R.h;
            }
            if (last) {
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    if (okx[CX[q] + 1] && oky[CY[q] + 1])
                        put<T>(a.lam_out, p, q, cell - (CX[q] * ny + CY[q]), hb[m][q]);
            } else {
#pragma unroll
                for (int q = 0; q < 9; ++q) {
                    const int n = q * CAP + c0 - (CX[q] * h0 + CY[q]);
                    lds[okx[CX[q] + 1] && oky[CY[q] + 1] ? n : 9 * CAP + 4] = hb[m][q];
                }
            }
            if (m == 0 && type != NODE_INNER && okx[1] && oky[1]) {
                // an entry of this node that no node pulls carries no adjoint
#pragma unroll
                for (int q = 1; q < 9; ++q) {
                    const int tx = x + CX[q], ty = y + CY[q];
                    if (tx >= 0 && tx <= lx && ty >= 0 && ty <= ly) continue;
                    if (last) put<T>(a.lam_out, p, q, cell, T(0));
                    else lds[q * CAP + c0] = T(0);
                }
            }
        }
        if (!last) __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < M; ++m)
        if (lm[m] == K) a.s_bar[xs[m] * ny + ys[m]] = sacc[m];
    if (type == NODE_LEFT && lm[0] == K) a.a_bar[ys[0]] = aacc;
}

// Sum of a row of nb tile sums, in order: a wave per row stages them in LDS,
// work-item 0 adds (401 rows of 256: 6 us; a work-item per row reading 1024
// terms one by one took 99).
constexpr int SUM_CHUNK = 1024;
__global__ __launch_bounds__(64) void k_pbb_sum_rows(const double *__restrict__ part, int nb,
                                                     double *__restrict__ out)
{
    __shared__ double sh[SUM_CHUNK];
    const double *r = part + (size_t)blockIdx.x * nb;
    double acc = 0.0;
    for (int k0 = 0; k0 < nb; k0 += SUM_CHUNK) {
        const int n = min(SUM_CHUNK, nb - k0);
        for (int k = threadIdx.x; k < n; k += 64) sh[k] = r[k0 + k];
        __syncthreads();
        if (threadIdx.x == 0) acc = ordered_sum(sh, n, acc);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = acc;
}

__global__ void k_zero_f64(double *p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

template <typename T> __global__ void k_zero_t(T *p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = T(0);
}

inline hipStream_t SS(void *s) { return reinterpret_cast<hipStream_t>(s); }

}  // namespace
}  // namespace lbm

using namespace lbm;

// A plan on the device.
struct PbbTiles {
    int n = 0, K = 0, cfg = 0;
    TileDesc *d = nullptr;
};

struct lbm_pbb {
    int nx = 0, ny = 0, N = 0, storage = 0, T = 0, window = 0, every = 0;
    double om_p = 0, om_m = 0, rho_out = 1;
    double *d_prof = nullptr;
    std::vector<double> ramp;          // ramp(it), it = 0..T
    double u_max = 0;
    size_t sb = 0;                     // bytes of one state
    std::vector<void *> ckpt;          // H at it = 0, every, 2 every, ...
    void *ping[2] = {nullptr, nullptr};
    void *stack = nullptr;             // one segment of states
    void *lam[2] = {nullptr, nullptr};
    PbbTiles fwd, adj;                 // plans of the forward and adjoint launches
    const void *last = nullptr;        // H_T of the last forward run
    double *d_part = nullptr;          // [T+1][fwd.n]
    double *d_drag = nullptr;          // [T+1]
    double *d_abar = nullptr;          // [ny]
    const void *s = nullptr;           // solid fraction of the last forward
    std::vector<double> drag;          // host copy
};

namespace {

int pbb_plan(lbm_pbb *h, bool adjoint, PbbTiles &t)
{
    int dev = 0, cus = 0, lds = 0;
    LBM_HIP_TRY(hipGetDevice(&dev));
    LBM_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    LBM_HIP_TRY(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const bool f64 = h->storage == LBM_STORE_F64;
    int n = 0;
    const TileKind *kinds = adjoint ? adjoint_kinds(f64, n) : tile_kinds(f64, n);
    const std::vector<PlanLink> none;
    TilePlan plan;
    // 1 KiB: the kernels' own LDS arrays
    const TileKind *k = plan_cases({{h->nx, h->ny, &none}}, kinds, n, adjoint, f64, cus,
                                   (size_t)lds - 1024, plan);
    if (!k) return set_error(LBM_ERR_UNSUPPORTED, "lbm_pbb: no tile plan for this lattice");
    const size_t bytes = sizeof(TileDesc) * plan.tiles.size();
    if (hipMalloc((void **)&t.d, bytes) != hipSuccess ||
        hipMemcpy(t.d, plan.tiles.data(), bytes, hipMemcpyHostToDevice) != hipSuccess)
        return set_error(LBM_ERR_HIP, "lbm_pbb: tile plan upload");
    t.n = (int)plan.tiles.size();
    t.K = k->K;
    t.cfg = k->cfg;
    return LBM_OK;
}

PbbParams pbb_params(const lbm_pbb *h)
{
    PbbParams p{};
    p.nx = h->nx;
    p.ny = h->ny;
    p.N = h->N;
    p.om_p = h->om_p;
    p.om_m = h->om_m;
    p.rho_out = h->rho_out;
    p.prof = h->d_prof;
    p.s = h->s;
    return p;
}

void pbb_free(lbm_pbb *h)
{
    for (void *c : h->ckpt) (void)hipFree(c);
    void *ptrs[] = {h->d_prof, h->ping[0], h->ping[1], h->stack, h->lam[0], h->lam[1],
                    h->d_part, h->d_drag, h->d_abar, h->fwd.d, h->adj.d};
    for (void *q : ptrs)
        if (q) (void)hipFree(q);
}

template <typename T, int NT, int M>
void launch_fwd(const lbm_pbb *h, const PbbFwd &a, hipStream_t s)
{
    const size_t lds = sizeof(T) * 9 * NT * M + sizeof(double) * TILE_MAX_LEVELS * (NT / 64);
    k_pbb_fwd<T, NT, M><<<h->fwd.n, NT, lds, s>>>(a, h->fwd.d);
}

// the shapes of tile_kinds
template <typename T> void launch_fwd_t(const lbm_pbb *h, const PbbFwd &a, hipStream_t s)
{
    switch (h->fwd.cfg) {
    case 0: launch_fwd<T, 512, 1>(h, a, s); break;
    case 1: launch_fwd<T, 512, 2>(h, a, s); break;
    case 2: launch_fwd<T, 1024, 2>(h, a, s); break;
    case 3: if constexpr (sizeof(T) == 4) launch_fwd<T, 512, 4>(h, a, s); break;
    default: if constexpr (sizeof(T) == 4) launch_fwd<T, 1024, 4>(h, a, s); break;
    }
}

// Iterations t .. t + n - 1 (n <= fwd.K) from state src.
void fwd(const lbm_pbb *h, PbbFwd a, int t, int n, hipStream_t s)
{
    for (int j = 0; j < n; ++j) a.amp[j] = h->ramp[t + j - 1] * h->u_max;
    a.K = h->fwd.K;
    a.lev0 = h->fwd.K - n;
    if (h->storage == LBM_STORE_F64) launch_fwd_t<double>(h, a, s);
    else launch_fwd_t<float>(h, a, s);
}

template <typename T, int NT, int M> void launch_adj(const lbm_pbb *h, const PbbAdj &a, hipStream_t s)
{
    k_pbb_adj<T, NT, M><<<h->adj.n, NT, sizeof(T) * (9 * NT * M + 5), s>>>(a, h->adj.d);
}

template <typename T> void launch_adj_t(const lbm_pbb *h, const PbbAdj &a, hipStream_t s)
{
    constexpr bool f64 = sizeof(T) == 8;
    switch (h->adj.cfg) {
    case 0: launch_adj<T, f64 ? 512 : 1024, 1>(h, a, s); break;
    case 1: launch_adj<T, f64 ? 512 : 1024, 2>(h, a, s); break;
    default: launch_adj<T, 512, f64 ? 4 : 3>(h, a, s); break;
    }
}

// Adjoint iterations t, t - 1, .. t - n + 1 (n <= adj.K); state(t) = H_t.
template <class F>
void adj(const lbm_pbb *h, PbbAdj a, int t, int n, F state, hipStream_t s)
{
    for (int j = 0; j < n; ++j) {
        const int it = t - j;
        a.h[j] = state(it - 1);
        a.ramp[j] = h->ramp[it - 1];
        a.amp[j] = h->ramp[it - 1] * h->u_max;
        a.W[j] = it > h->T - h->window ? 1.0 / h->window : 0.0;
    }
    a.K = h->adj.K;
    a.lev0 = h->adj.K - n;
    if (h->storage == LBM_STORE_F64) launch_adj_t<double>(h, a, s);
    else launch_adj_t<float>(h, a, s);
}

}  // namespace

extern "C" int lbm_pbb_create(const lbm_pbb_desc *d, lbm_pbb **out)
{
    if (!d || !out || d->nx < 4 || d->ny < 4 || d->iterations < 1 || d->window < 1 ||
        d->window > d->iterations || d->checkpoint_every < 1 || !d->inlet_profile_host ||
        !d->ramp_host || (d->storage != LBM_STORE_F64 && d->storage != LBM_STORE_F32))
        return set_error(LBM_ERR_ARG, "lbm_pbb_create: bad argument");
    if ((long long)d->nx * d->ny * 9 >= (1LL << 31))
        return set_error(LBM_ERR_ARG, "lattice too large");
    auto h = std::make_unique<lbm_pbb>();
    h->nx = d->nx;
    h->ny = d->ny;
    h->N = d->nx * d->ny;
    h->storage = d->storage;
    h->T = d->iterations;
    h->window = d->window;
    h->every = d->checkpoint_every;
    h->om_p = d->om_p;
    h->om_m = d->om_m;
    h->rho_out = d->rho_out;
    h->ramp.assign(d->ramp_host, d->ramp_host + d->iterations + 1);
    h->sb = (size_t)9 * h->N * (d->storage == LBM_STORE_F64 ? 8 : 4);
    auto alloc = [&](void **p, size_t bytes) {
        return hipMalloc(p, bytes) == hipSuccess;
    };
    int e;
    if ((e = pbb_plan(h.get(), false, h->fwd)) || (e = pbb_plan(h.get(), true, h->adj))) {
        pbb_free(h.get());
        return e;
    }
    const int nck = h->T / h->every + 1;
    h->ckpt.assign(nck, nullptr);
    bool ok = alloc((void **)&h->d_prof, sizeof(double) * 2 * h->ny) &&
              alloc(&h->ping[0], h->sb) && alloc(&h->ping[1], h->sb) &&
              alloc(&h->stack, h->sb * (size_t)h->every) && alloc(&h->lam[0], h->sb) &&
              alloc(&h->lam[1], h->sb) &&
              alloc((void **)&h->d_part, sizeof(double) * (size_t)(h->T + 1) * h->fwd.n) &&
              alloc((void **)&h->d_drag, sizeof(double) * (h->T + 1)) &&
              alloc((void **)&h->d_abar, sizeof(double) * h->ny);
    for (int i = 0; ok && i < nck; ++i) ok = alloc(&h->ckpt[i], h->sb);
    if (!ok) {
        pbb_free(h.get());
        return set_error(LBM_ERR_HIP, "lbm_pbb_create: allocation failed");
    }
    if (hipMemcpy(h->d_prof, d->inlet_profile_host, sizeof(double) * 2 * h->ny,
                  hipMemcpyHostToDevice) != hipSuccess) {
        pbb_free(h.get());
        return set_error(LBM_ERR_HIP, "lbm_pbb_create: profile upload");
    }
    *out = h.release();
    return LBM_OK;
}

extern "C" void lbm_pbb_destroy(lbm_pbb *h)
{
    if (!h) return;
    (void)hipDeviceSynchronize();
    pbb_free(h);
    delete h;
}

extern "C" int lbm_pbb_forward(lbm_pbb *h, const void *s_dev, double u_max, double *loss,
                               void *stream)
{
    if (!h || !s_dev || !loss) return set_error(LBM_ERR_ARG, "lbm_pbb_forward: bad argument");
    hipStream_t st = SS(stream);
    h->s = s_dev;
    h->u_max = u_max;
    PbbFwd a{};
    a.p = pbb_params(h);
    // iteration 0: from rest
    if (h->storage == LBM_STORE_F64)
        k_pbb_start<double><<<h->fwd.n, 256, 0, st>>>(a.p, static_cast<double *>(h->ckpt[0]), h->d_part);
    else
        k_pbb_start<float><<<h->fwd.n, 256, 0, st>>>(a.p, static_cast<float *>(h->ckpt[0]), h->d_part);
    LBM_LAUNCH_CHECK();
    // launches of up to fwd.K iterations, ending at every checkpoint
    a.src = h->ckpt[0];
    for (int t = 1, k = 0, n; t <= h->T; t += n, k ^= 1) {
        const int stop = std::min(h->T, ((t - 1) / h->every + 1) * h->every);
        n = std::min(h->fwd.K, stop - t + 1);
        const int end = t + n - 1;
        a.dst = static_cast<char *>(end % h->every == 0 ? h->ckpt[end / h->every] : h->ping[k]);
        a.drag_part = h->d_part + (size_t)t * h->fwd.n;
        fwd(h, a, t, n, st);
        a.src = h->last = a.dst;
    }
    LBM_LAUNCH_CHECK();
    k_pbb_sum_rows<<<h->T + 1, 64, 0, st>>>(h->d_part, h->fwd.n, h->d_drag);
    LBM_LAUNCH_CHECK();
    h->drag.assign(h->T + 1, 0.0);
    LBM_HIP_TRY(hipMemcpyAsync(h->drag.data(), h->d_drag, sizeof(double) * (h->T + 1),
                               hipMemcpyDeviceToHost, st));
    LBM_HIP_TRY(hipStreamSynchronize(st));
    double acc = 0.0;
    for (int t = h->T - h->window + 1; t <= h->T; ++t) acc += h->drag[t];
    *loss = acc / h->window;
    return LBM_OK;
}

extern "C" int lbm_pbb_backward(lbm_pbb *h, double *s_grad_dev, double *umax_grad, void *stream)
{
    if (!h || !s_grad_dev || !umax_grad || !h->s)
        return set_error(LBM_ERR_ARG, "lbm_pbb_backward: call lbm_pbb_forward first");
    hipStream_t st = SS(stream);
    const size_t nstate = (size_t)9 * h->N;
    const int zb = (int)((nstate + 255) / 256);
    if (h->storage == LBM_STORE_F64)
        k_zero_t<double><<<zb, 256, 0, st>>>(static_cast<double *>(h->lam[0]), nstate);
    else
        k_zero_t<float><<<zb, 256, 0, st>>>(static_cast<float *>(h->lam[0]), nstate);
    k_zero_f64<<<(h->N + 255) / 256, 256, 0, st>>>(s_grad_dev, h->N);
    k_zero_f64<<<(h->ny + 255) / 256, 256, 0, st>>>(h->d_abar, h->ny);
    LBM_LAUNCH_CHECK();
    PbbFwd f{};
    f.p = pbb_params(h);
    f.stride = h->sb;
    PbbAdj a{};
    a.p = f.p;
    a.s_bar = s_grad_dev;
    a.a_bar = h->d_abar;
    int cur = 0;                       // lam[cur]: the adjoint of the latest state
    // segments [t0, t1] of states, last first
    for (int t0 = ((h->T - 1) / h->every) * h->every; t0 >= 0; t0 -= h->every) {
        const int t1 = std::min(t0 + h->every - 1, h->T - 1);
        const auto state = [&](int t) -> char * {
            return t == t0 ? static_cast<char *>(h->ckpt[t0 / h->every])
                           : static_cast<char *>(h->stack) + h->sb * (size_t)(t - t0);
        };
        // recompute H_{t0+1} .. H_{t1} from the checkpoint H_{t0} into the stack
        for (int t = t0 + 1, n; t <= t1; t += n) {
            n = std::min(h->fwd.K, t1 - t + 1);
            f.src = state(t - 1);
            f.dst = state(t);
            fwd(h, f, t, n, st);
        }
        LBM_LAUNCH_CHECK();
        // adjoint iterations t = t1+1 .. t0+1, reading H_{t-1}
        for (int t = t1 + 1, n; t > t0; t -= n) {
            n = std::min(h->adj.K, t - t0);
            a.lam_in = h->lam[cur];
            a.lam_out = h->lam[cur ^= 1];
            adj(h, a, t, n, state, st);
        }
        LBM_LAUNCH_CHECK();
    }
    std::vector<double> ab(h->ny);
    LBM_HIP_TRY(hipMemcpyAsync(ab.data(), h->d_abar, sizeof(double) * h->ny,
                               hipMemcpyDeviceToHost, st));
    LBM_HIP_TRY(hipStreamSynchronize(st));
    double g = 0.0;
    for (int j = 0; j < h->ny; ++j) g += ab[j];
    *umax_grad = g;
    return LBM_OK;
}

extern "C" int lbm_pbb_drag_history(const lbm_pbb *h, double *out_host)
{
    if (!h || !out_host || h->drag.empty())
        return set_error(LBM_ERR_ARG, "lbm_pbb_drag_history: no forward run");
    std::copy(h->drag.begin(), h->drag.end(), out_host);
    return LBM_OK;
}

extern "C" int lbm_pbb_final_state(lbm_pbb *h, void *dst_dev, void *stream)
{
    if (!h || !dst_dev) return set_error(LBM_ERR_ARG, "lbm_pbb_final_state: bad argument");
    LBM_HIP_TRY(hipMemcpyAsync(dst_dev, h->last ? h->last : h->ping[0], h->sb, hipMemcpyDeviceToDevice,
                               SS(stream)));
    return LBM_OK;
}
