// d2q9_tile.hip -- several iterations per launch, in LDS.  Compiled once per
// storage form (LBM_TILE_STORE).
//
// A work-group loads a rectangle r[0] of the lattice (post-collision state of
// iteration it - 1), advances it K iterations in LDS, each on a rectangle r[l]
// one node smaller on the sides that face other tiles, and stores the
// rectangle r[K] it owns (d2q9_plan.h).  Every iteration evaluates the
// one-iteration kernels' expressions on the same values -- float forms round
// each population through the storage form between iterations -- so the state
// after K iterations is theirs bit for bit.
//
// Why: one iteration per launch is bound by HBM on large lattices (18
// populations per update; FP64 8192x2048 434 us) and by the launch and its
// chain of memory rounds on small ones (7 us whatever the size up to 200x200).
// K iterations per launch move the populations once, plus the overlap of the
// rectangles, and pay the chain once; an iteration is then bound by the
// collision's arithmetic, ~175 FP64 instructions per node, with 1.2-1.5 times
// as many nodes computed as owned.  Measured per iteration (MI355X, one
// iteration per launch in brackets): FP64 cavity 100x100 1.7 us (7.0),
// 200x200 1.9 (7.5), Turek channel 1073x200 4.1 (10.7), 8192x2048 obstacle
// array 214 (428); FP32 channel 541x101 1.9 (9.4), array 83 (212); FP16 array
// 88 (107), BF16 88 (112), f16e 116 (144), f16e8 115 (140).  On the array the
// vector units are 60 (FP64) to 80 % (FP16) busy at the 1.9-2.2 GHz held.
//
// Layout: the nine planes of the rectangle lie one after the other in LDS, in
// float or double.  Every work-item keeps its M nodes for the whole launch:
// all pulls of an iteration go to registers, a barrier, then all results go
// back to the same planes, so one copy of the state suffices and the LDS holds
// twice the nodes.  Perimeter nodes go to waves of their own, one kind per
// wave, so that the wall routines run beside the inner nodes' collision
// instead of after it (corner tile 4600 -> 1650 cycles per iteration).  Wall
// inputs of all iterations are fetched with the first loads (one chain of
// dependent loads instead of one per iteration).  Link values are computed
// link-major, one per work-item, between the pulls and the barrier.
#include "d2q9_tile.h"

namespace lbm {
namespace {

// A copy the compiler knows nothing about: what is derived from it inside a
// rarely taken branch of the iteration loop is not computed ahead of the loop
// by every work-item (in registers every wave then pays for).
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// A node as stored, and decoded to the values the pulls return (f in FP64,
// h = f - w in the float forms).
template <int S> struct Raw {
    typename Store<S>::s_t q[9];
    uint32_t v;                                 // velocity word (shifted forms)
};
template <int S> __device__ __forceinline__ void tile_load(const Params &p, int cell, Raw<S> &r)
{
    using s_t = typename Store<S>::s_t;
    const s_t *src = static_cast<const s_t *>(p.src);
#pragma unroll
    for (int q = 0; q < 9; ++q)
        r.q[q] = ld_base<s_t>(sbase(src + (size_t)q * p.N), (uint32_t)cell * (uint32_t)sizeof(s_t));
    if constexpr (shifted(S)) {
        using w_t = typename Vel<S>::w_t;
        r.v = ld_base<w_t>(sbase(Store<S>::vel(src, p.N)), (uint32_t)cell * (uint32_t)sizeof(w_t));
    }
}
template <int S>
__device__ __forceinline__ void tile_decode(const Params &p, const Raw<S> &r, typename Store<S>::T *v)
{
    using St = Store<S>;
    if constexpr (S == LBM_STORE_F16E8) {
        float a, b, e[9];
        e8_unpack(r.v, a, b);
        e8_shifts(a, b, e);
#pragma unroll
        for (int q = 0; q < 9; ++q) v[q] = add_lo(e[q], __builtin_bit_cast(uint16_t, r.q[q]));
    } else {
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            if constexpr (S == LBM_STORE_F64 || S == LBM_STORE_F32) v[q] = r.q[q];
            else if constexpr (S == LBM_STORE_F16) v[q] = from_half(__builtin_bit_cast(uint16_t, r.q[q]));
            else if constexpr (shifted(S)) v[q] = St::dec(q, r.q[q], (typename Vel<S>::w_t)r.v);
            else v[q] = St::dec(p, q, r.q[q]);
        }
    }
}

// w: pairs (1,2) (3,4) (5,6) (7,8), then 0
template <class E>
__device__ __forceinline__ void tile_store_halves(const Params &p, E *dst, int cell, const uint32_t *w)
{
    const uint32_t off = (uint32_t)opaque(cell) * 2u;
    st_off(sbase(dst), off, (uint16_t)w[4]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        st_off(sbase(dst + (size_t)(2 * j + 1) * p.N), off, (uint16_t)w[j]);
        st_off(sbase(dst + (size_t)(2 * j + 2) * p.N), off, (uint16_t)(w[j] >> 16));
    }
}

// Post-collision values of one node: to LDS as the next iteration's pulls
// read them (the stored value decoded), or to the state buffer.
template <int S, int CAP>
__device__ __forceinline__ void tile_store(const Params &p, bool last, int cell, int li,
                                           typename Store<S>::T *lds, float *h, float ux, float uy)
{
    using St = Store<S>;
    using s_t = typename St::s_t;
    s_t *dst = static_cast<s_t *>(p.dst);
    if constexpr (S == LBM_STORE_F32) {
        if (last) {
            const uint32_t off = (uint32_t)opaque(cell) * 4u;
#pragma unroll
            for (int q = 0; q < 9; ++q) st_off(sbase(dst + (size_t)q * p.N), off, h[q]);
        } else {
#pragma unroll
            for (int q = 0; q < 9; ++q) lds[q * CAP + li] = h[q];
        }
    } else if constexpr (shifted(S)) {
        using w_t = typename Vel<S>::w_t;
        float a, b;   // the velocity as the reader unpacks it
        w_t v;
        if constexpr (S == LBM_STORE_F16E8) {
            v = e8_pack(ux, uy, a, b);
        } else {
            v = Vel<S>::pack(ux, uy);
            Vel<S>::unpack(v, a, b);
        }
        float e[9];
        if constexpr (S == LBM_STORE_F16E8) {
            e8_shifts(a, b, e);
        } else {
#pragma unroll
            for (int q = 0; q < 9; ++q) e[q] = eq_shift(q, a, b);
        }
        uint32_t w[5];                          // pairs (1,2) (3,4) (5,6) (7,8); 0
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = to_half2(h[2 * j + 1] - e[2 * j + 1], h[2 * j + 2] - e[2 * j + 2]);
        w[4] = __builtin_bit_cast(uint16_t, to_half(h[0] - e[0]));
        if (last) {
            st_off(sbase(dst + vel_offset(p.N)), (uint32_t)opaque(cell) * (uint32_t)sizeof(w_t), v);
            tile_store_halves(p, dst, cell, w);
        } else {
            lds[li] = add_lo(e[0], w[4]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int q = 2 * j + 1;
                lds[q * CAP + li] = add_lo(e[q], w[j]);
                lds[(q + 1) * CAP + li] = add_hi(e[q + 1], w[j]);
            }
        }
    } else if constexpr (S == LBM_STORE_F16) {
        uint32_t w[5];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = to_half2(h[2 * j + 1], h[2 * j + 2]);
        w[4] = __builtin_bit_cast(uint16_t, to_half(h[0]));
        if (last) {
            tile_store_halves(p, dst, cell, w);
        } else {
            const auto half = [](uint32_t u) { return (float)__builtin_bit_cast(_Float16, (uint16_t)u); };
            lds[li] = half(w[4]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                lds[(2 * j + 1) * CAP + li] = half(w[j]);
                lds[(2 * j + 2) * CAP + li] = half(w[j] >> 16);
            }
        }
    } else {
        s_t raw[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) raw[q] = St::enc(p, q, h[q]);
        if (last) {
            const uint32_t off = (uint32_t)opaque(cell) * (uint32_t)sizeof(s_t);
#pragma unroll
            for (int q = 0; q < 9; ++q) st_off(sbase(dst + (size_t)q * p.N), off, raw[q]);
        } else {
#pragma unroll
            for (int q = 0; q < 9; ++q) lds[q * CAP + li] = St::dec(p, q, raw[q]);
        }
    }
}

// Collision of one node's post-boundary values v (f or h) and its store.
template <int S, int CAP>
__device__ __forceinline__ void tile_collide(const Params &p, bool last, int cell, int li,
                                             typename Store<S>::T *lds, typename Store<S>::T *v)
{
    if constexpr (S == LBM_STORE_F64) {
        double o[9], r, ux, uy;
        collide_f64(p, v, o, r, ux, uy);
        double *dst = static_cast<double *>(p.dst);
        if (last) {
            const uint32_t off = (uint32_t)opaque(cell) * 8u;
#pragma unroll
            for (int q = 0; q < 9; ++q) st_off(sbase(dst + (size_t)q * p.N), off, o[q]);
        } else {
#pragma unroll
            for (int q = 0; q < 9; ++q) lds[q * CAP + li] = o[q];
        }
    } else {
        float rho, ux, uy;
        collide_h(coll_consts(p), v, rho, ux, uy);
        tile_store<S, CAP>(p, last, cell, li, lds, v, ux, uy);
    }
}

// Wall input v (0 or 1) of perimeter slot `slot` of region r (tile_input_slots
// order: bottom, top, left, right) in ring row `row`: the velocity components
// of a velocity wall; density and tangential velocity of the pressure outlet.
__device__ __forceinline__ double tile_input(const Params &p, const TileRect &r, int row, int slot,
                                             int v)
{
    const int nb = r.y == 0 ? r.w : 0, nt = r.y + r.h == p.ny ? r.w : 0;
    const int nl = r.x == 0 ? r.h : 0;
    int side, i, len;
    if (slot < nb + nt) {
        side = slot < nb ? LBM_SIDE_BOTTOM : LBM_SIDE_TOP;
        i = r.x + (slot < nb ? slot : slot - nb);
        len = p.nx;
    } else {
        const bool left = slot - nb - nt < nl;
        side = left ? LBM_SIDE_LEFT : LBM_SIDE_RIGHT;
        i = r.y + slot - nb - nt - (left ? 0 : nl);
        len = p.ny;
        if (!left && v == 0 && p.bc_right == LBM_BC_PRESSURE) side = LBM_SIDE_RHO_RIGHT;
    }
    i += v * len;
    if (p.amp) {
        // selected one by one: indexing the parameter block with a run-time
        // value would move it to scratch memory
        const double *pr = side == LBM_SIDE_BOTTOM  ? p.prof[0]
                           : side == LBM_SIDE_LEFT  ? p.prof[1]
                           : side == LBM_SIDE_TOP   ? p.prof[2]
                           : side == LBM_SIDE_RIGHT ? p.prof[3]
                                                    : p.prof[4];
        return p.amp[(size_t)row * p.amp_stride + side] * pr[i];
    }
    return p.pool[p.inlet_off[row * 5 + side] + i];
}

// Post-link populations of a wall node from its pulls v (deviations in the
// float forms).  Sources beyond the wall hold a neighbouring value: they are
// the populations the wall or corner routine sets without reading them.
template <int S>
__device__ __forceinline__ void tile_full(const typename Store<S>::T *v, uint32_t tab,
                                          const typename Store<S>::T *s_lv,
                                          typename Store<S>::T *f)
{
    using T = typename Store<S>::T;
#pragma unroll
    for (int q = 0; q < 9; ++q) f[q] = S == LBM_STORE_F64 ? v[q] : weight<T>(q) + v[q];
    if (tab & 511u) {
        const T *lv = s_lv + (tab >> 9);
#pragma unroll
        for (int q = 1; q < 9; ++q)
            if ((tab >> q) & 1u) {
                const T t = lv[__popc(tab & ((1u << q) - 1u) & 511u)];
                f[q] = S == LBM_STORE_F64 ? t : weight<T>(q) + t;
            }
    }
}

// Last level of a launch that computes node (x, y) of r[lev0 + 1] (the
// rectangles are nested): K less its distance from r[K], or by the rectangles
// where a link stencil or a corner made one of them larger.
__device__ __forceinline__ int tile_last_level(const TileDesc &D, int K, int lev0, int x, int y)
{
    if (D.regular) {
        const TileRect r = D.r[K];
        return K - max(max(max(r.x - x, x - r.x - r.w + 1), max(r.y - y, y - r.y - r.h + 1)), 0);
    }
    int lm = lev0 + 1;
#pragma unroll
    for (int l = 2; l <= TILE_MAX_LEVELS; ++l) {
        const TileRect r = D.r[l];
        const bool in = (unsigned)(x - r.x) < (unsigned)r.w && (unsigned)(y - r.y) < (unsigned)r.h;
        if (l > lev0 + 1 && l <= K && in) lm = l;
    }
    return lm;
}

// NT work-items, M nodes each, regions of up to CAP = NT * M nodes.
template <int S, int NT, int M, bool LINKS>
__device__ __forceinline__ void tile_run(const Params &p, const TileDesc &D,
                                         const TileLink *__restrict__ links,
                                         const uint32_t *__restrict__ nodes, int K, int lev0,
                                         int n_in, char *smem)
{
    using T = typename Store<S>::T;
    constexpr int CAP = NT * M;
    constexpr bool F64 = S == LBM_STORE_F64;
    T *const lds = reinterpret_cast<T *>(smem);
    T *const s_in = lds + 9 * CAP;              // wall inputs [level][2][n_in]
    T *const s_lv = s_in + 2 * K * n_in;        // link values
    const int tid = threadIdx.x;
    const int nx = p.nx, ny = p.ny, lx = nx - 1, ly = ny - 1;
    const TileRect r0 = D.r[lev0], r1 = D.r[lev0 + 1];
    const int a0 = r0.w * r0.h, h0 = r0.h;
    const int n_links = D.n_links;
    // the device counter of the launch's first ring row, ahead of its use
    const int base = *(const __attribute__((address_space(4))) int *)p.base;

    // ---- load r0: all planes of all nodes in flight
    Raw<S> raw[M];
    {
        const uint32_t mg = D.mh[lev0];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int n = tid + m * NT;
            const int x = (int)__umulhi((uint32_t)n, mg), y = n - x * h0;
            const int cell = (r0.x + x) * ny + r0.y + y;
            if (n < a0) tile_load<S>(p, cell, raw[m]);
        }
    }
    const TilePerim P = tile_perim(r1, nx, ny);
    int row0 = 0;                               // ring row of iteration it - 1
    if (P.slots || (LINKS && n_links)) {
        row0 = (base + p.k) % p.ring;
        if (row0 < 0) row0 += p.ring;
    }
    // the wall inputs of every iteration of the launch
    int in_at = -1;                             // the first one is stored after the set-up
    double in_v = 0.0;
    if (P.slots) {
        const int ns = tile_input_slots(r0, nx, ny);
        for (int i = tid; i < 2 * ns * (K - lev0); i += NT) {
            const int j = i / ns, sl = i - j * ns;      // j = 2 * level + component
            const double t = tile_input(p, r0, (row0 + (j >> 1)) % p.ring, sl, j & 1);
            if (i == tid) {
                in_at = j * n_in + sl;
                in_v = t;
            } else {
                s_in[j * n_in + sl] = T(t);
            }
        }
    }

    // ---- this work-item's nodes of r1: perimeter nodes first, a wave of one
    // kind each (their routines then run beside the inner nodes' waves)
    int li[M], cell[M], lm[M];                  // node in LDS, in the lattice; last level
    uint32_t lk[M];                             // link table entry
    int type = NODE_INNER, slot = 0;            // perimeter nodes: m = 0 only
    {
        const int hi = r1.h - P.tb - P.tt;
        const uint32_t mg = D.mi[lev0 + 1];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            li[m] = cell[m] = lm[m] = 0;
            lk[m] = 0;
            int n = tid + m * NT, x = 0, y = 0;
            bool on;
            if (m == 0 && n < P.slots) {
                int t;
                on = tile_perim_node(r1, P, n, x, y, t);
                type = t;
                if (t == NODE_CORNER)           // the wall node beside it
                    slot = (y == 0 || !(r0.y == 0) ? 0 : r0.w) + (x == 0 ? 1 : lx - 1) - r0.x;
                else if (t == NODE_BOTTOM || t == NODE_TOP)
                    slot = (t == NODE_BOTTOM || !(r0.y == 0) ? 0 : r0.w) + x - r0.x;
                else
                    slot = (r0.y == 0 ? r0.w : 0) + (r0.y + r0.h == ny ? r0.w : 0) +
                           (t == NODE_LEFT || !(r0.x == 0) ? 0 : r0.h) + y - r0.y;
            } else {
                n -= P.slots;
                on = n < P.inner;
                const int xx = hi == 1 ? n : (int)__umulhi((uint32_t)n, mg);
                x = r1.x + P.tl + xx;
                y = r1.y + P.tb + n - xx * hi;
            }
            if (!on) continue;
            li[m] = (x - r0.x) * h0 + (y - r0.y);
            cell[m] = x * ny + y;
            lm[m] = tile_last_level(D, K, lev0, x, y);
            if (LINKS && n_links) lk[m] = nodes[D.node0 + (x - D.r[0].x) * D.r[0].h + (y - D.r[0].y)];
        }
    }
    // ---- this work-item's link (at most NT per tile)
    int lli = 0, llev = 0;                      // its node in LDS; last level
    int lsA = 0, lsB = 0, lsC = 0, lslot = -1;  // sources; drag slot, if it is stored here
    int lq = 0;
    T lc0 = T(1), lc1 = T(0), lc2 = T(0);
    bool lmode = false;
    if (LINKS && tid < n_links) {
        const TileLink L = links[D.link0 + tid];
        const int x = D.r[0].x + L.x, y = D.r[0].y + L.y;
        if ((unsigned)(x - r1.x) < (unsigned)r1.w && (unsigned)(y - r1.y) < (unsigned)r1.h) {
            lli = (x - r0.x) * h0 + (y - r0.y);
            int dx = 0, qb = 0;                 // step along -c_q = c_qb in LDS
#pragma unroll
            for (int q = 1; q < 9; ++q)
                if (q == L.q) {
                    dx = -CX[q] * h0 - CY[q];
                    qb = NS[q];
                }
            lq = L.q;
            lmode = L.mode != 0;
            lsA = L.q * CAP + lli;
            lsB = L.mode == 1 ? lsA + dx : qb * CAP + lli;
            lsC = L.mode == 1 ? lsA + 2 * dx : qb * CAP + lli + dx;
            lc0 = T(L.c0);
            lc1 = T(L.c1);
            lc2 = T(L.c2);
            // the drag terms of a perimeter node follow its wall routine
            if (x > 0 && x < lx && y > 0 && y < ly) lslot = L.dslot;
            llev = tile_last_level(D, K, lev0, x, y);
        }
    }
    if (in_at >= 0) s_in[in_at] = T(in_v);
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int n = opaque(tid + m * NT);      // (so that no decoding moves up to its loads)
        if (n < a0) {
            T v[9];
            tile_decode<S>(p, raw[m], v);
#pragma unroll
            for (int q = 0; q < 9; ++q) lds[q * CAP + n] = v[q];
        }
    }
    __syncthreads();

    // ---- iterations
    int row = row0;
#pragma unroll 1
    for (int l = lev0 + 1; l <= K; ++l) {
        const bool last = l == K;
        T f[M][9];
        T fn[6];                                // corner: the wall node beside it
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (l > lm[m]) continue;
            const int c = li[m], e = c - h0, w = c + h0;   // columns x, x - 1, x + 1
            f[m][0] = lds[0 * CAP + c];
            f[m][1] = lds[1 * CAP + e];
            f[m][2] = lds[2 * CAP + w];
            f[m][3] = lds[3 * CAP + c - 1];
            f[m][4] = lds[4 * CAP + c + 1];
            f[m][5] = lds[5 * CAP + e - 1];
            f[m][6] = lds[6 * CAP + w + 1];
            f[m][7] = lds[7 * CAP + w - 1];
            f[m][8] = lds[8 * CAP + e + 1];
        }
        if (type == NODE_CORNER && l <= lm[0]) {
            // the populations its wall routine reads: 0, 1, 2 and those that
            // leave through the wall
            const int node = opaque(cell[0]);
            const bool left = node < ny, low = node == 0 || node == lx * ny;
            const int c = left ? li[0] + h0 : li[0] - h0, e = c - h0, w = c + h0;
            fn[0] = lds[c];
            fn[1] = lds[1 * CAP + e];
            fn[2] = lds[2 * CAP + w];
            fn[3] = lds[low ? 4 * CAP + c + 1 : 3 * CAP + c - 1];
            fn[4] = lds[low ? 6 * CAP + w + 1 : 5 * CAP + e - 1];
            fn[5] = lds[low ? 8 * CAP + e + 1 : 7 * CAP + w - 1];
        }
        if (LINKS && l <= llev) {
            const T A = lds[lsA];
            T t = A;
            if (lmode) t = (lc0 * A + lc1 * lds[lsB]) + lc2 * lds[lsC];
            s_lv[tid] = t;
            if (lslot >= 0) {
                double *ring = p.drag_ring + (size_t)row * p.n_links;
                if constexpr (F64) ring[lslot] = A + t;
                else ring[lslot] = 2.0 * weight<double>(lq) + ((double)A + (double)t);
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (l > lm[m]) continue;
            if (m == 0 && type != NODE_INNER) {
                T fo[9], r = T(0), ux = T(0);
                const uint32_t own = LINKS ? (uint32_t)opaque((int)lk[0]) : 0u;
                tile_full<S>(f[0], own, s_lv, fo);
                const int j = 2 * (l - lev0 - 1) * n_in + slot;
                const T a = s_in[j], b = s_in[j + n_in];
                if (type == NODE_CORNER) {
                    const int node = opaque(cell[0]);
                    const bool left = node < ny, low = node == 0 || node == lx * ny;
                    uint32_t tab = 0;
                    if (LINKS && n_links)
                        tab = nodes[D.node0 + ((left ? 1 : lx - 1) - D.r[0].x) * D.r[0].h +
                                    ((low ? 0 : ly) - D.r[0].y)];
                    T h[6];
#pragma unroll
                    for (int k = 0; k < 6; ++k) {
                        const int qh = k < 3 ? k : 2 * k - 3, q = k < 3 || !low ? qh : qh + 1;
                        T t = fn[k];
                        if ((tab >> q) & 1u)
                            t = s_lv[(tab >> 9) + __popc(tab & ((1u << q) - 1u) & 511u)];
                        h[k] = F64 ? t : weight<T>(qh) + t;
                    }
                    zh_corner_beside(fo, left, low, h, a, b);
                } else if (type == NODE_BOTTOM) {
                    zh_bottom(fo, a, b, r);
                } else if (type == NODE_TOP) {
                    zh_top(fo, a, b, r);
                } else if (type == NODE_LEFT) {
                    zh_left(fo, a, b, r);
                } else if (p.bc_right == LBM_BC_VELOCITY) {
                    zh_right_vel(fo, a, b, r);
                } else {
                    zh_right_pres(fo, a, b, ux);
                }
#pragma unroll
                for (int q = 0; q < 9; ++q) f[0][q] = F64 ? fo[q] : fo[q] - weight<T>(q);
#pragma unroll 1
                for (int k = 0; k < __popc(own & 511u); ++k) {
                    const TileLink &Q = links[D.link0 + (own >> 9) + k];
                    if (Q.dslot < 0) continue;
                    const T A = lds[Q.q * CAP + li[0]];
                    T t = T(0);
#pragma unroll
                    for (int q = 1; q < 9; ++q)
                        if (q == NS[Q.q]) t = f[0][q];
                    double *ring = p.drag_ring + (size_t)row * p.n_links;
                    if constexpr (F64) ring[Q.dslot] = A + t;
                    else ring[Q.dslot] = 2.0 * weight<double>(Q.q) + ((double)A + (double)t);
                }
            } else if (LINKS && (lk[m] & 511u)) {
                const uint32_t own = (uint32_t)opaque((int)lk[m]);
                const T *lv = s_lv + (own >> 9);
#pragma unroll
                for (int q = 1; q < 9; ++q)
                    if ((own >> q) & 1u) f[m][q] = lv[__popc(own & ((1u << q) - 1u) & 511u)];
            }
            tile_collide<S, CAP>(p, last, cell[m], li[m], lds, f[m]);
        }
        if (++row >= p.ring) row -= p.ring;
        if (!last) __syncthreads();
    }
}

// One lattice.
template <int S, int NT, int M, bool LINKS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_tile(
    Params p, const TileDesc *__restrict__ tiles, const TileLink *__restrict__ links,
    const uint32_t *__restrict__ nodes, int K, int lev0, int n_in)
{
    extern __shared__ __align__(16) char smem[];
    touch_params(p);
    tile_run<S, NT, M, LINKS>(p, tiles[xcd_tile(blockIdx.x, gridDim.x)], links, nodes, K, lev0,
                              n_in, smem);
}

// The cases of a batch: parameters per case and parity, as k_batch_step's.
template <int S, int NT, int M, bool LINKS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_batch_tile(
    const Params *__restrict__ cases, const TileDesc *__restrict__ tiles,
    const TileLink *__restrict__ links, const uint32_t *__restrict__ nodes, int K, int lev0,
    int n_in, int k, const int *base, int parity)
{
    extern __shared__ __align__(16) char smem[];
    const TileDesc &D = tiles[xcd_tile(blockIdx.x, gridDim.x)];
    touch_params(cases[2 * D.cse + parity]);
    Params p = cases[2 * D.cse + parity];
    p.k = k;
    p.base = base;
    tile_run<S, NT, M, LINKS>(p, D, links, nodes, K, lev0, n_in, smem);
}

template <int S, int NT, int M, bool LINKS> void launch_tile_k(const TileLaunch &a)
{
    const TileSet &t = a.t;
    if (a.p)
        k_tile<S, NT, M, LINKS><<<t.n, NT, t.lds, a.s>>>(*a.p, t.d_tiles, t.d_links, t.d_nodes, t.K,
                                                        t.K - a.n, t.n_in);
    else
        k_batch_tile<S, NT, M, LINKS><<<t.n, NT, t.lds, a.s>>>(a.cases, t.d_tiles, t.d_links,
                                                              t.d_nodes, t.K, t.K - a.n, t.n_in,
                                                              a.k, a.base, a.parity);
}

template <int S, int NT, int M> void launch_tile_m(const TileLaunch &a)
{
    if (a.t.links) launch_tile_k<S, NT, M, true>(a);
    else launch_tile_k<S, NT, M, false>(a);
}

}  // namespace

// the shapes of tile_kinds
template <int S> void launch_tile_s(const TileLaunch &a)
{
    switch (a.t.cfg) {
    case 0: launch_tile_m<S, 512, 1>(a); break;
    case 1: launch_tile_m<S, 512, 2>(a); break;
    case 2: launch_tile_m<S, 1024, 2>(a); break;
    case 3: if constexpr (S != LBM_STORE_F64) launch_tile_m<S, 512, 4>(a); break;
    default: if constexpr (S != LBM_STORE_F64) launch_tile_m<S, 1024, 4>(a); break;
    }
}

template void launch_tile_s<LBM_TILE_STORE>(const TileLaunch &a);

}  // namespace lbm
