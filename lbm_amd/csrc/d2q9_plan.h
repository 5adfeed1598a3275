// d2q9_plan.h -- host-side plan of the multi-iteration launches: which nodes
// each work-group loads, computes and stores when one launch advances a
// lattice by several iterations in LDS (d2q9_tile.h).  Plain C++, no device
// code: a CPU test includes it.
#pragma once
#include <stdint.h>
#include <algorithm>
#include <vector>

#ifdef __HIPCC__
#define LBM_HD __host__ __device__
#else
#define LBM_HD
#endif

namespace lbm {

constexpr int TILE_MAX_LEVELS = 7;   // iterations of one launch, at most

struct TileRect {
    int x, y, w, h;                  // nodes [x, x + w) x [y, y + h)
};

// One work-group's share of a K-iteration launch.  r[K] are the nodes it owns
// and stores; r[l - 1] holds every node that level l of r[l] reads, clipped to
// the lattice; r[0] is loaded.  A launch of fewer iterations, k, starts from
// r[K - k].
struct TileDesc {
    TileRect r[TILE_MAX_LEVELS + 1];
    int link0, n_links;              // its records in the link list
    int node0;                       // its node table (r[0], y fastest), if n_links
    int cse;                         // case of a batch
    int regular;                     // r[l - 1] is r[l] grown by one node, clipped
    uint32_t mh[TILE_MAX_LEVELS + 1], mi[TILE_MAX_LEVELS + 1];   // 2^32 / height, of r[l] and of
                                     // its inner nodes: n / height for n < 2^16
};

// An obstacle link seen from a tile.  mode 0: plain bounce-back; 1: sources
// plane q at the node and at 1 and 2 nodes along -c_q (p < 0.5); 2: plane q at
// the node, plane qb at the node and 1 node along -c_q.
struct TileLink {
    int16_t x, y;                    // node, relative to r[0]
    int8_t q, mode, pad0, pad1;
    int32_t dslot;                   // drag ring slot, or -1 when the tile does not own the node
    int32_t pad2;
    double c0, c1, c2;
};

// A link as the planner reads it, sorted by node (x major) and direction.
struct PlanLink {
    int x, y, q, mode, dslot;
    double c0, c1, c2;
};

struct TileShape {
    int K;                           // iterations per launch (odd: the state buffers alternate)
    int ntx, nty;                    // tiles along x and y
    int cap, nt;                     // nodes of r[0] and work-items, at most
    bool adjoint = false;            // levels compute r[l - 1] and write into r[l]
};

struct TilePlan {
    std::vector<TileDesc> tiles;
    std::vector<TileLink> links;
    std::vector<uint32_t> nodes;     // link tiles: first link << 9 | directions qb with a link
    int max_area = 0, max_links = 0, max_inputs = 0;
};

// Wall inputs of a tile: one value pair per perimeter node of r[0] and level;
// bottom, top, left, right in this order.
LBM_HD inline int tile_input_slots(const TileRect &r, int nx, int ny)
{
    return (r.y == 0 ? r.w : 0) + (r.y + r.h == ny ? r.w : 0) + (r.x == 0 ? r.h : 0) +
           (r.x + r.w == nx ? r.h : 0);
}

enum { NODE_INNER = 0, NODE_BOTTOM, NODE_TOP, NODE_LEFT, NODE_RIGHT, NODE_CORNER };

// Order of a region's nodes over the work-items: its corners, its bottom and
// top wall nodes, its left and right ones, each group padded to whole waves,
// then the inner nodes.
struct TilePerim {
    int tl, tr, tb, tt;              // 1: the region touches that side of the lattice
    int bt0, lr0, slots;             // first bottom/top and left/right slot, first inner slot
    int nc, nbt, nlr, inner;         // nodes of each group
};

LBM_HD inline TilePerim tile_perim(const TileRect &r, int nx, int ny)
{
    TilePerim P;
    P.tl = r.x == 0;
    P.tr = r.x + r.w == nx;
    P.tb = r.y == 0;
    P.tt = r.y + r.h == ny;
    const int wi = r.w - P.tl - P.tr, hi = r.h - P.tb - P.tt;
    P.nc = (P.tl + P.tr) * (P.tb + P.tt);
    P.nbt = (P.tb + P.tt) * wi;
    P.nlr = (P.tl + P.tr) * hi;
    P.inner = wi * hi;
    P.bt0 = P.nc ? 64 : 0;
    P.lr0 = P.bt0 + ((P.nbt + 63) & ~63);
    P.slots = P.lr0 + ((P.nlr + 63) & ~63);
    return P;
}

// Perimeter slot n < P.slots -> node and kind; false on padding.
LBM_HD inline bool tile_perim_node(const TileRect &r, const TilePerim &P, int n, int &x, int &y,
                                   int &type)
{
    const int x1 = r.x + r.w - 1, y1 = r.y + r.h - 1;
    type = NODE_INNER;
    if (n < P.bt0) {
        if (n >= P.nc) return false;
        const int per = P.tb + P.tt, a = n / per, b = n - a * per;
        x = a == 0 && P.tl ? r.x : x1;
        y = b == 0 && P.tb ? r.y : y1;
        type = NODE_CORNER;
    } else if (n < P.lr0) {
        const int k = n - P.bt0, wi = r.w - P.tl - P.tr;
        if (k >= P.nbt) return false;
        const bool low = P.tb && k < wi;
        x = r.x + P.tl + (low || !P.tb ? k : k - wi);
        y = low ? r.y : y1;
        type = low ? NODE_BOTTOM : NODE_TOP;
    } else {
        const int k = n - P.lr0, hi = r.h - P.tb - P.tt;
        if (k >= P.nlr) return false;
        const bool left = P.tl && k < hi;
        y = r.y + P.tb + (left || !P.tl ? k : k - hi);
        x = left ? r.x : x1;
        type = left ? NODE_LEFT : NODE_RIGHT;
    }
    return true;
}

// A link near a tile: its node, its stencil's direction and reach (0, 1, 2 nodes).
struct NearLink {
    int x, y;
    int8_t dx, dy, reach;
    const PlanLink *link;
};

// Plans the tile of nodes [xa, xb) x [ya, yb): adds it to the plan, or its two
// halves where a link stencil makes it larger than the shape allows.
// recip[h] = 2^32 / h.  near: the links (sorted as the lattice's) within 2 K + 2 nodes of the tile,
// at least: a level's stencils reach two nodes beyond the next one.
inline bool plan_one(int nx, int ny, const TileShape &s, const std::vector<NearLink> &near,
                     const std::vector<uint32_t> &recip, int cse, int xa, int xb, int ya, int yb,
                     TilePlan &out)
{
    static const int ns[9] = {0, 2, 1, 4, 3, 6, 5, 8, 7};
    if (xb - xa < 2 || yb - ya < 2) return false;
    out.tiles.emplace_back();
    TileDesc &d = out.tiles.back();                  // taken back if it does not fit
    d.cse = cse;
    d.regular = 1;
    int lo_x = xa, hi_x = xb - 1, lo_y = ya, hi_y = yb - 1;   // inclusive
    static thread_local std::vector<int> far;
    far.resize(4 * near.size());
    int *const fx = far.data(), *const fy = fx + near.size(), *const dx = fy + near.size(),
              *const dy = dx + near.size();
    size_t n_far = 0;
    for (const NearLink &L : near) {
        if (L.reach != 2) continue;
        fx[n_far] = L.x;
        fy[n_far] = L.y;
        dx[n_far] = L.dx;
        dy[n_far++] = L.dy;
    }
    for (int l = s.K; l >= 0; --l) {
        d.r[l] = TileRect{lo_x, lo_y, hi_x - lo_x + 1, hi_y - lo_y + 1};
        const int h = d.r[l].h, hi = h - (lo_y == 0) - (hi_y == ny - 1);
        d.mh[l] = recip[h];
        d.mi[l] = hi > 1 ? recip[hi] : 0u;
        if (l == 0) break;
        // a stencil of two nodes reaches beyond the next level from the edge only
        int wide = 0;
        for (size_t i = 0; i < n_far; ++i) {
            const int x = fx[i], y = fy[i];
            const int in = (x >= lo_x) & (x <= hi_x) & (y >= lo_y) & (y <= hi_y);
            const int w = ((x == lo_x) & (dx[i] < 0)) | ((x == hi_x) & (dx[i] > 0)) << 1 |
                          ((y == lo_y) & (dy[i] < 0)) << 2 | ((y == hi_y) & (dy[i] > 0)) << 3;
            wide |= -in & w;
        }
        int px = wide & 1 ? lo_x - 2 : std::max(lo_x - 1, 0);
        int qx = wide & 2 ? hi_x + 2 : std::min(hi_x + 1, nx - 1);
        int py = wide & 4 ? lo_y - 2 : std::max(lo_y - 1, 0);
        int qy = wide & 8 ? hi_y + 2 : std::min(hi_y + 1, ny - 1);
        if (wide) d.regular = 0;
        const int px0 = px, qx0 = qx, py0 = py, qy0 = qy;
        // a wall node beside a corner carries the corner's adjoint
        if (s.adjoint && (py == 0 || qy == ny - 1)) {
            if (px == 1) px = 0;
            if (qx == nx - 2) qx = nx - 1;
        }
        // a corner takes the density of the wall node beside it
        if (lo_y == 0 || hi_y == ny - 1) {
            if (lo_x == 0) qx = std::max(qx, std::min(2, nx - 1));
            if (hi_x == nx - 1) px = std::min(px, std::max(nx - 3, 0));
        }
        if (px != px0 || qx != qx0 || py != py0 || qy != qy0) d.regular = 0;
        lo_x = px;
        hi_x = qx;
        lo_y = py;
        hi_y = qy;
    }
    const TileRect &r0 = d.r[0], &r1 = d.r[1];
    const TilePerim P = tile_perim(s.adjoint ? r0 : r1, nx, ny);
    bool fits = (int64_t)r0.w * r0.h <= s.cap && P.slots <= s.nt && P.slots + P.inner <= s.cap;
    const auto inside = [&](const NearLink &L) {
        return L.x >= r1.x && L.x < r1.x + r1.w && L.y >= r1.y && L.y < r1.y + r1.h;
    };
    for (const NearLink &n : near) d.n_links += inside(n);
    fits = fits && d.n_links <= s.nt;
    if (!fits) {
        out.tiles.pop_back();
        if (xb - xa >= yb - ya) {
            const int m = (xa + xb) / 2;
            return plan_one(nx, ny, s, near, recip, cse, xa, m, ya, yb, out) &&
                   plan_one(nx, ny, s, near, recip, cse, m, xb, ya, yb, out);
        }
        const int m = (ya + yb) / 2;
        return plan_one(nx, ny, s, near, recip, cse, xa, xb, ya, m, out) &&
               plan_one(nx, ny, s, near, recip, cse, xa, xb, m, yb, out);
    }
    out.max_area = std::max(out.max_area, r0.w * r0.h);
    out.max_inputs = std::max(out.max_inputs, tile_input_slots(r0, nx, ny));
    out.max_links = std::max(out.max_links, d.n_links);
    d.link0 = (int)out.links.size();
    d.node0 = (int)out.nodes.size();
    if (d.n_links) {
        out.nodes.resize(out.nodes.size() + (size_t)r0.w * r0.h, 0u);
        int n = 0;
        for (const NearLink &l : near) {
            if (!inside(l)) continue;
            const PlanLink &L = *l.link;
            const bool own = L.x >= xa && L.x < xb && L.y >= ya && L.y < yb;
            TileLink t{};
            t.x = (int16_t)(L.x - r0.x);
            t.y = (int16_t)(L.y - r0.y);
            t.q = (int8_t)L.q;
            t.mode = (int8_t)L.mode;
            t.dslot = own ? L.dslot : -1;
            t.c0 = L.c0;
            t.c1 = L.c1;
            t.c2 = L.c2;
            uint32_t &e = out.nodes[d.node0 + (size_t)t.x * r0.h + t.y];
            if (!(e & 511u)) e = (uint32_t)n << 9;
            e |= 1u << ns[L.q];
            out.links.push_back(t);
            ++n;
        }
    }
    return true;
}

// Tiles of one lattice: the split into at most `most` tiles whose regions r[0]
// are smallest; 0 when none is within `area` nodes.
inline int split_tiles(int nx, int ny, int K, int most, int area, int &ntx, int &nty)
{
    int best = 0;
    for (int b = 1; b <= std::min(most, ny / 2); ++b) {
        const int a = std::min(most / b, nx / 2);
        if (a < 1) break;
        const int w = std::min((nx + a - 1) / a + 2 * K, nx), h = std::min((ny + b - 1) / b + 2 * K, ny);
        if ((int64_t)w * h <= area && (!best || w * h < best)) {
            best = w * h;
            ntx = a;
            nty = b;
        }
    }
    return best;
}

// A work-group shape and the regions it is used for.
struct TileKind {
    int cfg, K, cap, nt;             // launch shape (tile_launch), iterations, nodes, work-items
    int area;                        // regions of at most so many nodes
    int groups;                      // 0: one tile per CU; else as many tiles as it takes
};

// Launch shape of a set of lattices (one, or the cases of a batch).
//
// Small ones take one tile per CU and advance 5-7 iterations per launch: an
// iteration then costs its dependent chain (pulls, barrier, collision,
// barrier: 0.8-1.2 us), not a launch of 7 us.  Larger ones take the shape with
// the most nodes per second, two work-groups per CU, so that one loads or
// stores while the other computes.  The lines below are where the next shape
// became the faster one (MI355X, us per iteration; one iteration per launch in
// brackets):
//   FP64  100^2 K7 512x1 1.64 (7.0), 5 iterations 1.80, 3 1.98;
//         151^2 K7 512x2 1.81, K5 512x1 1.87 (6.9);
//         200^2 K5 512x2 2.03, K7 512x2 2.18, K3 512x1 2.35 (7.0);
//         300^2 K5 512x2 2.66, K7 1024x2 2.69; 400^2 K7 1024x2 3.35, K5 3.35,
//         K5 512x2 3.92 (9.0); 1073x200 (links) K7 1024x2 4.09, K5 4.67;
//         600^2 K3 1024x2 6.45, K3 512x2 8.27; 800^2 K3 512x2 10.3, 1024x2 11.6;
//         8192x2048 K3 512x2 237, K5 512x2 248, K5 1024x2 284, K3 512x1 307 (434)
//   FP32  100^2 K7 512x1 1.26 (9.0); 200^2 K7 1024x2 1.45, 512x2 1.56 (8.9);
//         1073x240 (links) K5 1024x2 3.30, K7 1024x4 3.59; 700^2 K7 1024x4 4.03 (12.7);
//         8192x2048 K5 512x4 101, K7 512x4 106, K5 512x2 114, K3 512x4 116,
//         K5 1024x4 123 (211)
inline const TileKind *tile_kinds(bool f64, int &n)
{
    static const TileKind d[] = {{0, 7, 512, 512, 512, 0},
                                 {1, 7, 1024, 512, 600, 0},
                                 {1, 5, 1024, 512, 1024, 0},
                                 {2, 7, 2048, 1024, 2048, 0},
                                 {2, 5, 2048, 1024, 2048, 0},
                                 {2, 3, 2048, 1024, 2048, 0},
                                 {1, 3, 1024, 512, 1024, 1}};
    static const TileKind f[] = {{0, 7, 512, 512, 512, 0},
                                 {1, 7, 1024, 512, 640, 0},
                                 {2, 7, 2048, 1024, 2048, 0},
                                 {2, 5, 2048, 1024, 2048, 0},
                                 {4, 7, 4096, 1024, 4096, 0},
                                 {3, 5, 2048, 512, 2048, 1}};
    n = f64 ? 7 : 6;
    return f64 ? d : f;
}

// The same for the launches of the channel adjoint (cfg: nodes per work-item,
// the smallest first).  A node's adjoint takes four times the arithmetic of a
// collision: two waves per SIMD in double (up to 256 registers each), four in
// float; regions shrink less per CU, so K 5 rather than 7.  us per iteration,
// recomputation included (one iteration per launch in brackets):
//   FP64  240x64 K7 512x1 6.3, K5 6.4; 384x128 K5 512x2 7.1, K3 512x1 7.4;
//         1024x256 K5 512x4 15.4, K3 512x3 16.0 (33);
//         2048x512 K3 512x4 69, K5 512x4 73, K3 512x3 73
//   FP32  240x64 K7 1024x1 5.3; 384x128 K7 1024x1 5.7, K4 5.8;
//         768x160 K5 1024x1 7.2, K3 7.4; 1024x256 K5 1024x2 10.0, K3 10.8,
//         K3 512x3 11.8 (27); 2048x512 K5 512x3 36.9, K3 1024x2 37.7
inline const TileKind *adjoint_kinds(bool f64, int &n)
{
    static const TileKind d[] = {{0, 7, 512, 512, 512, 0},
                                 {1, 5, 1024, 512, 1024, 0},
                                 {2, 5, 2048, 512, 2048, 0},
                                 {2, 3, 2048, 512, 2048, 1}};
    static const TileKind f[] = {{0, 7, 1024, 1024, 800, 0},
                                 {0, 5, 1024, 1024, 1024, 0},
                                 {1, 5, 2048, 1024, 2048, 0},
                                 {2, 5, 1536, 512, 1536, 1}};
    n = 4;
    return f64 ? d : f;
}

// Builds the plan of one lattice (links sorted by x, y and the direction they
// set); false when it does not fit the shape: a link stencil that leaves the
// lattice (wrapped links), two links that set the same population of a node,
// or tiles of less than two nodes a side.
inline bool plan_tiles(int nx, int ny, const TileShape &s, const std::vector<PlanLink> &links,
                       int cse, TilePlan &out)
{
    if (s.K < 1 || s.K > TILE_MAX_LEVELS || s.ntx < 1 || s.nty < 1 || s.cap > 65536 ||
        nx / s.ntx < 2 || ny / s.nty < 2)
        return false;
    for (size_t k = 1; k < links.size(); ++k)
        if (links[k].x == links[k - 1].x && links[k].y == links[k - 1].y &&
            links[k].q == links[k - 1].q)
            return false;
    const auto tile_of = [](int v, int n, int nt) {  // tile t: [n t / nt, n (t + 1) / nt)
        v = std::min(std::max(v, 0), n - 1);
        return (int)((((int64_t)v + 1) * nt - 1) / n);
    };
    static const int cx[9] = {0, 1, -1, 0, 0, 1, -1, -1, 1};
    static const int cy[9] = {0, 0, 0, 1, -1, 1, -1, 1, -1};
    static const int ns[9] = {0, 2, 1, 4, 3, 6, 5, 8, 7};
    std::vector<NearLink> all;
    all.reserve(links.size());
    for (const PlanLink &L : links) {
        const int far = L.mode == 1 ? 2 : L.mode ? 1 : 0, qb = ns[L.q];
        const int x = L.x + far * cx[qb], y = L.y + far * cy[qb];
        if (x < 0 || x >= nx || y < 0 || y >= ny) return false;
        const NearLink n{L.x, L.y, (int8_t)cx[qb], (int8_t)cy[qb], (int8_t)far, &L};
        all.push_back(n);
    }
    // room at once (fresh pages cost more than what is written to them): a link
    // lies in about two tiles' regions, which hold some 20 nodes per link
    const auto room = [](auto &v, size_t n) {
        if (v.size() + n > v.capacity()) v.reserve(std::max(v.size() + n, 2 * v.capacity()));
    };
    room(out.tiles, (size_t)s.ntx * s.nty);
    room(out.links, 2 * links.size());
    room(out.nodes, 20 * links.size());
    const int margin = 2 * s.K + 2;
    std::vector<std::vector<NearLink>> near(s.nty);  // of a column's tiles, in the links' order
    std::vector<uint32_t> recip(ny + 1, 0u);         // 2^32 / height
    for (int h = 1; h <= ny; ++h) recip[h] = 0xffffffffu / (uint32_t)h + 1u;
    const auto before = [](const NearLink &L, int x) { return L.x < x; };
    for (int tx = 0; tx < s.ntx; ++tx) {
        const int xa = (int)((int64_t)nx * tx / s.ntx), xb = (int)((int64_t)nx * (tx + 1) / s.ntx);
        for (auto &n : near) n.clear();
        for (auto l = std::lower_bound(all.begin(), all.end(), xa - margin, before);
             l != all.end() && l->x < xb + margin; ++l)
            for (int ty = tile_of(l->y - margin, ny, s.nty); ty <= tile_of(l->y + margin, ny, s.nty); ++ty)
                near[ty].push_back(*l);
        for (int ty = 0; ty < s.nty; ++ty) {
            const int ya = (int)((int64_t)ny * ty / s.nty),
                      yb = (int)((int64_t)ny * (ty + 1) / s.nty);
            if (!plan_one(nx, ny, s, near[ty], recip, cse, xa, xb, ya, yb, out)) return false;
        }
    }
    return true;
}

// Bytes of LDS: populations, wall inputs of every iteration, link values.
inline size_t tile_lds(const TileKind &k, bool f64, const TilePlan &plan)
{
    return (f64 ? 8 : 4) *
           ((size_t)9 * k.cap + (size_t)2 * k.K * plan.max_inputs + (size_t)plan.max_links);
}

struct PlanCase {
    int nx, ny;
    const std::vector<PlanLink> *links;
};

// The plan of a set of lattices that share one launch on a GPU of n_cu CUs
// with lds_max bytes of LDS per work-group, in the first of the n shapes that
// fits; null when they have none.
inline const TileKind *plan_cases(const std::vector<PlanCase> &cases, const TileKind *kinds, int n,
                                  bool adjoint, bool f64, int n_cu, size_t lds_max, TilePlan &out)
{
    int64_t total = 0;
    for (const PlanCase &c : cases) total += (int64_t)c.nx * c.ny;
    for (int i = 0; i < n; ++i) {
        const TileKind &k = kinds[i];
        if (!k.groups && (total > (int64_t)n_cu * k.area || (int)cases.size() > n_cu)) continue;
        // square tiles of the largest region, where there may be any number
        int side = 2;
        while ((side + 1 + 2 * k.K) * (side + 1 + 2 * k.K) <= k.area) ++side;
        // one tile per CU: a few less where links split some of them, as one
        // more tile than CUs costs a second round
        for (int slack = 0; slack < (k.groups ? 1 : 4); ++slack) {
            bool ok = true;
            out = TilePlan();
            for (size_t c = 0; ok && c < cases.size(); ++c) {
                const int nx = cases[c].nx, ny = cases[c].ny;
                TileShape s{k.K, 0, 0, k.cap, k.nt, adjoint};
                if (k.groups) {
                    s.ntx = std::max(1, std::min((nx + side - 1) / side, nx / 2));
                    s.nty = std::max(1, std::min((ny + side - 1) / side, ny / 2));
                } else {
                    const int64_t cus = n_cu - (int64_t)n_cu * slack / 24;
                    const int most = (int)std::max<int64_t>(1, cus * nx * ny / total);
                    ok = split_tiles(nx, ny, k.K, most, k.area, s.ntx, s.nty) > 0;
                }
                ok = ok && plan_tiles(nx, ny, s, *cases[c].links, (int)c, out);
            }
            if (ok && tile_lds(k, f64, out) <= lds_max &&
                (k.groups || (int)out.tiles.size() <= n_cu))
                return &k;
        }
    }
    out = TilePlan();
    return nullptr;
}

inline const TileKind *plan_cases(const std::vector<PlanCase> &cases, bool f64, int n_cu,
                                  size_t lds_max, TilePlan &out)
{
    int n = 0;
    const TileKind *kinds = tile_kinds(f64, n);
    return plan_cases(cases, kinds, n, false, f64, n_cu, lds_max, out);
}

}  // namespace lbm
