// Host check of the tile plans (lbm_amd/csrc/d2q9_plan.h; test infrastructure,
// built by tests/test_tile_plan.py).  For lattices of all sizes, with and
// without links near walls, corners and tile edges, every launch shape: the
// owned rectangles cover each node once; every level's reads (pulls, link
// stencils, the wall node beside a corner) lie in the level before; a tile
// holds its links once, in the order of its node table; every perimeter slot
// maps to one node of the region; limits hold.  Exit status 0 with "ok".
#include "../lbm_amd/csrc/d2q9_plan.h"

#include <cstdio>
#include <cstdlib>
#include <random>

using namespace lbm;

static const int CX[9] = {0, 1, -1, 0, 0, 1, -1, -1, 1}, CY[9] = {0, 0, 0, 1, -1, 1, -1, 1, -1};
static const int NS[9] = {0, 2, 1, 4, 3, 6, 5, 8, 7};
static long checks = 0;

#define REQUIRE(c)                                                              \
    do {                                                                        \
        ++checks;                                                               \
        if (!(c)) {                                                             \
            std::printf("%s (line %d): %d x %d, K %d, %zu links\n", #c, __LINE__, nx, ny, K, \
                        links.size());                                          \
            std::exit(1);                                                       \
        }                                                                       \
    } while (0)

static bool in(const TileRect &r, int x, int y)
{
    return x >= r.x && x < r.x + r.w && y >= r.y && y < r.y + r.h;
}

static void check(int nx, int ny, int K, int cap, int nt, const std::vector<PlanLink> &links,
                  const TilePlan &plan)
{
    std::vector<int> owner((size_t)nx * ny, 0), slots(links.size(), 0);
    for (const TileDesc &d : plan.tiles) {
        const TileRect &o = d.r[K];
        for (int x = o.x; x < o.x + o.w; ++x)
            for (int y = o.y; y < o.y + o.h; ++y) ++owner[(size_t)x * ny + y];
        REQUIRE(d.r[0].w * d.r[0].h <= cap && d.n_links <= nt);
        REQUIRE(d.r[0].x >= 0 && d.r[0].y >= 0 && d.r[0].x + d.r[0].w <= nx &&
                d.r[0].y + d.r[0].h <= ny);
        for (int l = K; l >= 1; --l) {
            const TileRect &r = d.r[l], &q = d.r[l - 1];
            for (int x : {r.x, r.x + r.w - 1})
                for (int y : {r.y, r.y + r.h - 1}) {
                    REQUIRE(in(q, x, y));
                    for (int k = 1; k < 9; ++k) {
                        const int sx = x - CX[k], sy = y - CY[k];
                        if (sx >= 0 && sx < nx && sy >= 0 && sy < ny) REQUIRE(in(q, sx, sy));
                    }
                }
            // the wall node beside a corner, its pulls and its links
            for (int x : {0, nx - 1})
                for (int y : {0, ny - 1})
                    if (in(r, x, y)) {
                        const int xn = x == 0 ? 1 : nx - 2;
                        REQUIRE(in(r, xn, y));
                        for (int k = 0; k < 9; ++k) {
                            const int sx = xn - CX[k], sy = y - CY[k];
                            if (sx >= 0 && sx < nx && sy >= 0 && sy < ny) REQUIRE(in(q, sx, sy));
                        }
                    }
            for (const PlanLink &L : links)
                if (L.mode && in(r, L.x, L.y)) {
                    const int far = L.mode == 1 ? 2 : 1, qb = NS[L.q];
                    REQUIRE(in(q, L.x + far * CX[qb], L.y + far * CY[qb]));
                }
            // n / height by the stored reciprocals
            const int hi = r.h - (r.y == 0) - (r.y + r.h == ny);
            for (int n : {0, 1, r.h - 1, r.h, cap - 1}) {
                REQUIRE((int)(((uint64_t)n * d.mh[l]) >> 32) == (r.h == 1 ? 0 : n / r.h) ||
                        r.h == 1);
                if (hi > 1) REQUIRE((int)(((uint64_t)n * d.mi[l]) >> 32) == n / hi);
            }
            // work-item slots
            const TilePerim P = tile_perim(r, nx, ny);
            REQUIRE(P.slots <= nt && P.slots + P.inner <= cap);
            std::vector<int> seen((size_t)r.w * r.h, 0);
            int count = 0;
            for (int n = 0; n < P.slots; ++n) {
                int x, y, t;
                if (!tile_perim_node(r, P, n, x, y, t)) continue;
                REQUIRE(in(r, x, y) && !seen[(size_t)(x - r.x) * r.h + y - r.y]++);
                const bool xe = x == 0 || x == nx - 1, ye = y == 0 || y == ny - 1;
                REQUIRE(t == (xe && ye   ? NODE_CORNER
                              : y == 0   ? NODE_BOTTOM
                              : ye       ? NODE_TOP
                              : x == 0   ? NODE_LEFT
                              : xe       ? NODE_RIGHT
                                         : NODE_INNER));
                ++count;
            }
            REQUIRE(count + P.inner == r.w * r.h);
        }
        int n = 0;
        for (const PlanLink &L : links) {
            if (!in(d.r[1], L.x, L.y)) continue;
            const TileLink &t = plan.links[d.link0 + n];
            REQUIRE(t.x == L.x - d.r[0].x && t.y == L.y - d.r[0].y && t.q == L.q);
            REQUIRE((t.dslot >= 0) == in(o, L.x, L.y));
            if (t.dslot >= 0) ++slots[t.dslot];
            const uint32_t e = plan.nodes[d.node0 + (size_t)t.x * d.r[0].h + t.y];
            int before = 0;
            for (int b = 1; b < NS[L.q]; ++b) before += (e >> b) & 1;
            REQUIRE(((e >> NS[L.q]) & 1) && (int)(e >> 9) + before == n);
            ++n;
        }
        REQUIRE(n == d.n_links);
    }
    for (int c : owner) REQUIRE(c == 1);
    for (int c : slots) REQUIRE(c == 1);
}

// Adjoint plans: a node's entry at a level comes from its neighbours at the
// level before, the corner's from the wall node beside it.
static void check_adjoint(int nx, int ny, int K, int cap, int nt, const TilePlan &plan)
{
    const std::vector<PlanLink> links;
    std::vector<int> owner((size_t)nx * ny, 0);
    for (const TileDesc &d : plan.tiles) {
        const TileRect &o = d.r[K], &r0 = d.r[0];
        for (int x = o.x; x < o.x + o.w; ++x)
            for (int y = o.y; y < o.y + o.h; ++y) ++owner[(size_t)x * ny + y];
        REQUIRE(r0.w * r0.h <= cap && r0.x >= 0 && r0.y >= 0 && r0.x + r0.w <= nx &&
                r0.y + r0.h <= ny);
        for (int l = K; l >= 1; --l) {
            const TileRect &r = d.r[l], &q = d.r[l - 1];
            for (int x = r.x; x < r.x + r.w; ++x)
                for (int y = r.y; y < r.y + r.h; ++y)
                    for (int k = 0; k < 9; ++k) {
                        const int tx = x + CX[k], ty = y + CY[k];
                        if (tx >= 0 && tx < nx && ty >= 0 && ty < ny) REQUIRE(in(q, tx, ty));
                    }
            for (int y : {0, ny - 1}) {
                if (in(q, 1, y)) REQUIRE(in(q, 0, y));
                if (in(q, nx - 2, y)) REQUIRE(in(q, nx - 1, y));
            }
        }
        // launches of fewer levels start at r[1], r[2], ..
        for (int l = 0; l < K; ++l) {
            const TileRect &r = d.r[l];
            const TilePerim P = tile_perim(r, nx, ny);
            REQUIRE(P.slots <= nt && P.slots + P.inner <= cap);
            const int hi = r.h - (r.y == 0) - (r.y + r.h == ny);
            if (hi > 1)
                for (int n : {0, hi - 1, hi, P.inner - 1})
                    if (n >= 0) REQUIRE((int)(((uint64_t)n * d.mi[l]) >> 32) == n / hi);
        }
    }
    for (int c : owner) REQUIRE(c == 1);
}

static void adjoint_plans()
{
    const int sizes[][2] = {{4, 4},     {4, 5},     {5, 9},    {33, 7},   {7, 900},   {64, 32},
                            {150, 130}, {240, 230}, {500, 260}, {760, 440}, {1024, 256}, {4, 20000}};
    const std::vector<PlanLink> links;
    for (auto &sz : sizes)
        for (int f64 = 0; f64 < 2; ++f64) {
            const int nx = sz[0], ny = sz[1];
            int n = 0, K = 0;
            const TileKind *kinds = adjoint_kinds(f64, n);
            for (int i = 0; i < n; ++i) {            // each shape by itself, then the rule
                TilePlan plan;
                const TileKind *k = plan_cases({{nx, ny, &links}}, kinds + i, 1, true, f64, 256,
                                               162816, plan);
                K = kinds[i].K;
                REQUIRE(k || !kinds[i].groups);
                if (k) check_adjoint(nx, ny, K, k->cap, k->nt, plan);
            }
            TilePlan plan;
            const TileKind *k = plan_cases({{nx, ny, &links}}, kinds, n, true, f64, 256, 162816, plan);
            REQUIRE(k);
            check_adjoint(nx, ny, k->K, k->cap, k->nt, plan);
        }
}

int main()
{
    adjoint_plans();
    std::mt19937 rng(7);
    const int sizes[][2] = {{4, 4},    {5, 4},    {4, 9},    {13, 200}, {64, 64},  {97, 33},
                            {100, 100}, {151, 149}, {256, 40}, {301, 299}, {541, 101}, {700, 650}};
    for (auto &sz : sizes) {
        const int nx = sz[0], ny = sz[1];
        for (int with = 0; with < 3; ++with) {
            std::vector<PlanLink> links;
            // square obstacles: at a corner, across the middle, somewhere
            for (int b = 0; with && b < (with == 1 ? 1 : 6); ++b) {
                const int side = 2 + (int)(rng() % std::max(1, std::min(nx, ny) / 6));
                const int x0 = b == 0 ? 3 : (int)(rng() % nx), y0 = b == 0 ? 3 : (int)(rng() % ny);
                for (int x = x0; x < x0 + side; ++x)
                    for (int y = y0; y < y0 + side; ++y)
                        for (int q = 1; q < 9; ++q) {
                            const int fx = x - CX[q], fy = y - CY[q];
                            const int mode = (int)(rng() % 3), far = mode == 1 ? 2 : mode == 2 ? 1 : 0;
                            const int gx = fx - far * CX[q], gy = fy - far * CY[q];
                            if (fx >= x0 && fx < x0 + side && fy >= y0 && fy < y0 + side) continue;
                            if (fx < 0 || fy < 0 || fx >= nx || fy >= ny || gx < 0 || gy < 0 ||
                                gx >= nx || gy >= ny)
                                continue;
                            links.push_back(PlanLink{fx, fy, q, mode, 0, 1, 0, 0});
                        }
            }
            std::stable_sort(links.begin(), links.end(), [](const PlanLink &a, const PlanLink &b) {
                return a.x != b.x ? a.x < b.x : a.y != b.y ? a.y < b.y : NS[a.q] < NS[b.q];
            });
            links.erase(std::unique(links.begin(), links.end(),
                                    [](const PlanLink &a, const PlanLink &b) {
                                        return a.x == b.x && a.y == b.y && a.q == b.q;
                                    }),
                        links.end());
            for (size_t k = 0; k < links.size(); ++k) links[k].dslot = (int)k;
            for (int f64 = 0; f64 < 2; ++f64) {
                int n = 0;
                const TileKind *kinds = tile_kinds(f64, n);
                for (int i = 0; i < n; ++i) {
                    const int K = kinds[i].K;
                    TileShape s{K, 1, 1, kinds[i].cap, kinds[i].nt};
                    if (!split_tiles(nx, ny, K, 256, kinds[i].area, s.ntx, s.nty)) continue;
                    TilePlan plan;
                    if (plan_tiles(nx, ny, s, links, 0, plan))
                        check(nx, ny, K, s.cap, s.nt, links, plan);
                    else
                        REQUIRE(with);       // a stencil or a split can refuse, an empty lattice not
                }
                // the chosen plan, alone and with a second lattice
                for (int cases = 1; cases <= 2; ++cases) {
                    const std::vector<PlanLink> none;
                    std::vector<PlanCase> pc{{nx, ny, &links}};
                    if (cases == 2) pc.push_back({33, 47, &none});
                    TilePlan plan;
                    const TileKind *k = plan_cases(pc, f64, 256, 163840, plan);
                    const int K = k ? k->K : 0;
                    REQUIRE(k || with);
                    if (!k) continue;
                    REQUIRE(tile_lds(*k, f64, plan) <= 163840);
                    TilePlan own = plan;
                    own.tiles.clear();
                    for (const TileDesc &d : plan.tiles)
                        if (d.cse == 0) own.tiles.push_back(d);
                    check(nx, ny, K, k->cap, k->nt, links, own);
                }
            }
            // what a plan must refuse: a stencil beyond the lattice, two links
            // on one population
            const int K = 3;
            TilePlan plan;
            REQUIRE(!plan_tiles(nx, ny, TileShape{K, 1, 1, 65536, 1024},
                                {PlanLink{0, 1, 1, 1, 0, 1, 0, 0}}, 0, plan));
            REQUIRE(!plan_tiles(nx, ny, TileShape{K, 1, 1, 65536, 1024},
                                {PlanLink{1, 1, 3, 0, 0, 1, 0, 0}, PlanLink{1, 1, 3, 0, 1, 1, 0, 0}},
                                0, plan));
        }
    }
    std::printf("ok %ld\n", checks);
    return 0;
}
