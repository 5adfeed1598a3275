"""Several iterations per launch (lbm_amd/csrc/d2q9_tile.hip) against one per
launch: lbm_steps must leave, bit for bit, the
state, fields and drag sums of the one-iteration kernels (lbm_step, which the
other GPU tests compare with the oracle), for every storage form, at
the smallest lattices, at the edges of the launch shapes, with links near
walls, for every remainder of iterations, and with the state of the last
iteration but one still readable."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = np.array([4. / 9.] + [1. / 9.] * 4 + [1. / 36.] * 4)


def _square_links(nx, ny, squares, seed):
    """IBB and plain links of solid squares (x0, y0, side), as one obstacle
    each; stencils that leave the lattice are left out."""
    from lbm_amd.geometry import C, NS
    rng = np.random.default_rng(seed)
    out = []
    for x0, y0, side in squares:
        links = []
        for x in range(x0, x0 + side):
            for y in range(y0, y0 + side):
                for q in range(1, 9):
                    i, j = x - C[q, 0], y - C[q, 1]
                    gi, gj = i - 2 * C[q, 0], j - 2 * C[q, 1]
                    if x0 <= i < x0 + side and y0 <= j < y0 + side:
                        continue
                    if 0 <= i < nx and 0 <= j < ny and 0 <= gi < nx and 0 <= gj < ny:
                        links.append((i, j, q))
        links = np.unique(np.array(links, dtype=np.int64), axis=0)
        assert (NS[NS[links[:, 2]]] == links[:, 2]).all()
        out.append((links, rng.uniform(0.05, 0.95, len(links))))
    return out


def _run(nx, ny, storage, n, squares=(), pressure=True, pool=False, ring=None, single=False,
         replays=1, ibb=True):
    import torch
    from lbm_amd import _lib
    from lbm_amd.domain import FusedDomain, q16_range
    ring = ring or n + 2
    rng = np.random.default_rng(nx * 1000 + ny)
    g0 = W[:, None, None] * (1.0 + 0.01 * rng.standard_normal((9, nx, ny)))
    g0 = torch.from_numpy(np.ascontiguousarray(g0)).cuda()
    bc = [_lib.BC_VELOCITY] * 3 + [_lib.BC_PRESSURE if pressure else _lib.BC_VELOCITY]
    dom = FusedDomain(nx, ny, 1 / 0.62, 1 / (0.25 / 0.12 + 0.5), bc,
                      _square_links(nx, ny, squares, 3), ibb=ibb, storage=storage, ring=ring,
                      q16_range=q16_range(0.1) if storage == "q16" else None)
    prof = [0.02 * rng.standard_normal(s) for s in ((2, nx), (2, ny), (2, nx), (2, ny))]
    prof.append(1.0 + 0.01 * rng.standard_normal(ny))
    amp = rng.uniform(0.5, 1.0, (ring, 5))
    if pool:
        rows = [tuple(a[k] * prof[k] for k in range(5)) for a in amp]
        dom.set_inlet_rows(0, rows)
    else:
        dom.set_profiles(prof)
        dom.set_amplitudes(0, amp)
    out = []
    for _ in range(replays):
        dom.init(g0)
        if single:
            for it in range(1, n + 1):
                dom.step(it)
        else:
            dom.steps(1, n)
        g, g_up = torch.empty_like(g0), torch.empty_like(g0)
        rho = torch.zeros((nx, ny), dtype=torch.float64, device="cuda")
        u = torch.zeros((2, nx, ny), dtype=torch.float64, device="cuda")
        res = dict(mass=dom.mass(n), before=dom.mass(n - 1))
        if squares:
            dom.drag_only(n)
            m = min(n + 1, ring)
            res["drag"] = dom.drag_read(n + 1 - m, m)
        dom.epilogue(n, g, g_up, rho, u)
        res.update(g=g.cpu().numpy(), g_up=g_up.cpu().numpy(), rho=rho.cpu().numpy(),
                   u=u.cpu().numpy())
        out.append(res)
    dom.close()
    return out


def _same(a, b, what):
    for k in a:
        assert np.array_equal(a[k], b[k], equal_nan=True), \
            (what, k, float(np.nanmax(np.abs(np.asarray(a[k]) - np.asarray(b[k])))))


# smallest lattices; a tile per CU of 2 to 40 nodes a side; several tiles per
# CU; obstacles beside a corner, on a wall, across tile edges
SIZES = [(4, 4, ()), (5, 9, ()), (9, 5, ()), (33, 64, ((14, 20, 5),)), (47, 31, ((3, 3, 4), (30, 26, 5))),
         (130, 101, ((60, 40, 17), (2, 50, 6), (100, 95, 6))), (401, 53, ((30, 20, 9),)),
         (520, 260, ((100, 100, 40), (300, 30, 33), (480, 200, 12)))]


@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "bf16", "f16e", "f16e8", "q16"])
@pytest.mark.parametrize("nx,ny,squares", SIZES)
def test_steps_equal_one_iteration_kernels(nx, ny, squares, storage):
    n = 16
    _same(_run(nx, ny, storage, n, squares)[0], _run(nx, ny, storage, n, squares, single=True)[0],
          (nx, ny, storage))


@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_several_tiles_per_cu(storage):
    nx, ny = (701, 610) if storage == "f64" else (1301, 1100)
    squares = ((3, 300, 30), (350, 200, 90), (600, 570, 40))
    _same(_run(nx, ny, storage, 9, squares)[0], _run(nx, ny, storage, 9, squares, single=True)[0], storage)


@pytest.mark.parametrize("storage,nx,ny", [("f64", 530, 519), ("f32", 530, 519), ("f64", 601, 600)])
def test_largest_single_round(storage, nx, ny):
    """Lattices whose largest regions just fit a work-group: fewer iterations."""
    squares = ((3, 300, 30), (250, 200, 60), (480, 470, 40))
    _same(_run(nx, ny, storage, 11, squares)[0], _run(nx, ny, storage, 11, squares, single=True)[0],
          (nx, ny, storage))


@pytest.mark.parametrize("nx,ny", [(1999, 1000), (2003, 1000)])
def test_q16_either_side_of_one_iteration_launches(nx, ny):
    squares = ((3, 300, 30), (900, 200, 90), (1900, 900, 40))
    _same(_run(nx, ny, "q16", 9, squares)[0], _run(nx, ny, "q16", 9, squares, single=True)[0], nx)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 15])
def test_every_remainder(n):
    kw = dict(squares=((10, 12, 6),), pressure=False, pool=True)
    _same(_run(61, 40, "f64", n, **kw)[0], _run(61, 40, "f64", n, single=True, **kw)[0], n)


def test_short_ring_plain_links_and_replays():
    """A ring shorter than a launch, plain bounce-back, replays of one graph."""
    kw = dict(squares=((10, 12, 6),), ring=3, ibb=False, replays=3)
    a, b = _run(80, 45, "f64", 20, **kw), _run(80, 45, "f64", 20, single=True, **kw)
    for x in a:
        _same(x, b[0], "replay")


@pytest.mark.parametrize("storage", ["f64", "f32", "f16e8"])
def test_batch_equals_one_iteration_kernels(storage):
    import torch
    from lbm_amd.batch import Batch, cavity_amplitudes, cavity_ensemble
    cases = cavity_ensemble(5, seed=2, n_lo=9, n_hi=130)
    for c in cases:
        c["sigma"] = 10
    links, p = _square_links(cases[1]["nx"], cases[1]["ny"], ((4, 4, 3),), 1)[0]
    cases[1].update(links=links, ibb=p, ibb_on=np.ones(len(links), np.uint8))
    n = 18
    res = []
    for single in (False, True):
        b = Batch(cases, storage=storage, ring=n + 2)
        b.set_amplitudes(0, cavity_amplitudes(cases, 0, n + 1))
        b.init()
        if single:
            for it in range(1, n + 1):
                b.steps(it, 1)
        else:
            b.steps(1, n)
        out = []
        for k, c in enumerate(cases):
            d = b.case(k)
            g = torch.empty((9, c["nx"], c["ny"]), dtype=torch.float64, device="cuda")
            g_up = torch.empty_like(g)
            d.epilogue(n, g, g_up)
            r = dict(g=g.cpu().numpy(), g_up=g_up.cpu().numpy())
            if d.n_obs:
                r["drag"] = d.drag_read(0, n)
            out.append(r)
        res.append(out)
        b.close()
    for k, (x, y) in enumerate(zip(*res)):
        _same(x, y, (storage, k))
