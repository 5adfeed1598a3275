"""The adjoint's launches of several iterations (lbm_pbb_*) where their tiles
have edges: lattices of 4 nodes a side, one row of tiles, odd sizes, each
launch shape and the several-rounds one, iteration counts and checkpoint
intervals that no launch divides, solid fractions on walls and corners too.
Against torch autograd of the FP64 restatement (tests/pbb_reference.py) with
the bounds of its other comparisons: FP64 1e-12 of the loss and 1e-9 of the
largest gradient, FP32 1e-5 and 1e-4 (relative L2)."""
import numpy as np
import pytest
import torch

from lbm_amd.adjoint import PbbEngine, cylinder_case
from tests import pbb_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,iterations,every", [
    (4, 4, 9, 3), (4, 37, 8, 8), (41, 4, 7, 5), (5, 9, 15, 4), (33, 7, 13, 20), (150, 130, 9, 1),
    (240, 230, 8, 6), (500, 260, 12, 7), (760, 440, 6, 4)])
def test_gradients_at_tile_edges(nx, ny, iterations, every, storage):
    d = max(2.0, ny / 6)
    case = cylinder_case(nx=nx, ny=ny, diameter=d, cx=nx / 3, cy=ny / 2, box=2, seed=0, u_max=0.05,
                         Re=20.0, iterations=iterations, window=iterations - 2, every=every,
                         sigma=3.0)
    case["s"] = np.random.default_rng(nx + ny).uniform(0.0, 0.3, (nx, ny)).astype(np.float32)
    s = torch.tensor(case["s"], dtype=torch.float64, requires_grad=True)
    um = torch.tensor(case["u_max"], dtype=torch.float64, requires_grad=True)
    loss, _, final = pbb_reference.run(case, s, um)
    loss.backward()
    eng = PbbEngine(case, storage=storage)
    dt = torch.float64 if storage == "f64" else torch.float32
    got = eng.forward(torch.tensor(case["s"], dtype=dt, device="cuda"), case["u_max"])
    gs, gu = eng.backward()
    gs, state = gs.cpu().numpy(), eng.final_state().double().cpu().numpy()
    eng.close()
    ref, want, wu = s.grad.numpy(), float(loss.detach()), float(um.grad)
    assert np.abs(ref).max() > 0
    if storage == "f64":
        assert abs(got - want) <= 1e-12 * abs(want)
        assert np.abs(state - final.detach().numpy()).max() <= 1e-12
        assert np.abs(gs - ref).max() <= 1e-9 * np.abs(ref).max()
        assert abs(gu - wu) <= 1e-9 * abs(wu)
    else:
        assert abs(got - want) <= 1e-5 * abs(want)
        assert np.linalg.norm(gs - ref) <= 1e-4 * np.linalg.norm(ref)
        assert abs(gu - wu) <= 1e-4 * abs(wu)
