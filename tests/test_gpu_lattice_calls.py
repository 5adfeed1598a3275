"""Call-by-call use of the lattice while the stream is busy: a wall call has
taken its inputs when it returns, so arrays that the caller overwrites next
give the fields of arrays that are left alone, bit for bit (below and above
the sizes at which the runtime changes how it copies host memory)."""
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fields(nx, ny, overwrite, tmp_path):
    import torch
    from lbm_amd.lattice import lattice
    lat = lattice(types.SimpleNamespace(nx=nx, ny=ny, tau_lbm=0.6, IBB=True, verbose=False,
                                        results_dir=str(tmp_path) + "/"))
    rng = np.random.default_rng(1)
    lat.device_fields()["g"].copy_(torch.from_numpy(rng.uniform(0.1, 0.2, (9, nx, ny))))
    big = torch.ones(4096, 4096, device="cuda")
    for _ in range(3):
        lat.u_bot, lat.u_top = (rng.uniform(-0.05, 0.05, (2, nx)) for _ in range(2))
        lat.u_left, lat.u_right = (rng.uniform(-0.05, 0.05, (2, ny)) for _ in range(2))
        lat.rho_right = rng.uniform(0.9, 1.1, ny)
        lat.macro()
        lat.equilibrium()
        for _ in range(4):
            big = big @ big * 1e-4               # the calls below queue behind it
        lat.collision_stream()
        for call, used in ((lat.zou_he_bottom_wall_velocity, (lat.u_bot,)),
                           (lat.zou_he_left_wall_velocity, (lat.u_left,)),
                           (lat.zou_he_top_wall_velocity, (lat.u_top,)),
                           (lat.zou_he_right_wall_pressure, (lat.u_right, lat.rho_right))):
            call()
            for a in used:
                if overwrite:
                    a[...] = np.nan
        lat.zou_he_bottom_left_corner()
        lat.zou_he_top_left_corner()
        lat.zou_he_top_right_corner()
        lat.zou_he_bottom_right_corner()
    return {k: v.cpu().numpy() for k, v in lat.device_fields().items()}


@pytest.mark.parametrize("nx,ny", [(5, 4), (1073, 200), (9, 40001)])
def test_wall_inputs_may_be_overwritten(nx, ny, tmp_path):
    a, b = (_fields(nx, ny, o, tmp_path) for o in (False, True))
    for k in a:
        assert np.isfinite(a[k]).all() and np.array_equal(a[k], b[k]), k
