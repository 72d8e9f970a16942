"""The stage kernel at the edges of its tiles (16 x 15 cells in 2D, 8 x 8 x 3 in 3D): boxes of one cell, of
one tile, of a tile more or less a cell and of several tiles with a remainder, every scheme, with and without
THINC where it is supported, with and without face fluxes written. The right-hand side against the oracle's, per variable within
1e-12 of max |U| c_max / dx, the size of the fluxes it differences."""
import numpy as np
import pytest

import oracle
from compas_amd import make_geometry, make_params, rhs_box
from compas_amd.cases import prim_to_cons

pytestmark = pytest.mark.gpu

BOXES = [(1, 1), (16, 15), (17, 14), (15, 16), (1, 46), (33, 2), (47, 31),
         (1, 1, 1), (8, 8, 3), (9, 7, 4), (7, 9, 2), (1, 17, 7), (16, 2, 5), (25, 9, 1)]


@pytest.mark.parametrize("scheme,thinc", [("GODUNOV", 0), ("MUSCL", 0), ("WENO5", 0), ("WENO5", 1),
                                          ("WENO5B", 0), ("WENO5B", 1)])
@pytest.mark.parametrize("n", BOXES)
def test_tile_edges(gpu, n, scheme, thinc):
    import torch
    dim = len(n)
    P = make_params(dim, gamma=(1.4, 1.6), scheme=scheme, thinc=thinc)
    G = make_geometry(n, (0.0,) * dim, tuple(0.1 * e for e in n), (0,) * dim)
    ng = 4 if scheme == "WENO5B" else 3
    rng = np.random.default_rng(7)
    shape = tuple(e + 2 * ng for e in reversed(n))
    x = np.meshgrid(*[np.arange(s) for s in shape], indexing="ij")
    a = 0.5 + 0.5 * (1 - 2e-8) * np.tanh(0.7 * (x[-1] + 0.6 * x[-2] - 9.3)) * np.cos(0.4 * x[0])
    W = np.stack([a * rng.uniform(0.8, 1.2, shape), (1 - a) * rng.uniform(4.0, 5.0, shape)]
                 + [rng.uniform(-0.4, 0.4, shape) for _ in range(dim)] + [rng.uniform(0.8, 1.3, shape), a])
    U = np.ascontiguousarray(prim_to_cons(P, W))
    box = ([0] * dim, [e - 1 for e in n])
    ref, cref = oracle.rhs_box(P, G, box, ng, U)
    Ud = torch.from_numpy(U.ravel()).to(gpu)
    faces = [int(np.prod([e + (d == q) for q, e in enumerate(n)])) for d in range(dim)]
    for write in (False, True):
        dU = torch.zeros(ref.size, dtype=torch.float64, device=gpu)
        cm = torch.zeros(1, dtype=torch.float64, device=gpu)
        fl = [torch.zeros(f * P.nstate, dtype=torch.float64, device=gpu) if write else None for f in faces]
        rhs_box(P, G, box, ng, Ud, dU, cm, (fl + [None])[:3])
        torch.cuda.synchronize()
        got = dU.cpu().numpy().reshape(ref.shape)
        assert np.isfinite(ref).all() and np.isfinite(got).all()
        assert abs(cm.item() - cref) <= 1e-14 * cref
        for v in range(P.nstate):
            scale = max(np.abs(U[v]).max(), 1.3 / cref) * cref / 0.1      # (momentum fluxes: the pressure)
            assert np.abs(got[v] - ref[v]).max() <= 1e-12 * scale, (write, v, np.abs(got[v] - ref[v]).max() / scale)


@pytest.mark.parametrize("n", [(768, 480), (784, 480), (1000, 400)])
def test_weno5b_thinc_on_both_sides_of_its_workgroup_rules(gpu, n):
    """WENO5B with THINC in 2D: 1536 tiles (the last of the two-wave build), 1568 and 1701 tiles, and face blocks
    below (1442, 1470) and above (1564) the face kernel's bound."""
    test_tile_edges(gpu, n, "WENO5B", 1)
