"""The multigrid preconditioner of the implicit Grad_Q at the sizes where its one-workgroup coarse end changes
form: the largest first grid it takes (4096 cells), one past it, a single grid (odd extents), a second grid of
1023 cells, grids of at most one wave from the start, flat and long grids, both kinds of sides. Grad_Q against
the oracle's Jacobi-preconditioned solve, both run to the rounding floor: max |gpu - cpu| <= 1e-9 max |cpu| (the
bar of the other implicit solves), and an iteration count that only a working V-cycle reaches."""
import numpy as np
import pytest

import oracle
from compas_amd import FaceLayout, Layout, Level, make_geometry, make_params, make_pf_params
from compas_amd.cases import prim_to_cons

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("n", [(64, 64), (68, 64), (62, 66), (25, 31), (6, 10), (16, 4), (128, 32), (256, 128),
                               (16, 16, 16), (18, 16, 16), (12, 20, 4), (7, 9, 5), (4, 4, 4), (32, 16, 8)])
def test_gradq_at_the_edges_of_the_tail(gpu, n, periodic):
    import torch
    dim = len(n)
    P = make_params(dim, gamma=(1.4, 1.6))
    G = make_geometry(n, (0.0,) * dim, tuple(e / 32.0 for e in n), (periodic,) * dim)
    x = np.meshgrid(*[(np.arange(e) + 0.5) / e for e in reversed(n)], indexing="ij")
    d = np.sqrt(sum((q - 0.5) ** 2 for q in x)) - 0.27
    a = np.clip(0.5 - 0.5 * np.tanh(0.5 * min(n) * d), 1e-8, 1 - 1e-8)
    one = np.ones_like(a)
    W = np.stack([a, 0.2 * (1 - a), 0.3 * one] + [0.1 * np.cos(2 * np.pi * x[-2])] * (dim - 1) + [one, a])
    box = ([0] * dim, [e - 1 for e in n])
    lay, flay = Layout(dim, [box], 3, P.nstate), FaceLayout(dim, [box])
    buf = lay.pack(np.ascontiguousarray(prim_to_cons(P, W)))
    pf = make_pf_params(mechanism="CAC-Adv", explicit_rc=0, eta_multiplier=0.5)
    ref, _, _ = oracle.level_pf_gradq_step(P, pf, G, lay, buf, 0.01, flay.total)
    lev = Level(P, G, lay)
    lev.pf_setup(pf)
    gq = torch.full((flay.total,), float("nan"), dtype=torch.float64, device=gpu)
    lev.PhaseField_GradQPF(torch.from_numpy(buf).to(gpu), 0.01, gq)
    assert lev.check_errors() == 0
    it, got = lev.solver_iterations(), gq.cpu().numpy()
    lev.close()
    print(n, periodic, "iterations", it, flush=True)
    assert np.isfinite(got).all()
    assert np.max(np.abs(got - ref)) <= 1e-9 * np.max(np.abs(ref))
    assert it <= 60
