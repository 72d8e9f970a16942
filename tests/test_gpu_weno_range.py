"""The face reconstruction over the whole range of its data: fields whose differences die out by a factor a
cell (through every magnitude down to zero), steps between constant states (indicators that are exactly
zero), rounding-level differences, huge or tiny units and plateaus between jumps of very different size, where
the WENO weights' products leave the double range and the general form takes over. GPU right-hand side of one
box against the oracle's: everything finite and, per variable, within 1e-12 of max |U| c_max / dx, the size of
the fluxes it differences (the bar of the other right-hand-side tests; rounding differences of a right-hand side
are of the fluxes' size, and some of these right-hand sides are rounding alone)."""
import numpy as np
import pytest

import oracle
from compas_amd import make_geometry, make_params, rhs_box
from compas_amd.cases import np_prim_to_cons, prim_to_cons

pytestmark = pytest.mark.gpu

N = 24
KINDS = ["fringe-3", "fringe-20", "fringe-60", "step", "ramp-end", "noise", "huge", "tiny", "plateau"]


def _field(kind, nphase, rng):
    shape = (N + 6, N + 6)
    j, i = np.meshgrid(np.arange(shape[0]), np.arange(shape[1]), indexing="ij")
    u, v = np.zeros(shape), np.zeros(shape)
    p, a = np.ones(shape), np.full(shape, 1e-8)
    if kind.startswith("fringe"):
        f = 10.0 ** -int(kind.split("-")[1])
        u = 0.3 * f ** i.astype(float) * rng.uniform(0.5, 1.0, shape)
        v = -0.2 * f ** j.astype(float) * rng.uniform(0.5, 1.0, shape)
        p = 1.0 + 0.1 * f ** (i + j).astype(float)
    elif kind == "step":
        p = np.where(i < 14, 2.0, 1.0)
        u = np.where(i < 14, 0.5, 0.0)
        a = np.where(j < 11, 1.0 - 1e-8, 1e-8)
    elif kind == "ramp-end":
        u = np.maximum(0.0, 12.0 - i) * 0.01
        v = np.maximum(0.0, j - 15.0) * 0.01
        a = np.clip((i - 8) * 0.1, 1e-8, 1.0 - 1e-8)
    elif kind == "noise":
        p = 1.0 + 2.2e-16 * rng.integers(0, 3, shape)
        a = a * (1.0 + 2.2e-16 * rng.integers(0, 3, shape))
    elif kind == "plateau":
        # three equal cells between a jump of 1e55 and one of 1e29: the product of their squares overflows on one
        # side of the face in the middle while the other side's sums stay in range
        q = i % 7
        u = np.where(q == 0, 1e55, np.where(q <= 3, 1e30, 1e30 * (1.0 + 0.3 * rng.uniform(size=shape))))
        a = np.full(shape, 0.5)
    else:
        s = 1e30 if kind == "huge" else 1e-30
        p = s * s * (1.0 + 0.3 * rng.uniform(size=shape))
        u, v = s * rng.uniform(-0.3, 0.3, shape), s * rng.uniform(-0.3, 0.3, shape)
        a = rng.uniform(0.1, 0.9, shape)
    rho = 1e-110 if kind == "plateau" else 1.0
    if nphase:
        return np.stack([a * rho, (1 - a) * 0.6 * 0.14 * rho, (1 - a) * 0.4 * 5.0 * rho, u, v, p, a, (1 - a) * 0.6, (1 - a) * 0.4])
    return np.stack([a * rho, (1 - a) * 10.0 * rho, u, v, p, a])


@pytest.mark.parametrize("scheme,nphase", [("WENO5", 0), ("WENO5B", 0), ("WENO5", 3)])
@pytest.mark.parametrize("kind", KINDS)
def test_rhs_over_the_range(gpu, kind, scheme, nphase):
    import torch
    gam = (1.4, 1.67, 1.09) if nphase else (1.4, 1.6)
    P = make_params(2, gamma=gam, scheme=scheme, nphase=nphase)
    G = make_geometry((N, N), (0.0, 0.0), (1.0, 1.0), (0, 0))
    W = _field(kind, nphase, np.random.default_rng(3))
    U = np.ascontiguousarray(np_prim_to_cons(P, W) if nphase else prim_to_cons(P, W))
    box = ([0, 0], [N - 1, N - 1])
    ref, cref = oracle.rhs_box(P, G, box, 3, U)
    dU = torch.zeros(ref.size, dtype=torch.float64, device=gpu)
    cm = torch.zeros(1, dtype=torch.float64, device=gpu)
    rhs_box(P, G, box, 3, torch.from_numpy(U.ravel()).to(gpu), dU, cm)
    torch.cuda.synchronize()
    got = dU.cpu().numpy().reshape(ref.shape)
    assert np.isfinite(ref).all() and np.isfinite(got).all()
    assert abs(cm.item() - cref) <= 1e-14 * cref
    for n in range(P.nstate):
        scale = np.abs(U[n]).max() * cref / G.dx[0]
        if n in range(P.nstate - 1 - (nphase or 1) - 2, P.nstate - 1 - (nphase or 1)):
            scale = max(scale, np.abs(W[P.nstate - 1 - (nphase or 1)]).max() / G.dx[0])   # momentum: p / dx
        assert np.abs(got[n] - ref[n]).max() <= 1e-12 * scale, (n, np.abs(got[n] - ref[n]).max() / scale)
