"""Row walk of the pair kernel at its edges: particle counts and rows that are no multiple of an
iteration, empty and short rows, waves near and far from the periodic faces, every lane count."""
import math

import numpy as np
import pytest

import oracle
import pdx
from pdx import systems

pytestmark = pytest.mark.gpu


def _cloud(n, L, seed, dmin=0.85):
    """n random points of a box of side L, no two closer than dmin."""
    rng = np.random.default_rng(seed)
    pts = np.empty((0, 3))
    while len(pts) < n:
        p = rng.random(3) * L - L / 2
        d = pts - p
        d -= L * np.round(d / L)
        if len(pts) == 0 or (d * d).sum(1).min() > dmin * dmin:
            pts = np.vstack([pts, p])
    return pts.astype(np.float32)


# (particles, box side): a gas whose rows hold 0 to a few entries, a ragged liquid, and a box wide
# enough (side > 2 (cutoff + 2 skin)) for waves that skip the seam test
@pytest.mark.parametrize("n,L", [(1, 9.0), (67, 12.0), (341, 9.5), (1029, 13.7)])
@pytest.mark.parametrize("lanes", [0, 1, 2, 4, 16, 64])
def test_rows_at_their_edges(cuda, n, L, lanes):
    import torch
    P = _cloud(n, L, seed=n)
    X, Y, Z = (torch.from_numpy(np.ascontiguousarray(P[:, d])).cuda() for d in range(3))
    ws = pdx.DeviceNeighborWorkspace(n, (L,) * 3, 2.5, 0.4, 128)
    ws.update(X, Y, Z)
    pf = pdx.PairForce(pdx.LennardJones(), lanes=lanes)
    f = [torch.full((n,), 7.0, device="cuda") for _ in range(4)]
    V = torch.full((6, n), 7.0, device="cuda")
    tot = torch.zeros(7, dtype=torch.float64, device="cuda")
    pf.compute(ws, *f, V, tot, energy=True)
    g = [torch.full((n,), 7.0, device="cuda") for _ in range(3)]
    pf.compute(ws, *g, energy=False)
    ws.status()
    ref = oracle.pair_direct(P[:, 0], P[:, 1], P[:, 2], (L,) * 3, kind="lj", cutoff=2.5)
    scale = max(math.sqrt((ref["F"] ** 2).mean()), 1e-30)
    # FP32 positions and sums of at most ~90 terms, each within a few ulps of terms up to ~30 times the
    # net force: 90 * 4 * 6e-8 * 30 = 6.5e-4 at the worst particle, its square root of that in the mean
    for F in (f[:3], g):
        d = torch.stack(F, 1).double().cpu().numpy() - ref["F"]
        assert np.abs(d).max() <= 6.5e-4 * max(scale, np.abs(ref["F"]).max())
        assert math.sqrt((d ** 2).mean()) <= 2e-5 * scale
    E = float(np.sum(ref["energy"]))
    assert abs(tot[0].item() - E) <= 1e-5 * max(np.abs(ref["energy"]).sum(), 1e-30)
    W = ref["virial"].sum(0)
    assert np.abs(tot[1:].cpu().numpy() - W).max() <= 2e-5 * max(np.abs(ref["virial"]).sum(), 1e-30)


@pytest.mark.parametrize("energy", [False, True])
@pytest.mark.parametrize("model", ["lj", "coulomb", "fp64 sums", "typed"])
def test_wide_addresses_equal_one_lane(cuda, model, energy):
    """The walk with 64-bit addresses, which only lists beyond the 32-bit offsets take, against the walk of
    one lane: a wave without its whole iterations visits the same entries in the same order, so the
    results are the same bits."""
    import ctypes
    import torch
    n, L = 1029, 13.7
    P = _cloud(n, L, seed=n)
    X, Y, Z = (torch.from_numpy(np.ascontiguousarray(P[:, d])).cuda() for d in range(3))
    q = torch.from_numpy(np.where(np.arange(n) % 2, 1.0, -1.0).astype(np.float32)).cuda()
    ws = pdx.DeviceNeighborWorkspace(n, (L,) * 3, 2.5, 0.4, 128)
    ws.update(X, Y, Z, q)
    coul = pdx.RealSpaceCoulomb(1.0, 2.5, 1.2) if model == "coulomb" else None
    lj = pdx.MixedSigmaLJ(np.linspace(0.9, 1.0, n), rcut_factor=2.5) if model == "typed" else pdx.LennardJones()
    pf = pdx.PairForce(lj, coulomb=coul, lanes=1, accumulation="fp64" if model == "fp64 sums" else "fp32")
    test_pair_wide = ctypes.CDLL(pdx.LIB_PATH).pdx_test_pair_wide
    test_pair_wide.argtypes = [ctypes.c_void_p, ctypes.c_int32]
    out = []
    for wide in (0, 1):
        assert test_pair_wide(pf._h, wide) == 0
        f = [torch.full((n,), 7.0, device="cuda") for _ in range(4)]
        V = torch.full((6, n), 7.0, device="cuda")
        tot = torch.zeros(7, dtype=torch.float64, device="cuda")
        if energy:
            pf.compute(ws, *f, V, tot, energy=True)
        else:
            pf.compute(ws, *f[:3], energy=False)
        ws.status()
        out.append(torch.cat([*f, V.flatten(), tot.float()]))
    assert torch.equal(*out) and float(out[0][:3 * n].abs().max()) > 8.0
