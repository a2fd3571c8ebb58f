"""Row walk of the pair kernel: particle counts and rows that are no multiple of an iteration, empty and
short rows, and every lane count, in small boxes in random order; the walk with 64-bit addresses; and, in a
wide box in spatial order, waves that skip the seam test and whole iterations that skip the bounds test."""
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


# (particles, box side): a gas whose rows hold 0 to a few entries and ragged liquids; in random order, so
# that nearly every wave has a particle at a face
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


@pytest.mark.parametrize("coulomb", [False, True])
@pytest.mark.parametrize("lanes", [0, 1, 2, 4, 8])
def test_whole_iterations_away_from_the_faces(cuda, lanes, coulomb):
    """Spatially ordered rows of a wide box, as large systems have them: waves without a face particle,
    which skip the seam test, and iterations that every lane has in full, which take no bounds test;
    forces and energies of LJ, and of LJ with Coulomb, against FP64 sums."""
    import torch
    from pdx import systems
    s = systems.fcc_lattice(4 * 13 ** 3, 0.8442, 0.05, seed=3)
    n, L, rc, skin = s["N"], s["box"], 2.5, 0.4
    q = torch.from_numpy(np.where(np.random.default_rng(1).random(n) < 0.5, 1.0, -1.0).astype(np.float32)).cuda()
    X = [torch.from_numpy(s[k]).cuda() for k in "xyz"]
    ws = pdx.DeviceNeighborWorkspace(n, L, rc, skin, 160)
    ws.update(*X, q)
    p = ws.spatial_order()
    X, q = [t[p].contiguous() for t in X], q[p].contiguous()
    ws.invalidate()
    ws.update(*X, q)
    ws.status()
    # the two shortcuts of the walk are taken: counted as the kernel counts them (automatic lanes: 16)
    G = lanes or 16
    R = torch.stack(X, 1).double()
    Lt = torch.tensor(L, dtype=torch.float64, device="cuda")
    per = 64 // G
    m = n // per * per
    face = (R.abs() > Lt / 2 - 1.001 * (rc + 2 * skin)).any(1)[:m].view(-1, per).any(1)
    full = ws.counts()[:m].view(-1, per).min(1).values // (4 * G)
    assert ((~face) & (full > 0)).any() and (face & (full > 0)).any()

    coul = pdx.RealSpaceCoulomb(2.0, rc, 1.2) if coulomb else None
    pf = pdx.PairForce(pdx.LennardJones(cutoff=rc), coulomb=coul, lanes=lanes)
    f, g = ([torch.full((n,), 7.0, device="cuda") for _ in range(3)] for _ in range(2))
    E = torch.full((n,), 7.0, device="cuda")
    V = torch.full((6, n), 7.0, device="cuda")
    tot = torch.zeros(7, dtype=torch.float64, device="cuda")
    pf.compute(ws, *f, E, V, tot, energy=True)
    pf.compute(ws, *g, energy=False)
    F = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
    U = torch.zeros(n, dtype=torch.float64, device="cuda")
    W = torch.zeros(n, 6, dtype=torch.float64, device="cuda")
    size = torch.zeros(n, dtype=torch.float64, device="cuda")  # sum of the terms' magnitudes
    qd = q.double()
    for a in range(0, n, 512):
        d = R[a:a + 512, None, :] - R[None, :, :]
        d -= Lt * torch.round(d / Lt)
        r2 = (d * d).sum(-1)
        inside = (r2 > 0) & (r2 < rc * rc)
        r2 = torch.where(inside, r2, torch.ones_like(r2))
        s6 = r2 ** -3
        fr, u = 24 * (2 * s6 * s6 - s6) / r2, 4 * (s6 * s6 - s6)
        if coulomb:
            r, qq = r2.sqrt(), 2.0 * qd[a:a + 512, None] * qd[None, :]
            u = u + qq * torch.erfc(1.2 * r) / r
            fr = fr + qq * (torch.erfc(1.2 * r) / r + 2.4 / math.sqrt(math.pi) * torch.exp(-1.44 * r2)) / r2
        fr, u = torch.where(inside, fr, torch.zeros_like(fr)), torch.where(inside, u, torch.zeros_like(u))
        F[a:a + 512] = (fr[..., None] * d).sum(1)
        U[a:a + 512] = 0.5 * u.sum(1)
        size[a:a + 512] = (fr.abs() * r2.sqrt()).sum(1)
        for k, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
            W[a:a + 512, k] = 0.5 * (fr * d[..., i] * d[..., j]).sum(1)
    if coulomb:  # the self energy -C alpha / sqrt(pi) q^2
        U -= 2.0 * 1.2 / math.sqrt(math.pi) * qd * qd
    # FP32: about 90 terms, each rounded to some 30 ulps (the position difference's rounding enters
    # r^-14), against the sum of their magnitudes; the total energies and virials average that
    bound = (90 + 30 * 14) * 6e-8 * size
    for got in (f, g):
        dF = (torch.stack(got, 1).double() - F).abs().max(1).values
        assert (dF <= bound).all(), (dF / bound).max().item()
    assert (E.double() - U).abs().max() <= 1e-4 * U.abs().max()
    assert abs(tot[0] - U.sum()).item() <= 1e-5 * U.abs().sum().item()
    assert ((tot[1:] - W.sum(0)).abs() <= 2e-5 * W.abs().sum()).all()
