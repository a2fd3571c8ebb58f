"""Batched replicas: forces against the FP64 direct sums, short trajectories against the
FP64 velocity-Verlet oracle, every replica of a batch bitwise equal to the same box run
alone, launch shapes, graph replay, energy conservation."""
import numpy as np
import pytest

import oracle
import pdx
from pdx import replicas, systems

pytestmark = pytest.mark.gpu


def _host(state, k, off):
    a, b = off[k], off[k + 1]
    return {n: state[n][a:b].cpu().numpy().astype(np.float64) for n in state}


def _small_batch(seed=3, nrep=12, n_range=(256, 1500)):
    return systems.replica_batch(nrep, seed=seed, n_range=n_range)


def test_forces_match_direct_sums(cuda):
    b = _small_batch()
    for stencil in (1, 2):
        rb = pdx.ReplicaBatch(b["specs"], block=256, stencil=stencil)
        st = replicas.device_state(b)
        out = rb.forces(st).cpu().numpy()
        for k, s in enumerate(b["specs"]):
            h = _host(st, k, rb.offsets)
            d = oracle.pair_direct(h["x"], h["y"], h["z"], s["box"], kind=s["model"], cutoff=s.get("cutoff", 2.5))
            F = np.stack([h["fx"], h["fy"], h["fz"]], 1)
            err = np.linalg.norm(F - d["F"]) / np.linalg.norm(d["F"])
            assert err < 2e-5, (stencil, k, s["model"], s["n"], err)
            pe = d["energy"].sum()
            if s["model"] == "lj":
                s6 = (1.0 / 2.5) ** 6
                pe -= 0.5 * 4 * (s6 * s6 - s6) * d["counts"].sum()
            assert abs(out[k, 0] - pe) < 1e-5 * max(1.0, abs(pe)), (k, out[k, 0], pe)
            assert abs(out[k, 2] - d["virial"][:, :3].sum()) < 1e-5 * max(1.0, np.abs(d["virial"]).sum())
            assert out[k, 3] == s["n"]
    info = rb.info()
    print(f"[replicas] {info}", flush=True)


def test_all_pairs_boxes(cuda):
    """Boxes with fewer than three cells a side take the all-pairs traversal."""
    specs = [{"model": "lj", "n": 300, "box": (6.8, 6.8, 6.8), "cutoff": 2.5},
             {"model": "wca", "n": 256, "box": (6.6, 6.6, 6.6)}]
    rng = np.random.default_rng(4)
    xs = [rng.random((s["n"], 3)) * s["box"][0] - s["box"][0] / 2 for s in specs]
    X = np.concatenate(xs).astype(np.float32)
    bd = dict(x=X[:, 0], y=X[:, 1], z=X[:, 2], vx=np.zeros(len(X)), vy=np.zeros(len(X)), vz=np.zeros(len(X)))
    rb = pdx.ReplicaBatch(specs)
    assert rb.info()["allpairs_replicas"] == 1
    st = replicas.device_state(bd)
    rb.forces(st)
    for k, s in enumerate(specs):
        h = _host(st, k, rb.offsets)
        d = oracle.pair_direct(h["x"], h["y"], h["z"], s["box"], kind=s["model"], cutoff=s.get("cutoff", 2.5))
        F = np.stack([h["fx"], h["fy"], h["fz"]], 1)
        assert np.linalg.norm(F - d["F"]) / np.linalg.norm(d["F"]) < 2e-5


def test_trajectory_matches_fp64_verlet(cuda):
    b = _small_batch(seed=5, nrep=6, n_range=(256, 600))
    rb = pdx.ReplicaBatch(b["specs"])
    st = replicas.device_state(b)
    h0 = [_host(st, k, rb.offsets) for k in range(rb.nrep)]
    rb.forces(st, energy=False)
    rb.run(st, 20, dt=0.005)
    for k, s in enumerate(b["specs"]):
        h = _host(st, k, rb.offsets)
        X, V, F, *_ = oracle.vv_steps(h0[k]["x"], h0[k]["y"], h0[k]["z"], h0[k]["vx"], h0[k]["vy"], h0[k]["vz"],
                                      s["box"], kind=s["model"], cutoff=s.get("cutoff", 2.5), dt=0.005, nsteps=20)
        L = s["box"][0]
        d = np.stack([h["x"], h["y"], h["z"]], 1) - X
        d -= L * np.round(d / L)
        dv = np.stack([h["vx"], h["vy"], h["vz"]], 1) - V
        print(f"[replicas] {s['model']} n={s['n']} max|dx|={np.abs(d).max():.2e} max|dv|={np.abs(dv).max():.2e}",
              flush=True)
        assert np.abs(d).max() < 1e-4
        assert np.abs(dv).max() < 1e-3
        assert np.all(np.abs(np.stack([h["x"], h["y"], h["z"]], 1)) <= L / 2)


def test_batch_equals_each_box_alone(cuda):
    b = _small_batch(seed=7, nrep=24, n_range=(256, 3000))
    rb = pdx.ReplicaBatch(b["specs"])
    st = replicas.device_state(b)
    init = replicas.clone_state(st)
    rb.forces(st, energy=False)
    out = rb.run(st, 100, dt=0.005, energy=True).cpu().numpy()
    for k in (0, 5, 11, 23):
        s = b["specs"][k]
        a, e = rb.offsets[k], rb.offsets[k + 1]
        one = pdx.ReplicaBatch([s])
        st1 = {n: v[a:e].clone() for n, v in init.items()}
        one.forces(st1, energy=False)
        o1 = one.run(st1, 100, dt=0.005, energy=True).cpu().numpy()
        for n in st:
            assert np.array_equal(st[n][a:e].cpu().numpy(), st1[n].cpu().numpy()), (k, n)
        assert np.array_equal(out[k], o1[0]), k


def test_launch_shapes_and_graph_replay(cuda):
    import torch
    b = _small_batch(seed=9, nrep=10, n_range=(256, 2000))
    rb = pdx.ReplicaBatch(b["specs"], block=256, stencil=1)
    st0 = replicas.device_state(b)
    rb.forces(st0, energy=False)
    ref = replicas.clone_state(st0)
    rb.run(ref, 30)
    # the workgroup size does not change a replica's arithmetic
    for blk in (512, 1024):
        rb.set_launch(blk, 1)
        t = replicas.clone_state(st0)
        rb.run(t, 30)
        for n in t:
            assert torch.equal(t[n], ref[n]), (blk, n)
    # a graph of one 10-step launch, replayed three times, equals 30 eager steps
    rb.set_launch(256, 1)
    g_state = replicas.clone_state(st0)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        rb.run(g_state, 10)  # warm on the capture stream
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g_state = replicas.clone_state(st0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rb.run(g_state, 10)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
    for n in g_state:
        assert torch.equal(g_state[n], ref[n]), n
    best, times = replicas.autotune(rb, st0, steps=5, candidates=[(256, 1), (512, 2)])
    print(f"[replicas] autotune {best} {times}", flush=True)
    assert best in [(256, 1), (512, 2)]


def test_energy_conservation(cuda):
    """Over 1000 steps the total energy of each replica drifts as the FP64 integration of
    the same box does (the drift of these hot starts at dt = 0.005 is integration error,
    O(dt^2), not rounding)."""
    b = _small_batch(seed=11, nrep=4, n_range=(256, 700))
    rb = pdx.ReplicaBatch(b["specs"])
    st = replicas.device_state(b)
    h0 = [_host(st, k, rb.offsets) for k in range(rb.nrep)]
    e0 = rb.forces(st).cpu().numpy()
    e1 = rb.run(st, 1000, dt=0.005, energy=True).cpu().numpy()
    for k, s in enumerate(b["specs"]):
        E0, E1 = e0[k, 0] + e0[k, 1], e1[k, 0] + e1[k, 1]
        drift = (E1 - E0) / s["n"]
        h = h0[k]
        kw = dict(kind=s["model"], cutoff=s.get("cutoff", 2.5), shift=s["model"] == "lj", dt=0.005)
        *_, pa, ka, _ = oracle.vv_steps(h["x"], h["y"], h["z"], h["vx"], h["vy"], h["vz"], s["box"], nsteps=0, **kw)
        *_, pb, kb, _ = oracle.vv_steps(h["x"], h["y"], h["z"], h["vx"], h["vy"], h["vz"], s["box"], nsteps=1000,
                                        **kw)
        ref = ((pb + kb) - (pa + ka)) / s["n"]
        print(f"[replicas] {s['model']} n={s['n']} E/n {E0 / s['n']:.4f} drift {drift:.3e} (FP64 {ref:.3e})",
              flush=True)
        assert abs(E0 - (pa + ka)) < 1e-5 * abs(pa + ka) + 1e-3
        assert abs(drift - ref) < 1e-3 + 0.1 * abs(ref), (k, drift, ref)


@pytest.mark.parametrize("n", [3, 512, 513, 1024, 1025, 8192])
@pytest.mark.parametrize("model,aspect", [("lj", (1.0, 1.0, 1.0)), ("lj", (0.8, 1.0, 1.25)), ("wca", (1.3, 1.0, 0.77))])
def test_forces_at_the_size_steps(cuda, n, model, aspect):
    """The sizes where the lanes per atom change, the largest replica and a nearly empty box, cubic
    and not, with the cells chosen by the library: forces and energies against the FP64 sums."""
    rng = np.random.default_rng(n)
    side = max((n / 0.8) ** (1.0 / 3.0), 8.0)
    box = tuple(side * a for a in aspect)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[rng.permutation(m ** 3)[:n]]
    L = np.array(box)
    # on a lattice of m sites a side, jittered by 8 % of the spacing; some atoms on the faces
    X = ((g + 0.08 * rng.standard_normal(g.shape)) / m - 0.5) * L
    X = (X - L * np.floor(X / L + 0.5)).astype(np.float32)
    L32 = L.astype(np.float32)
    X = np.where(X >= L32 / 2, -L32 / 2, X)
    bd = dict(x=X[:, 0], y=X[:, 1], z=X[:, 2], vx=np.zeros(n), vy=np.zeros(n), vz=np.zeros(n))
    rb = pdx.ReplicaBatch([{"model": model, "n": n, "box": box, "cutoff": 2.5, "shift": False}])
    st = replicas.device_state(bd)
    out = rb.forces(st).cpu().numpy()[0]
    h = _host(st, 0, rb.offsets)
    d = oracle.pair_direct(h["x"], h["y"], h["z"], box, kind=model, cutoff=2.5)
    F = np.stack([h["fx"], h["fy"], h["fz"]], 1)
    # the FP32 bounds of the other force tests (2e-5 of the forces, 1e-5 of the energies)
    assert np.linalg.norm(F - d["F"]) <= 2e-5 * np.linalg.norm(d["F"])
    assert abs(out[0] - d["energy"].sum()) <= 1e-5 * max(np.abs(d["energy"]).sum(), 1e-30)
    assert abs(out[2] - d["virial"][:, :3].sum()) <= 1e-5 * max(np.abs(d["virial"]).sum(), 1e-30)
    assert out[3] == n


@pytest.mark.parametrize("stencil", [0, 1, 2])
def test_atoms_outside_the_box(cuda, stencil):
    """Coordinates that are images outside [-L/2, L/2): forces, energies and virials are those of the
    atoms in the box, and the first drift goes on from the coordinates as given."""
    import torch
    rng = np.random.default_rng(4)
    boxes = [(9.0, 10.0, 11.0), (9.5, 9.0, 8.75), (26.0, 25.0, 24.0)]
    specs, P, S = [], [], []
    for k, box in enumerate(boxes):
        n = (700, 520, 8192)[k]
        m = int(np.ceil(n ** (1 / 3)))
        g = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[rng.permutation(m ** 3)[:n]]
        L = np.array(box)
        X = ((g + 0.5 + 0.08 * rng.standard_normal(g.shape)) / m - 0.5) * L
        X = np.clip(X, -L / 2 + 0.01, L / 2 - 0.01)
        X = np.round(X * 2.0 ** 14) / 2.0 ** 14  # shifts by a box are then exact in FP32
        shift = np.zeros_like(X)
        some = rng.permutation(n)[:n // 4]
        shift[some] = rng.integers(-2, 3, (len(some), 3))
        for d in range(3):  # a little outside: an atom next to a face as the image across the other one
            shift[X[:, d] > L[d] / 2 - 0.3, d] = -1
        specs.append({"model": ("lj", "wca", "lj")[k], "n": n, "box": box, "cutoff": 2.5})
        P.append(X)
        S.append(shift * L)
    X, S = np.concatenate(P), np.concatenate(S)
    v = 0.3 * rng.standard_normal(X.shape)

    def state(X):
        return replicas.device_state(dict(x=X[:, 0], y=X[:, 1], z=X[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2]))
    rb = pdx.ReplicaBatch(specs, stencil=stencil)
    a, b = state(X), state(X + S)
    assert (np.abs(S) > 0).any() and np.array_equal((X + S).astype(np.float32).astype(np.float64), X + S)
    ea, eb = rb.forces(a), rb.forces(b)
    for k in ("fx", "fy", "fz"):
        assert torch.equal(a[k], b[k]), k
        assert torch.isfinite(a[k]).all() and a[k].abs().max() > 1
    assert torch.equal(ea, eb)
    # dt = 0: the step is the wrap alone, which shifts by one box at most
    c = state(X + S)
    rb.run(c, 1, dt=0.0, forces_valid=False)
    L = np.repeat(np.array(boxes), [s["n"] for s in specs], axis=0).astype(np.float32)
    Y = (X + S).astype(np.float32)
    Y = np.where(Y >= L / 2, Y - L, Y)
    Y = np.where(Y < -L / 2, Y + L, Y)
    for d, k in enumerate("xyz"):
        assert np.array_equal(c[k].cpu().numpy(), Y[:, d]), k


def test_coordinates_without_a_cell(cuda):
    """Huge coordinates stay inside the tables: the other atoms' forces are those of a box without these
    atoms. Infinite and undefined ones reach no other replica."""
    import torch
    b = _small_batch(seed=2, nrep=2, n_range=(600, 600))
    huge = {5: 3e38, 17: -3e38, 77: 1e20, 601: -1e20, 700: 1e9}
    rb = pdx.ReplicaBatch(b["specs"])
    good = replicas.device_state(b)
    st = replicas.clone_state(good)
    for i, x in huge.items():
        st["x"][i] = x
        st["y"][i] = x
    rb.forces(st)
    for k in range(2):
        lo, hi = int(rb.offsets[k]), int(rb.offsets[k + 1])
        keep = [i for i in range(lo, hi) if i not in huge]
        one = pdx.ReplicaBatch([dict(b["specs"][k], n=len(keep))])
        s1 = {a: t[keep].contiguous() for a, t in good.items()}
        one.forces(s1)
        for a in ("fx", "fy", "fz"):
            # the same pairs, in rows that the missing atoms pair differently: rounding of ~60 terms
            d = (s1[a] - st[a][keep]).abs().max()
            assert torch.isfinite(st[a][keep]).all() and d <= 1e-4 * s1[a].abs().max(), (k, a)
    rb.forces(good)
    st = replicas.clone_state(good)
    for i, x in {5: np.inf, 17: -np.inf, 77: np.nan}.items():
        st["x"][i] = x
    rb.forces(st)
    for a in ("fx", "fy", "fz"):
        assert torch.equal(st[a][600:], good[a][600:]), a


@pytest.mark.parametrize("sizes,copies,block", [((64,), 16, 256), ((64,), 600, 256), ((128, 64), 4, 256), ((200,), 8, 512),
                                                ((260,), 3, 512), ((700,), 3, 1024), ((64, 700), 300, 512),
                                                ((64, 700), 100, 1024)])
def test_default_workgroup(cuda, sizes, copies, block):
    """The default workgroup has a thread for every lane of the largest replica (two lanes an atom up to
    256 atoms on all pairs), of the mean one where there are more than two replicas a CU; the replicas'
    results are those of any other shape."""
    import torch
    specs, data = [], []
    for n in sizes:
        b = systems.replica_batch(1, seed=n, n_range=(n, n), models=("lj",) if n >= 200 else ("wca",))
        specs += b["specs"]
        data.append(b)
    st = {a: np.tile(np.concatenate([b[a] for b in data]), copies) for a in ("x", "y", "z", "vx", "vy", "vz")}
    rb = pdx.ReplicaBatch(specs * copies)
    assert rb.info()["block"] == block
    a = replicas.device_state(st)
    rb.forces(a)
    rb.run(a, 5)
    for k, (sp, b) in enumerate(zip(specs, data)):  # each replica alone, in workgroups of 256
        one = pdx.ReplicaBatch([sp], block=256)
        s1 = replicas.device_state(b)
        one.forces(s1)
        one.run(s1, 5)
        for t in ("x", "y", "z", "vx", "vy", "vz", "fx", "fy", "fz"):
            for at in (k, len(rb.specs) - len(specs) + k):
                lo, hi = int(rb.offsets[at]), int(rb.offsets[at + 1])
                assert torch.equal(a[t][lo:hi], s1[t]), (t, at)


def test_default_shape_can_be_set_again(cuda):
    """Shape 0, 0 returns a batch to the default it was created with, and the tuner times that default."""
    import torch
    b = _small_batch(seed=6, nrep=6, n_range=(200, 900))
    rb = pdx.ReplicaBatch(b["specs"])
    st = replicas.device_state(b)
    first = rb.info()
    rb.forces(st)
    ref = replicas.clone_state(st)
    rb.run(ref, 10)
    rb.set_launch(256, 1)
    assert (rb.info()["block"], rb.info()["stencil"]) == (256, 1)
    rb.set_launch(first["block"], first["stencil"])
    rb.set_launch(0, 0)
    assert rb.info() == first
    t = replicas.clone_state(st)
    rb.run(t, 10)
    for n in t:
        assert torch.equal(t[n], ref[n]), n
    for bad in ((128, 1), (-1, 0), (256, 3)):
        with pytest.raises(pdx.ArgumentError):
            rb.set_launch(*bad)
    best, times = replicas.autotune(rb, st, steps=2)
    assert "0x0" in times and times[f"{best[0]}x{best[1]}"] == min(times.values())
