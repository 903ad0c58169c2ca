"""Batched Ewald on the GPU through the C-ABI.

Bars:
  - FP64, structure by structure, against the oracle (real space + self term
    over the oracle's neighbour list, direct k-space sum with the same beta
    and kmax): energy, forces, virial and phi = dE/dq within 1e-10 relative;
  - the same structures through the single-structure Ewald path agree;
  - FP32-arithmetic real space: error against FP64 stated and bounded;
  - the 256-cell workload (64..4096 ions per cell): net force zero per cell,
    bitwise reproducible.
"""
import numpy as np
import pytest

from oracle import oracle as O
from atomistica_amd import workloads as W

pytestmark = pytest.mark.gpu

REL = 1e-10
RC = 10.0


def _params():
    beta = W.ewald_beta(RC, 1e-8)
    return beta, W.ewald_kmax(beta, 1e-8)


def _small_set():
    """Cubic rocksalt cells of 2^3 and 3^3 conventional cells plus a sheared
    (triclinic) one."""
    S, qs = [], []
    for n, seed in ((2, 1), (3, 2), (2, 3)):
        pos, cell, _, _, q = W.rocksalt(n, sigma=0.1, seed=seed)
        S.append((pos, cell))
        qs.append(q)
    pos, cell, _, _, q = W.rocksalt(2, sigma=0.1, seed=4)
    shear = np.array([[1.0, 0.0, 0.0], [0.12, 1.0, 0.0], [-0.07, 0.05, 1.0]])
    S.append((pos @ shear, cell @ shear))
    qs.append(q)
    return S, np.concatenate(qs)


def _oracle(pos, cell, q, beta, kmax):
    nl = O.nl_build(pos, cell, [True] * 3, RC, avgn=400)
    e1, f1, w1, p1 = O.ewald_real(pos, q, cell, nl, RC, beta)
    e2, f2, w2, p2 = O.ewald_kspace(pos, q, cell, beta, kmax)
    return e1 + e2, f1 + f2, w1 + w2, p1 + p2


def _close(a, b, rel=REL):
    a, b = np.asarray(a), np.asarray(b)
    return np.abs(a - b).max() <= rel * max(1.0, np.abs(b).max())


def test_ewald_batch_fp64_parity():
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    S, q = _small_set()
    b = Batch(S)
    e, f, w, p = ewald_batch(b, q, RC, beta, kmax, "fp64", phi=True)
    e, f, w, p = (t.cpu().numpy() for t in (e, f, w, p))
    print("ewald batch parity: %d cells, %d ions" % (b.nstruct, b.ntot), flush=True)
    for s, (pos, cell) in enumerate(S):
        a0, a1 = b.offsets[s], b.offsets[s + 1]
        re_, rf, rw, rp = _oracle(pos, cell, q[a0:a1], beta, kmax)
        assert abs(e[s] - re_) <= REL * abs(re_), (s, e[s], re_)
        assert _close(f[a0:a1], rf), s
        assert _close(w[s], rw), s
        assert _close(p[a0:a1], rp), s


def test_ewald_batch_matches_single_structure_path():
    from atomistica_amd import native as N
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    S, q = _small_set()
    b = Batch(S)
    e, f, _, _ = ewald_batch(b, q, RC, beta, kmax, "fp64", virial=False)
    e, f = e.cpu().numpy(), f.cpu().numpy()
    for s, (pos, cell) in enumerate(S):
        a0, a1 = b.offsets[s], b.offsets[s + 1]
        Z = np.where(q[a0:a1] > 0, 11, 17).astype(np.int32)
        p = N.from_atoms(pos, cell, np.array([True] * 3), Z)
        nl = N.Neighbors(400)
        pot = N.Ewald(cutoff=RC, beta=beta, kmax=kmax)
        pot.bind_to(p, nl)
        e1, f1, _ = pot.energy_and_forces(p, nl, q[a0:a1])
        assert abs(e[s] - e1) <= REL * abs(e1), s
        assert _close(f[a0:a1], f1), s


def test_ewald_batch_mixed_error():
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    S, q = _small_set()
    b = Batch(S)
    e64, f64, w64, _ = ewald_batch(b, q, RC, beta, kmax, "fp64")
    e32, f32, w32, _ = ewald_batch(b, q, RC, beta, kmax, "mixed")
    df = (f32 - f64).cpu().numpy()
    de = np.abs((e32 - e64).cpu().numpy()) / np.diff(b.offsets)
    rms = float(np.sqrt(np.mean(df ** 2)))
    print("ewald batch mixed: F rms %.3e max %.3e, |dE|/N max %.3e (e^2/A)" % (rms, np.abs(df).max(), de.max()),
          flush=True)
    assert rms <= 1e-5 and de.max() <= 1e-5


def test_ewald_batch_256_cells():
    import time
    import torch
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    S, q = W.rocksalt_cells(256, seed=5)
    b = Batch(S)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    e1, f1, w1, _ = ewald_batch(b, q, RC, beta, kmax, "fp64")
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    e2, f2, w2, _ = ewald_batch(b, q, RC, beta, kmax, "fp64")
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    print("ewald batch 256 cells: %d ions, first %.1f ms, second %.1f ms" % (b.ntot, 1e3 * (t1 - t0), 1e3 * (t2 - t1)),
          flush=True)
    assert torch.equal(e1, e2) and torch.equal(f1, f2) and torch.equal(w1, w2)
    fn = f1.cpu().numpy()
    for s in range(b.nstruct):
        a0, a1 = b.offsets[s], b.offsets[s + 1]
        assert np.abs(fn[a0:a1].sum(0)).max() < 1e-8, s
    # the two smallest cells against the oracle
    sizes = np.diff(b.offsets)
    for s in np.argsort(sizes, kind="stable")[:2]:
        a0, a1 = b.offsets[s], b.offsets[s + 1]
        pos, cell = S[s]
        re_, rf, _, _ = _oracle(pos, cell, q[a0:a1], beta, kmax)
        assert abs(float(e1[s]) - re_) <= REL * abs(re_)
        assert _close(fn[a0:a1], rf)


def test_wide_cell_does_not_grow_the_scratch_of_others():
    """200 cells of 512 ions and one of 100 A with 64: the wide cell's k are
    shared out over many workgroups.  The partial forces of each cell take the
    splits of that cell only, so a call with forces needs little more memory
    than one without: 32 bytes per ion and split, in all 64 ions x 6144
    workgroups and two more splits per ion.  The wide cell matches the oracle."""
    import torch
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    S, q = W.rocksalt_cells(200, nmin=4, nmax=4)
    n = sum(len(p) for p, _ in S)
    rng = np.random.default_rng(8)
    cell = np.diag([100.0, 100.0, 100.0])
    pos = rng.random((64, 3)) @ cell
    qw = np.where(np.arange(64) % 2, 1.0, -1.0)
    b = Batch(S + [(pos, cell)])
    q = np.concatenate([q, qw])
    print("ewald batch with a wide cell", n + 64, flush=True)
    ewald_batch(b, q, RC, beta, kmax, forces=False, virial=False)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    e, f, w, phi = ewald_batch(b, q, RC, beta, kmax, phi=True)
    torch.cuda.synchronize()
    grown = before - torch.cuda.mem_get_info()[0]
    print("  a call with forces takes %.1f MB more" % (grown / 1e6), flush=True)
    # the partial forces, and torch's blocks of the returned arrays
    assert grown <= 32 * (64 * 6144 + 2 * (n + 64)) + 64e6
    e0, f0, w0, p0 = _oracle(pos, cell, qw, beta, kmax)
    assert abs(e[-1].item() - e0) <= REL * abs(e0)
    assert _close(f[-64:].cpu(), f0) and _close(w[-1].cpu(), w0) and _close(phi[-64:].cpu(), p0)


@pytest.mark.parametrize("sizes", [(1, 2, 3, 4, 5), (7, 8, 9, 15, 16, 17), (31, 32, 33, 63, 64, 65),
                                   (64, 65, 127, 128, 129, 260), (8, 700)])
@pytest.mark.parametrize("scale", [2.6, 3.4])
def test_ewald_batch_small_cells(sizes, scale):
    """Cells of up to 128 ions keep one or two ions on each lane, or one on
    several lanes that take different images (around each power of two); a
    batch with larger cells takes two launches, or one if the small cells hold
    few of the ions.  Cells from a quarter of the cut-off up, sheared, ions
    outside them, a charge of zero."""
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    rng = np.random.default_rng(sum(sizes))
    S, qs = [], []
    for n in sizes:
        cell = np.diag([1.0, 1.1, 0.9]) * scale * n ** (1 / 3.0) @ (np.eye(3) + rng.uniform(-0.15, 0.15, (3, 3)))
        S.append((W.random_positions(n, cell, 1.2, int(rng.integers(1 << 30))) + rng.integers(-2, 3, (n, 3)) @ cell, cell))
        q = rng.normal(size=n)
        q[n // 2] = 0.0 if n > 6 else q[n // 2]
        qs.append(q - q.mean() * (q != 0) * n / max(1, (q != 0).sum()))
    b = Batch(S)
    print("ewald batch small cells", sizes, scale, flush=True)
    e, f, w, phi = ewald_batch(b, np.concatenate(qs), RC, beta, kmax, phi=True)
    for s, ((pos, cell), q) in enumerate(zip(S, qs)):
        nl = O.nl_build(pos, cell, [True] * 3, RC, avgn=2000)
        e1, f1, w1, p1 = O.ewald_real(pos, q, cell, nl, RC, beta)
        e2, f2, w2, p2 = O.ewald_kspace(pos, q, cell, beta, kmax)
        a = slice(b.offsets[s], b.offsets[s + 1])
        assert abs(e[s].item() - (e1 + e2)) <= REL * max(1.0, abs(e1 + e2)), len(pos)
        assert _close(f[a].cpu(), f1 + f2) and _close(w[s].cpu(), w1 + w2), len(pos)
        assert _close(phi[a].cpu(), p1 + p2), len(pos)


def test_ewald_batch_of_unit_cells_is_not_slow():
    """5000 cells of 8 ions: the real-space sum takes 0.16 ms and took 0.92 ms
    with an ion per lane and the other lanes idle."""
    from atomistica_amd import native as N
    from atomistica_amd.batch import Batch, ewald_batch
    beta, kmax = _params()
    S, q = W.rocksalt_cells(5000, nmin=1, nmax=1)
    b = Batch(S)
    best = np.inf
    for _ in range(5):
        N.profile_enable(True)
        N.profile_reset()
        ewald_batch(b, q, RC, beta, kmax)
        best = min(best, N.profile_query("ewald_batch_real_fp64")[0])
        N.profile_enable(False)
    print("ewald batch of unit cells: %.3f ms" % best, flush=True)
    assert best < 0.45
