"""PME (smooth particle-mesh Ewald) on the GPU against the oracle through the
C-ABI: the full class (real space + reciprocal - self, pme.f90:386-478) in
FP64 within 1e-10 relative -- energy, forces, virial and the electrostatic
potential -- on the reference's test case (NaCl a = 5.64, cutoff 5, grid
10^3, rattled) and larger grids and orders; convergence to the direct
Ewald sum on the GPU; bitwise reproducibility."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from atomistica_amd import native as N
from atomistica_amd import workloads as W

pytestmark = pytest.mark.gpu

REL = 1e-10


def close(a, b, rel=REL):
    a, b = np.asarray(a), np.asarray(b)
    return np.abs(a - b).max() <= rel * max(1.0, np.abs(b).max())


def oracle(pos, q, cell, pbc, cutoff, grid, order):
    beta = math.sqrt(math.log(10.0) * 12.0) / cutoff
    nl = O.nl_build(pos, cell, pbc, cutoff, avgn=400)
    er, fr, wr, pr = O.ewald_real(pos, q, cell, nl, cutoff, beta)
    ek, fk, wk, pk = O.pme_recip(pos, q, cell, beta, grid, order)
    return er + ek, fr + fk, wr + wk, pr + pk


def gpu(pos, q, cell, pbc, Z, cutoff, grid, order, cls=None):
    p = N.from_atoms(pos, cell, pbc, Z)
    nl = N.Neighbors(400)
    pot = cls if cls is not None else N.PME(cutoff=cutoff, order=order, grid=grid)
    pot.bind_to(p, nl)
    e, f, w = pot.energy_and_forces(p, nl, q)
    phi = pot.potential(p, nl, q)
    return e, f, w, phi


def _nacl(n, seed, amp=0.5):
    pos, cell, pbc, Z, q = W.rocksalt(n, sigma=0.0)
    pos = pos + 0.1 + np.random.default_rng(seed).uniform(-amp, amp, pos.shape)
    return pos, cell, pbc, Z, q


CASES = [("reference_case", 2, 1, 5.0, (10, 10, 10), 8),
         ("grid_16_18_20_order6", 2, 2, 5.0, (16, 18, 20), 6),
         ("nacl_3_grid24_order8", 3, 3, 6.0, (24, 24, 24), 8),
         ("order4_grid12", 2, 4, 4.5, (12, 12, 12), 4)]


@pytest.mark.parametrize("name,n,seed,cutoff,grid,order", CASES, ids=[c[0] for c in CASES])
def test_pme_parity(name, n, seed, cutoff, grid, order):
    pos, cell, pbc, Z, q = _nacl(n, seed)
    print("pme case", name, len(pos), grid, order, flush=True)
    e0, f0, w0, p0 = oracle(pos, q, cell, pbc, cutoff, grid, order)
    e, f, w, phi = gpu(pos, q, cell, pbc, Z, cutoff, grid, order)
    print("  E %.12f (oracle %.12f)" % (e, e0), flush=True)
    assert abs(e - e0) <= REL * abs(e0)
    assert close(f, f0) and close(w, w0) and close(phi, p0)


def test_pme_converges_to_direct_ewald_on_gpu():
    # beta = 0.66 (cutoff 8): the B-spline interpolation error at 48^3 and
    # order 10 is then below 1e-11 relative
    pos, cell, pbc, Z, q = _nacl(2, 6, amp=0.2)
    cutoff = 8.0
    beta = math.sqrt(math.log(10.0) * 12.0) / cutoff
    ep, fp, wp, pp = gpu(pos, q, cell, pbc, Z, cutoff, (48, 48, 48), 10)
    ee, fe, we, pe = gpu(pos, q, cell, pbc, Z, cutoff, None, None,
                         cls=N.Ewald(cutoff=cutoff, beta=beta, kmax=2 * beta * math.sqrt(-math.log(1e-16))))
    print("pme vs ewald: dE %.3e  dF %.3e" % (abs(ep - ee), np.abs(fp - fe).max()), flush=True)
    assert abs(ep - ee) < 1e-9 * abs(ee) and np.abs(fp - fe).max() < 1e-8 and np.abs(pp - pe).max() < 1e-8


def test_pme_reproducible_and_charge_derivative():
    pos, cell, pbc, Z, q = _nacl(2, 7)
    a = gpu(pos, q, cell, pbc, Z, 5.0, (10, 12, 14), 8)
    b = gpu(pos, q, cell, pbc, Z, 5.0, (10, 12, 14), 8)
    assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[3], b[3])
    # phi = dE/dq (central FD in one charge)
    h = 1e-5
    qp, qm = q.copy(), q.copy()
    qp[3] += h
    qm[3] -= h
    d = (gpu(pos, qp, cell, pbc, Z, 5.0, (10, 12, 14), 8)[0] - gpu(pos, qm, cell, pbc, Z, 5.0, (10, 12, 14), 8)[0]) / (2 * h)
    assert abs(d - a[3][3]) < 1e-7


EDGES = [(n, grid, order) for n in (2, 5) for grid, order in
         [((3, 3, 3), 3), ((4, 7, 9), 4), ((8, 8, 8), 5), ((9, 16, 17), 6), ((7, 24, 8), 7), ((8, 9, 31), 8),
          ((9, 9, 9), 9), ((10, 12, 23), 10), ((11, 24, 12), 11), ((12, 13, 40), 12)]] + [(900, (16, 9, 25), 8)]


@pytest.mark.parametrize("n,grid,order", EDGES)
@pytest.mark.parametrize("shear", [0.0, 0.15])
def test_pme_brick_edges(n, grid, order, shear):
    """Grids around the 8^3 cells of a brick, down to the order itself (a
    brick's points then cover the grid more than once), every order, odd and
    even lengths (the Nyquist terms of a sheared cell), few ions and many in
    one brick, ions outside the cell."""
    rng = np.random.default_rng(n + order)
    # symmetric strain: the reference's reciprocal indexing then holds
    m = np.eye(3) + shear * np.array([[0, 1, 0.5], [1, 0, -0.4], [0.5, -0.4, 0]])
    cell = np.diag([9.0, 10.0, 12.0]) @ m
    pos = (rng.random((n, 3)) + rng.integers(-1, 2, (n, 3))) @ cell
    q = rng.normal(size=n)
    # neutral: the m = 0 term, left in place as the reference does, then adds
    # nothing, while the oracle drops it
    q -= q.mean()
    Z = np.full(n, 11, np.int32)
    print("pme edges", n, grid, order, shear, flush=True)
    e0, f0, w0, p0 = oracle(pos, q, cell, [True] * 3, 4.0, grid, order)
    e, f, w, phi = gpu(pos, q, cell, [True] * 3, Z, 4.0, grid, order)
    assert abs(e - e0) <= REL * max(1.0, abs(e0))
    assert close(f, f0) and close(w, w0) and close(phi, p0)


@pytest.mark.parametrize("grid,order", [((16, 24, 40), 4), ((16, 24, 40), 8), ((41, 17, 24), 6)])
def test_pme_ions_on_brick_faces(grid, order):
    """Ions on the faces of bricks of 8^3 grid cells, or one ulp of a
    coordinate to either side, in a sheared cell and around it: the brick that
    an ion is sorted into and the place of its points there agree."""
    rng = np.random.default_rng(sum(grid))
    cell = np.diag([9.0, 10.0, 12.0]) @ (np.eye(3) + 0.15 * np.array([[0, 1, 0.5], [1, 0, -0.4], [0.5, -0.4, 0]]))
    n, K = 200, np.array(grid)
    frac = rng.integers(0, 1 + K // 8, (n, 3)) * 8.0 / K - 0.5 + rng.integers(-1, 2, (n, 3))
    frac[np.arange(n), rng.integers(0, 3, n)] = rng.random(n)
    pos = frac @ cell
    for step in (-np.inf, np.inf):
        pos = np.where(rng.random(pos.shape) < 0.25, np.nextafter(pos, step), pos)
    q = rng.normal(size=n)
    q -= q.mean()
    print("pme brick faces", grid, order, flush=True)
    e0, f0, w0, p0 = oracle(pos, q, cell, [True] * 3, 4.0, grid, order)
    e, f, w, phi = gpu(pos, q, cell, [True] * 3, np.full(n, 11, np.int32), 4.0, grid, order)
    assert abs(e - e0) <= REL * max(1.0, abs(e0))
    assert close(f, f0) and close(w, w0) and close(phi, p0)


@pytest.mark.parametrize("n", [60, 64, 65, 300, 2000, 20000])
def test_pme_cluster_in_one_brick(n):
    """n ions of a salt cluster in one brick and 40 more anywhere in the cell:
    the brick's ions are put into index order by comparing them, or, where that
    grows with the square, from the keys of all ions (n above 64).  20 000 ions
    in one brick take 306 ms by comparing and 0.035 ms by the walk."""
    rng = np.random.default_rng(n)
    grid, L = (64, 64, 64), 800.0
    m = int(np.ceil(n ** (1 / 3)))
    site = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = 105.0 + 2.82 * site + rng.uniform(-0.2, 0.2, (n, 3))
    q = np.where(site.sum(1) % 2, 1.0, -1.0)
    assert pos.max() < 200.0                     # the brick from 100 to 200 A
    pos = np.concatenate([pos, rng.random((40, 3)) * L])
    q = np.concatenate([q, rng.normal(size=40)])
    perm = rng.permutation(n + 40)
    pos, q = pos[perm], (q - q.mean())[perm]
    cell = np.diag([L, L, L])
    Z = np.full(n + 40, 11, np.int32)
    print("pme cluster", n, flush=True)
    e0, f0, w0, p0 = oracle(pos, q, cell, [True] * 3, 4.0, grid, 4)
    N.profile_enable(True)
    N.profile_reset()
    e, f, w, phi = gpu(pos, q, cell, [True] * 3, Z, 4.0, grid, 4)
    ms, calls = N.profile_query("pme_order")
    N.profile_enable(False)
    print("  pme_order %.3f ms" % (ms / calls), flush=True)
    assert abs(e - e0) <= REL * max(1.0, abs(e0))
    assert close(f, f0) and close(w, w0) and close(phi, p0)
    assert ms / calls < 20.0
    again = gpu(pos, q, cell, [True] * 3, Z, 4.0, grid, 4)
    assert e == again[0] and np.array_equal(f, again[1]) and np.array_equal(phi, again[3])


def test_pme_bricks_in_parts():
    """Order 12 on 480 x 464 x 472 points: the bricks' points take 11 GB, of
    which 4 GiB are kept at once, so their layers go through in three parts.  The
    call takes those, the grid and its transform (0.8 GB each) and what the
    transforms themselves need (bounded by 4 GB here).  More than 32 768 bricks
    also take the radix sort.  On a mesh this fine the sum agrees with the
    direct one."""
    import torch
    rng = np.random.default_rng(12)
    cell = np.diag([30.0, 28.0, 29.0])
    # ions next to all faces and in a layer across the middle
    pos = np.concatenate([rng.random((100, 3)), np.round(rng.random((60, 3))) + rng.normal(0, 0.01, (60, 3)),
                          rng.random((40, 3)) * [1, 1, 0.02] + [0, 0, 0.49]]) @ cell
    q = rng.normal(size=200)
    q -= q.mean()
    cutoff = 6.0
    beta = math.sqrt(math.log(10.0) * 12.0) / cutoff
    print("pme bricks in parts", flush=True)
    Z = np.full(200, 11, np.int32)
    # the direct sum first: its memory stays with it
    ee, fe, we, pe = gpu(pos, q, cell, [True] * 3, Z, cutoff, None, None,
                         cls=N.Ewald(cutoff=cutoff, beta=beta, kmax=2 * beta * math.sqrt(-math.log(1e-16))))
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    p = N.from_atoms(pos, cell, [True] * 3, Z)
    nl = N.Neighbors(400)
    pot = N.PME(cutoff=cutoff, order=12, grid=(480, 464, 472))
    pot.bind_to(p, nl)
    e, f, w = pot.energy_and_forces(p, nl, q)
    phi = pot.potential(p, nl, q)
    grown = before - torch.cuda.mem_get_info()[0]
    print("  memory of the call %.2f GB, dE %.1e dF %.1e" % (grown / 1e9, abs(e - ee), np.abs(f - fe).max()), flush=True)
    assert grown < 10e9
    assert abs(e - ee) <= REL * np.abs(q * pe).sum()
    assert close(f, fe) and close(w, we) and close(phi, pe)
    e2, f2, _ = pot.energy_and_forces(p, nl, q)
    assert e2 == e and np.array_equal(f2, f)


@pytest.mark.parametrize("n,grid,order", [(200, (8, 8, 8), 6), (400, (8, 16, 16), 5), (770, (16, 16, 16), 4),
                                          (60, (136, 136, 136), 4)])
def test_pme_sorts(n, grid, order):
    """More than 96 ions per brick on the average take the radix sort (200 in
    one brick, 100 in each of four; 770 in eight are just above the line); 4913
    bricks take the one-workgroup scan a second trip."""
    rng = np.random.default_rng(n)
    cell = np.diag([9.0, 10.0, 12.0])
    pos = (rng.random((n, 3)) + rng.integers(-1, 2, (n, 3))) @ cell
    q = rng.normal(size=n)
    q -= q.mean()
    print("pme sorts", n, grid, order, flush=True)
    e0, f0, w0, p0 = oracle(pos, q, cell, [True] * 3, 4.0, grid, order)
    e, f, w, phi = gpu(pos, q, cell, [True] * 3, np.full(n, 11, np.int32), 4.0, grid, order)
    assert abs(e - e0) <= REL * max(1.0, abs(e0))
    assert close(f, f0) and close(w, w0) and close(phi, p0)
