"""Energy and forces into host arrays, through the C-ABI: the arrays of a call
are staged through a block on the device, and none of the caller's memory is
touched once the call is over, also when it returned an error.  The reference
computes in place (default_compute_func.f90:25-45), so a caller may free or
reuse its arrays at once."""
import ctypes

import numpy as np
import pytest
import torch

from atomistica_amd import _lib
from atomistica_amd import native as N

pytestmark = pytest.mark.gpu


def test_no_copy_under_way_after_an_error():
    """An Ewald call with a mask is refused.  Its arrays are page-locked
    and too large for the packed block, so the copies queued before the refusal
    read them directly; matrix products queued ahead of them keep the stream
    busy for a while."""
    n = 250000
    rng = np.random.default_rng(1)
    L = 150.0
    p = N.from_atoms(rng.random((n, 3)) * L, np.eye(3) * L, [True] * 3, np.full(n, 11, np.int32))
    nl = N.Neighbors(100)
    pot = N.Ewald(cutoff=3.0, beta=1.0, kmax=1.0)
    pot.bind_to(p, nl)
    f = torch.zeros((n, 3), dtype=torch.float64, pin_memory=True)
    w = torch.zeros(9, dtype=torch.float64, pin_memory=True)
    q = torch.zeros(n, dtype=torch.float64, pin_memory=True)
    m = torch.ones(n, dtype=torch.int32, pin_memory=True)
    e = ctypes.c_double(0.0)

    def ptr(t):
        return ctypes.c_void_p(t.data_ptr())

    a = torch.rand((8192, 8192), device="cuda")
    torch.cuda.synchronize()
    print("error with host arrays", n, flush=True)
    with torch.cuda.stream(torch.cuda.Stream()):
        N.use_torch_stream()
        for _ in range(20):
            b = a @ a
        rc = _lib.load().agpu_potential_energy_and_forces(
            pot._h, p._h, nl._h, ptr(q), ctypes.byref(e), ptr(f), ptr(w), ptr(m), None, None, None, None, None,
            _lib.HOST)
        idle = torch.cuda.current_stream().query()
        torch.cuda.current_stream().synchronize()
    N.use_torch_stream()
    assert rc == _lib.ERR_UNSUPPORTED
    assert idle
    del b


def test_block_of_a_large_call_is_given_back():
    """A call with per-bond arrays needs 104 bytes per list entry on the card,
    143 MB here, and a potential keeps the block of small calls only.  The first
    call without them settles the memory that the potential keeps for itself."""
    from atomistica_amd import workloads as W
    pos, cell, pbc, Z = W.diamond_si(35, sigma=0.05, seed=2)
    p = N.from_atoms(pos, cell, pbc, Z)
    nl = N.Neighbors(100)
    pot = N.Tersoff()
    pot.bind_to(p, nl)
    print("per-bond host arrays", len(pos), flush=True)
    nl.update(p)
    size = 104 * len(nl.get_list(p)[1])
    pot.energy_and_forces(p, nl)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    pot.energy_and_forces(p, nl, epot_per_bond=True, f_per_bond=True, wpot_per_bond=True)
    kept = before - torch.cuda.mem_get_info()[0]
    print("  block of %.0f MB, kept %.0f MB" % (size / 1e6, kept / 1e6), flush=True)
    assert size > 130e6
    assert kept < 8 << 20
