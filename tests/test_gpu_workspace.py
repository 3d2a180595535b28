"""The adjoint's workspace between calls: reused by every context of the device, never larger
than a call's limit, returned on request, with the last context, and to an allocation that
would fail without it; the results do not depend on what block a call runs in."""
import gc
import threading

import numpy as np
import pytest
import torch

import test_gpu_adjoint as ta

pytestmark = pytest.mark.gpu

MB = 1 << 20
SLACK = 16 * MB     # allocation granularity


def used_since(free0):
    return free0 - torch.cuda.mem_get_info()[0]


@pytest.fixture
def free0(cpmp):
    """free device memory with no workspace kept from before"""
    gc.collect()
    g = cpmp.Lattice(cpmp.make_params(8, 8, 8, nwall=0))
    g.release_workspace()
    g.close()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


DIMS = (48, 48, 48)
N = DIMS[0] * DIMS[1] * DIMS[2]
TAPE = 80 * N           # bytes of one taped step


def lattice(cpmp):
    return ta._small_lattice(cpmp, DIMS)


def test_a_small_limit_leaves_no_larger_block(cpmp, free0):
    g, target = lattice(cpmp)
    own = used_since(free0)
    g.adjoint(20, target, checkpoint_every=20, tape_budget_bytes=20 * TAPE)
    big = used_since(free0) - own
    plan = g.adjoint_plan(20, 4)
    limit = plan["device_bytes"]
    assert limit + 2 * SLACK < big
    g.adjoint(20, target, checkpoint_every=4, memory_limit_bytes=limit)
    assert used_since(free0) - own <= limit + SLACK
    g.close()


def test_one_block_serves_every_context_and_closes_with_the_last(cpmp, free0):
    a, target = lattice(cpmp)
    b, _ = lattice(cpmp)
    own = used_since(free0)
    ra = a.adjoint(12, target, checkpoint_every=12)
    one = used_since(free0) - own
    rb = b.adjoint(12, target, checkpoint_every=12)
    assert used_since(free0) - own <= one + SLACK
    assert ra[0] == rb[0] and np.array_equal(ra[1], rb[1]) and ra[3] == rb[3]
    a.close()
    b.close()
    assert used_since(free0) <= SLACK


def test_release_returns_the_block(cpmp, free0):
    g, target = lattice(cpmp)
    own = used_since(free0)
    need = g.adjoint_plan(12, 12)["device_bytes"]
    g.adjoint(12, target, checkpoint_every=12)
    assert need <= g.release_workspace() <= need + SLACK
    assert g.release_workspace() == 0
    assert used_since(free0) - own <= SLACK
    g.close()


def test_an_allocation_gets_the_kept_block(cpmp, free0):
    """a lattice that fits the device only without the kept block can be created"""
    g, target = lattice(cpmp)
    g.adjoint(60, target, checkpoint_every=60, tape_budget_bytes=60 * TAPE)
    kept = 60 * TAPE
    p = cpmp.make_params(96, 96, 96, eos="PRW", tr=0.75)
    probe = cpmp.Lattice(p)
    need = probe.memory()
    probe.close()
    assert 2 * SLACK < need - kept // 2 < need - 2 * SLACK
    hogs = []
    try:
        for _ in range(2):      # what the first leaves is more than asked for
            left = torch.cuda.mem_get_info()[0] - (need - kept // 2)
            hogs.append(torch.empty(max(left, 0), dtype=torch.uint8, device="cuda"))
        assert torch.cuda.mem_get_info()[0] < need - SLACK
        other = cpmp.Lattice(p)
        other.close()
    finally:
        hogs.clear()
        torch.cuda.empty_cache()
    g.step(1)           # no error of the first attempt is left behind
    g.close()


def test_results_do_not_depend_on_the_block(cpmp):
    """one context through growing and shrinking plans and released blocks against fresh
    contexts, whose calls allocate"""
    plans = [dict(checkpoint_every=3), dict(checkpoint_every=20, tape_budget_bytes=20 * TAPE), dict(checkpoint_every=6),
             dict(checkpoint_every=20), dict(checkpoint_every=5, tape_budget_bytes=7 * TAPE)]
    g, target = lattice(cpmp)
    rho0 = g.get("rho")
    for i, kw in enumerate(plans + plans[::-1]):
        if i == 7:
            g.release_workspace()
        g.init_from_rho(rho0)
        r = g.adjoint(20, target, **kw)
        f, _ = lattice(cpmp)
        f.release_workspace()
        s = f.adjoint(20, target, **kw)
        f.close()
        assert r[0] == s[0] and r[3] == s[3] and np.array_equal(r[1], s[1]) and np.array_equal(r[2], s[2]), i
    g.close()


def test_calls_of_several_threads(cpmp):
    """contexts on three threads at once: each call has a block of its own while it runs"""
    g, target = lattice(cpmp)
    want = g.adjoint(20, target, checkpoint_every=4)
    out = [None] * 3

    def work(k):
        h, _ = lattice(cpmp)
        rho0 = h.get("rho")
        res = []
        for every in (4, 20, 4):
            h.init_from_rho(rho0)
            res.append(h.adjoint(20, target, checkpoint_every=every))
        h.close()
        out[k] = res

    ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for res in out:
        for r in res:
            assert r[0] == want[0] and r[3] == want[3] and np.array_equal(r[1], want[1])
    g.close()
