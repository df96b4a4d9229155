"""Hand-overs between the workgroups of one launch when a workgroup does not
get what it waits for in time (the poll limit set from the host: every kernel
exits normally), against the oracle."""
import ctypes as C
import sys

import numpy as np
import pytest

from obvh_amd import _lib, ops, synth
from obvh_amd.layouts import TRACE_DTYPE

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t

    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("polls", [0, 1, 8, 1 << 12])
def test_single_fit_tiles_that_give_up(torch, oracle_lib, polls):
    """Fits of 5, 64 and 128 tiles whose tiles stop waiting after `polls` polls: the exact box and trace every time, also
    on a workspace whose counters were cleared before the first fit only."""
    lib = _lib.lib()
    fit = lib.obvh_dito_soa_polls
    fit.restype = C.c_char_p
    ws = torch.zeros(lib.obvh_dito_workspace_size(262144), dtype=torch.uint8, device="cuda")
    for call, n in enumerate((8193, 131072, 262144, 8193, 131072)):
        say(f"[dito_soa_polls] polls={polls} n={n}")
        p = synth.gaussian_points(n, seed=10 * polls % 97 + call)
        x, y, z = (torch.from_numpy(np.ascontiguousarray(p[:, k])).cuda() for k in range(3))
        out = torch.zeros(15, dtype=torch.float32, device="cuda")
        tr = torch.zeros(TRACE_DTYPE.itemsize, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        err = fit(ptr(x), ptr(y), ptr(z), C.c_uint64(n), ptr(out), ptr(tr), ptr(ws), C.c_uint64(ws.numel()),
                  C.c_uint32(polls), C.c_uint32(call == 0), None)
        assert err is None, err
        torch.cuda.synchronize()
        exp, etr = oracle_lib.points_obb(p, trace=True)
        assert np.array_equal(out.cpu().numpy(), exp)
        got = tr.cpu().numpy().view(TRACE_DTYPE)[0]
        for f in ("slab_min_idx", "slab_max_idx", "best", "degenerate", "result_aabb"):
            assert np.array_equal(got[f], etr[f]), f


@pytest.mark.parametrize("nf", [4097, 40000, 140000, 1300000])
def test_sort_tiles_that_give_up(torch, oracle_lib, nf):
    """The LBVH's sort with a poll limit of 0: every tile counts all earlier tiles' keys itself (1, 2, 4 and 8 pairs per
    thread).  The same tree as with waiting, and as the oracle's."""
    say(f"[lbvh_build_polls] nf={nf}")
    lib = _lib.lib()
    build = lib.obvh_lbvh_build_polls
    build.restype = C.c_char_p
    rng = np.random.default_rng(nf)
    V = rng.uniform(0, 1, (nf, 1, 3)).astype(np.float32) + rng.uniform(0, 1e-4, (nf, 3, 3)).astype(np.float32)
    V = np.ascontiguousarray(V.reshape(-1, 3))
    F = np.zeros((nf, 4), dtype=np.uint32)
    F[:, :3] = np.arange(3 * nf).reshape(nf, 3)
    Vd, Fd = torch.from_numpy(V).cuda(), torch.from_numpy(F.view(np.int32)).cuda()
    t = ops.lbvh_build(Vd, Fd)
    ws = torch.zeros(lib.obvh_lbvh_workspace_size(nf), dtype=torch.uint8, device="cuda")
    for polls in (0, 1):
        o = {k: torch.zeros_like(t[k]) for k in ("nodes", "parents", "counts", "costs", "mortons")}
        torch.cuda.synchronize()
        err = build(ptr(Vd), ptr(Fd), C.c_uint32(nf), ptr(o["nodes"]), ptr(o["parents"]), ptr(o["counts"]), ptr(o["costs"]),
                    ptr(o["mortons"]), ptr(ws), C.c_uint64(ws.numel()), C.c_uint32(polls), None)
        assert err is None, err
        torch.cuda.synchronize()
        for k in o:
            assert torch.equal(o[k], t[k]), k
    nodes, parents, counts, costs, mortons = oracle_lib.lbvh_build(V, F)
    assert np.array_equal(t["mortons"].cpu().numpy().view(np.uint32), mortons)
    assert np.array_equal(t["parents"].cpu().numpy().view(np.uint32), parents)
    assert np.array_equal(ops.nodes_to_numpy(t["nodes"]).view(np.uint8), nodes.view(np.uint8))
