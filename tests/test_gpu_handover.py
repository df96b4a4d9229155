"""Hand-overs between the workgroups of one launch, against the oracle: calls at
the same time, calls captured in a graph, and launches in which a workgroup
stops waiting (the poll limit set from the host; every kernel exits normally)."""
import ctypes as C
import sys
import threading

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


def bits(t):
    import torch

    return t.contiguous().view(torch.uint8)


class Job:
    """One call that hands over between workgroups, with its own inputs, workspace and expected outputs."""

    def __init__(self, torch, oracle_lib, kind, seed):
        self.kind, lib = kind, _lib.lib()
        if kind in ("fit", "large"):  # 64 tiles in one launch, 196 in two
            n = 131072 if kind == "fit" else 400001
            p = synth.gaussian_points(n, seed=seed)
            self.xyz = [torch.from_numpy(np.ascontiguousarray(p[:, k])).cuda() for k in range(3)]
            need = lib.obvh_dito_workspace_size(n)
        else:
            V, F = synth.icosphere(80, seed=seed) if kind == "lbvh" else synth.hairball(tubes=1500, seed=seed)
            self.mesh = torch.from_numpy(V).cuda(), torch.from_numpy(F.view(np.int32)).cuda()
            need = (lib.obvh_lbvh_workspace_size if kind == "lbvh" else lib.obvh_atrbvh_workspace_size)(len(F))
        self.ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        self.expect = self.call()
        torch.cuda.synchronize()
        if kind in ("fit", "large"):
            assert np.array_equal(self.expect[0].cpu().numpy(), oracle_lib.points_obb(p))
        else:
            build = oracle_lib.lbvh_build if kind == "lbvh" else oracle_lib.atrbvh_build
            assert np.array_equal(ops.nodes_to_numpy(self.expect[0]).view(np.uint8), build(V, F)[0].view(np.uint8))

    def call(self, stream=None):
        if self.kind in ("fit", "large"):
            return (ops.dito(*self.xyz, stream=stream, workspace=self.ws),)
        build = ops.lbvh_build if self.kind == "lbvh" else ops.atrbvh_build
        t = build(*self.mesh, stream=stream, workspace=self.ws)
        return t["nodes"], t["parents"], t["counts"], t["costs"]

    def check(self, got):
        return all(bool((bits(a) == bits(b)).all()) for a, b in zip(got, self.expect))


@pytest.mark.parametrize("kinds", [("fit", "fit"), ("large", "large"), ("lbvh", "lbvh"), ("atrbvh", "atrbvh"),
                                   ("fit", "large", "lbvh", "atrbvh")],
                         ids="-".join)
def test_handovers_on_several_streams(torch, oracle_lib, kinds):
    """Calls that hand over inside a launch, at the same time from a host thread and a stream each."""
    say(f"[handover] {kinds} at the same time")
    jobs = [Job(torch, oracle_lib, k, seed=20 + i) for i, k in enumerate(kinds)]
    streams = [torch.cuda.Stream() for _ in jobs]
    torch.cuda.synchronize()
    start, got, errors = threading.Barrier(len(jobs)), [[] for _ in jobs], []

    def run(i):
        try:
            start.wait()
            for _ in range(8):
                got[i].append(jobs[i].call(streams[i]))
        except Exception as e:  # reported from the main thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(jobs))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i, job in enumerate(jobs):
        for k, out in enumerate(got[i]):
            assert job.check(out), (i, k)


@pytest.mark.parametrize("kind", ["fit", "large", "lbvh", "atrbvh"])
def test_handovers_captured(torch, oracle_lib, kind):
    """The same calls captured in a HIP graph and replayed, with eager calls between the replays."""
    say(f"[handover] {kind} captured, 4 replays")
    job, other = Job(torch, oracle_lib, kind, seed=30), Job(torch, oracle_lib, kind, seed=31)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = job.call()
    torch.cuda.synchronize()
    for rep in range(4):
        for t in out:
            t.zero_()
        eager = other.call()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert job.check(out) and other.check(eager), rep
