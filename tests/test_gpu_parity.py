"""GPU parity: every HIP entry point against the CPU oracle on the same
seeded inputs.  Integer/index results must be bit-exact; float results are
compared bit-exactly too (== on values, so -0 == +0), which is stricter than
the 1e-5 relative bound the path is specified to.  Full-size runs are
checked through size-independent properties (enclosure, determinism)."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from obvh_amd import ops, synth  # noqa: E402
from obvh_amd.layouts import NODE_DTYPE, TRACE_DTYPE  # noqa: E402
from treeutil import contiguous_tree, doubled_vertices, flat_grid, slivers  # noqa: E402


@pytest.fixture(scope="module")
def torch():
    import torch as t

    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def to_dev(torch, a, dtype=None):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def soa(torch, p):
    p = np.ascontiguousarray(p, np.float32)
    return [torch.from_numpy(np.ascontiguousarray(p[:, k])).cuda() for k in range(3)]


TRACE_INT_FIELDS = ["slab_min_idx", "slab_max_idx", "pair_k", "p2_sel", "q0_sel", "q1_sel", "q0_valid",
                    "q1_valid", "degenerate", "best", "result_aabb"]


def assert_trace_equal(got, exp):
    for f in TRACE_INT_FIELDS:
        assert np.array_equal(got[f], exp[f]), f


DITO_CASES = {
    "gaussian131072": lambda: synth.gaussian_points(131072, seed=1),
    "gaussian1000": lambda: synth.gaussian_points(1000, seed=2),
    "n1": lambda: np.array([[1.0, 2.0, 3.0]], np.float32),
    "n3": lambda: synth.gaussian_points(3, seed=3),
    "n14": lambda: synth.gaussian_points(14, seed=4),
    "n15": lambda: synth.gaussian_points(15, seed=5),
    "dups": lambda: (np.random.default_rng(6).integers(-8, 8, (5000, 3)) * 0.25).astype(np.float32),
    "line": lambda: (np.linspace(-1, 1, 777)[:, None] * np.array([0.3, -0.5, 0.8])).astype(np.float32),
    "point": lambda: np.tile(np.array([[0.5, 0.5, 0.5]], np.float32), (600, 1)),
    # coplanar points (a tilted plane through the origin, exact in float): no apex off the base triangle
    "plane": lambda: (np.random.default_rng(8).integers(-64, 64, (3000, 2)) @ np.array(
        [[0.5, 0.25, 0.0], [0.0, 0.5, 0.25]])).astype(np.float32),
    "ragged": lambda: synth.gaussian_points(512 * 7 + 13, seed=7),
}


@pytest.mark.parametrize("case", sorted(DITO_CASES))
def test_dito_soa_matches_oracle(torch, oracle_lib, case):
    say(f"[dito_soa] case={case}")
    p = DITO_CASES[case]()
    exp, etr = oracle_lib.points_obb(p, trace=True)
    x, y, z = soa(torch, p)
    out, tr = ops.dito(x, y, z, trace=True)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.array_equal(got, exp), (got, exp)
    assert_trace_equal(ops.trace_to_numpy(tr)[0], etr)


@pytest.mark.parametrize("case", ["gaussian131072", "n3", "dups", "point"])
def test_legacy_points_obb_matches_oracle(torch, oracle_lib, case):
    say(f"[kr_cuda_points_obb] case={case}")
    p = DITO_CASES[case]()
    got, ms = ops.points_obb(p, return_time=True)
    assert np.array_equal(got, oracle_lib.points_obb(p))
    assert ms >= 0.0


@pytest.mark.parametrize("tile", [0, 512, 4096])
def test_dito_batch_matches_oracle(torch, oracle_lib, tile):
    say(f"[dito_batch] tile={tile}")
    sizes = np.concatenate([[0, 1, 2, 14, 15, 64, 513], synth.batch_sizes(120, lo=64, hi=1 << 15, seed=9)])
    pts, off = synth.batch_sets(sizes, seed=10)
    exp, etr = oracle_lib.points_obb_batch(pts, off)
    x, y, z = soa(torch, pts)
    offs = torch.from_numpy(off.astype(np.int64)).cuda()
    out, tr = ops.dito_batch(x, y, z, offs, tile_points=tile, trace=True)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    gtr = ops.trace_to_numpy(tr)[: len(sizes)]
    for s in range(len(sizes)):
        assert np.array_equal(got[s], exp[s]), (s, sizes[s])
        assert_trace_equal(gtr[s], etr[s])


def build_gpu_tree(torch, V, F):
    Vd = torch.from_numpy(V).cuda()
    Fd = torch.from_numpy(F.view(np.int32)).cuda()
    t = ops.lbvh_build(Vd, Fd)
    return Vd, Fd, t


MESHES = {
    "ico16": lambda: synth.icosphere(16, seed=1),
    "flat": lambda: flat_grid(60, seed=9),
    "dupverts": lambda: doubled_vertices(seed=10),
    "slivers": lambda: slivers(seed=11),
    "ico_n256": lambda: synth.icosphere(8, seed=2),  # 1280 faces = 5 * 256
    "hair200": lambda: synth.hairball(tubes=200, seed=3),
    "single": lambda: (np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32),
                       np.array([[0, 1, 2, 0]], np.uint32)),
    "two": lambda: (np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32),
                    np.array([[0, 1, 2, 0], [0, 1, 3, 0]], np.uint32)),
}


@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_lbvh_matches_oracle(torch, oracle_lib, mesh):
    say(f"[lbvh] mesh={mesh}")
    V, F = MESHES[mesh]()
    Vd, Fd, t = build_gpu_tree(torch, V, F)
    torch.cuda.synchronize()
    en, ep, ec, eco, em = oracle_lib.lbvh_build(V, F)
    gn = ops.nodes_to_numpy(t["nodes"])
    assert np.array_equal(t["mortons"].cpu().numpy().view(np.uint32), em)
    assert np.array_equal(t["parents"].cpu().numpy().view(np.uint32), ep)
    assert np.array_equal(t["counts"].cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(t["costs"].cpu().numpy(), eco)
    for f in ("bmin", "bmax", "a", "nprim", "axis"):
        assert np.array_equal(gn[f], en[f]), f
    I = len(F) - 1
    assert np.array_equal(gn["b"][:I], en["b"][:I])


@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_obb_tree_matches_oracle(torch, oracle_lib, mesh):
    say(f"[obb_tree] mesh={mesh}")
    V, F = MESHES[mesh]()
    Vd, Fd, t = build_gpu_tree(torch, V, F)
    obbs, mats, ids = ops.obb_tree(t["nodes"], t["parents"], Vd, Fd, with_ids=True)
    torch.cuda.synchronize()
    nodes = ops.nodes_to_numpy(t["nodes"])
    parents = t["parents"].cpu().numpy().view(np.uint32)
    eo, em, ei = oracle_lib.obb_tree(nodes, parents, V, F, with_ids=True)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), ei)
    go, gm = obbs.cpu().numpy(), mats.cpu().numpy()
    # equal, or NaN in both (a zero-area leaf triangle's frame is NaN in the
    # reference's leaf OBB as well)
    bad = np.where(~np.all((go == eo) | (np.isnan(go) & np.isnan(eo)), axis=1))[0]
    assert bad.size == 0, (bad[:10], go[bad[:3]], eo[bad[:3]])
    assert np.all((gm == em) | (np.isnan(gm) & np.isnan(em)))
    if mesh != "slivers":
        assert not np.isnan(go).any()


def test_legacy_obb_tree_equals_async(torch, oracle_lib):
    say("[kr_cuda_bvh_obb_tree] ico16")
    V, F = synth.icosphere(16, seed=4)
    Vd, Fd, t = build_gpu_tree(torch, V, F)
    total = 2 * len(F) - 1
    o1 = torch.zeros((total, 15), dtype=torch.float32, device="cuda")
    m1 = torch.zeros((total, 16), dtype=torch.float32, device="cuda")
    ops.bvh_obb_tree(t["nodes"], t["parents"], Vd, Fd, o1, m1, len(F), len(F) - 1,
                     primitive_counts=t["counts"], costs=t["costs"])
    o2, m2 = ops.obb_tree(t["nodes"], t["parents"], Vd, Fd)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(m1, m2)


def test_legacy_obb_tree_rejects_malformed_parents(torch):
    say("[kr_cuda_bvh_obb_tree] malformed parents")
    V, F = synth.icosphere(4, seed=5)
    Vd, Fd, t = build_gpu_tree(torch, V, F)
    parents = t["parents"].clone()
    parents[7] = 3  # disagrees with the children of node 3 (bounds stay valid)
    total = 2 * len(F) - 1
    o = torch.zeros((total, 15), dtype=torch.float32, device="cuda")
    m = torch.zeros((total, 16), dtype=torch.float32, device="cuda")
    from obvh_amd._lib import ObvhError

    with pytest.raises(ObvhError):
        ops.bvh_obb_tree(t["nodes"], parents, Vd, Fd, o, m, len(F), len(F) - 1)


def test_full_size_transform_properties(torch, oracle_lib):
    # 1 003 520-triangle icosphere (f = 224): determinism across runs and
    # parity with the oracle on the whole tree (the oracle takes seconds).
    say("[obb_tree] ico224 full size")
    V, F = synth.icosphere(224, seed=2)
    Vd, Fd, t = build_gpu_tree(torch, V, F)
    o1, m1 = ops.obb_tree(t["nodes"], t["parents"], Vd, Fd)
    o2, m2 = ops.obb_tree(t["nodes"], t["parents"], Vd, Fd)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(m1, m2)
    nodes = ops.nodes_to_numpy(t["nodes"])
    parents = t["parents"].cpu().numpy().view(np.uint32)
    en, ep, *_ = oracle_lib.lbvh_build(V, F)
    assert np.array_equal(parents, ep)
    eo, em = oracle_lib.obb_tree(nodes, parents, V, F)
    go = o1.cpu().numpy()
    mism = int((~np.all(go == eo, axis=1)).sum())
    assert mism == 0, mism
    assert np.array_equal(m1.cpu().numpy(), em)


def random_tree(n_leaves: int, seed: int):
    """Random binary tree over shuffled leaves: internal nodes numbered in
    breadth-first order (root 0), leaves I..2N-2 holding a random face
    permutation.  Sibling leaves are rarely adjacent, so the bottom-up
    kernels exchange most k-DOPs across workgroups."""
    rng = np.random.default_rng(seed)
    I = n_leaves - 1
    nodes = np.zeros(2 * n_leaves - 1, dtype=NODE_DTYPE)
    parents = np.zeros(2 * n_leaves - 1, dtype=np.uint32)
    parents[0] = 0xFFFFFFFF
    leaf_slots = rng.permutation(n_leaves)  # leaf slot of each face
    queue = [(0, np.arange(n_leaves))]
    next_internal = 1
    head = 0
    while head < len(queue):
        idx, faces = queue[head]
        head += 1
        cut = int(rng.integers(1, len(faces)))
        kids = []
        for part in (faces[:cut], faces[cut:]):
            if len(part) == 1:
                kids.append(I + int(leaf_slots[part[0]]))
            else:
                kids.append(next_internal)
                queue.append((next_internal, part))
                next_internal += 1
        nodes[idx]["a"], nodes[idx]["b"] = kids
        for k in kids:
            parents[k] = idx
    for f in range(n_leaves):
        L = nodes[I + leaf_slots[f]]
        L["a"] = f
        L["nprim"] = 1
    return nodes, parents


@pytest.mark.parametrize("n", [5000, 20000, 100000])
def test_obb_tree_random_topology(torch, oracle_lib, n):
    """n = 100 000 spans four 32768-leaf chunks: nearly every node has leaves
    in several workgroups, so the climb defers most parents across workgroups,
    folds split pairs into the global arrival words, overflows the last
    phase's LDS slots into global arrivals, and the refit's tiles have
    gapped ancestors everywhere."""
    say(f"[obb_tree] random topology n={n}")
    V, F = synth.hairball(tubes=n // 40 + 1, seed=6)
    F = F[:n]
    nodes, parents = random_tree(n, seed=n)
    Vd = torch.from_numpy(V).cuda()
    Fd = torch.from_numpy(np.ascontiguousarray(F).view(np.int32)).cuda()
    nd = torch.from_numpy(nodes.view(np.uint8)).cuda()
    pd = torch.from_numpy(parents.view(np.int32)).cuda()
    obbs, mats, ids = ops.obb_tree(nd, pd, Vd, Fd, with_ids=True)
    torch.cuda.synchronize()
    eo, em, ei = oracle_lib.obb_tree(nodes, parents, V, F, with_ids=True)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), ei)
    assert np.array_equal(obbs.cpu().numpy(), eo)
    assert np.array_equal(mats.cpu().numpy(), em)


@pytest.mark.parametrize("n,spine", [(30000, 0), (81920, 512), (81920, 384), (40000, 16)])
def test_obb_tree_contiguous_topology(torch, oracle_lib, n, spine):
    """Trees whose subtrees hold contiguous leaf runs but whose internal nodes
    are numbered breadth-first (not Karras): the refit's LDS copy of the
    tile's index range mostly misses.  spine=512: the leftmost tile has 127
    ancestors holding it, more than the 64 listed per tile, so the rest are
    walked by every wave; spine=384: 171.  spine=16: a 2000-deep spine
    whose nodes mostly span more than one 32768-leaf chunk, so the
    top-of-tree climb phases walk long chains."""
    say(f"[obb_tree] contiguous topology n={n} spine={spine}")
    V, F = synth.hairball(tubes=n // 40 + 1, seed=7)
    F = F[:n]
    nodes, parents = contiguous_tree(n, seed=n, spine_block=spine)
    Vd = torch.from_numpy(V).cuda()
    Fd = torch.from_numpy(np.ascontiguousarray(F).view(np.int32)).cuda()
    nd = torch.from_numpy(nodes.view(np.uint8)).cuda()
    pd = torch.from_numpy(parents.view(np.int32)).cuda()
    obbs, mats, ids = ops.obb_tree(nd, pd, Vd, Fd, with_ids=True)
    torch.cuda.synchronize()
    eo, em, ei = oracle_lib.obb_tree(nodes, parents, V, F, with_ids=True)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), ei)
    assert np.array_equal(obbs.cpu().numpy(), eo)
    assert np.array_equal(mats.cpu().numpy(), em)


# edges of the climb's forms: one 512-leaf tile (nothing above it), the first sizes with a top of the tree, more paths
# than one wave takes at once, and both sides of the size from which the search runs on two streams; eager and captured
@pytest.mark.parametrize("kind,n", [("random", 512), ("random", 513), ("contiguous", 1025), ("random", 9000),
                                    ("contiguous", 262144), ("contiguous", 262145)])
def test_obb_tree_climb_edges(torch, oracle_lib, kind, n):
    say(f"[obb_tree] climb edges {kind} n={n}")
    V, F = synth.hairball(tubes=n // 40 + 1, seed=11)
    F = F[:n]
    nodes, parents = random_tree(n, seed=n) if kind == "random" else contiguous_tree(n, seed=n)
    a = (torch.from_numpy(nodes.view(np.uint8)).cuda(), torch.from_numpy(parents.view(np.int32)).cuda(),
         torch.from_numpy(V).cuda(), torch.from_numpy(np.ascontiguousarray(F).view(np.int32)).cuda())
    obbs, mats, ids = ops.obb_tree(*a, with_ids=True)
    torch.cuda.synchronize()
    eo, em, ei = oracle_lib.obb_tree(nodes, parents, V, F, with_ids=True)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), ei)
    assert np.array_equal(obbs.cpu().numpy(), eo)
    assert np.array_equal(mats.cpu().numpy(), em)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = ops.obb_tree(*a, with_ids=True)
    for _ in range(3):
        for x in captured:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x.view(torch.int32), y.view(torch.int32)) for x, y in zip(captured, (obbs, mats, ids)))


def renumber(nodes, parents, perm, lperm):
    """The same tree with internal node i stored at perm[i] (perm[0] = 0) and
    the leaf at position j stored at position lperm[j]."""
    n = len(lperm)
    I = n - 1
    old2new = np.concatenate([perm, I + lperm]).astype(np.int64)
    new_nodes = np.zeros_like(nodes)
    new_parents = np.zeros_like(parents)
    new_nodes[old2new] = nodes
    for i in range(I):
        j = old2new[i]
        new_nodes[j]["a"] = old2new[nodes[i]["a"]]
        new_nodes[j]["b"] = old2new[nodes[i]["b"]]
    p = parents.astype(np.int64)
    new_parents[old2new] = np.where(p == 0xFFFFFFFF, 0xFFFFFFFF, old2new[np.minimum(p, 2 * n - 2)]).astype(np.uint32)
    return new_nodes, new_parents, old2new


@pytest.mark.parametrize("mesh,builder", [("ico", "lbvh"), ("hair", "atrbvh")])
def test_obb_tree_renumbering_canary(torch, oracle_lib, mesh, builder):
    """Determinism canary: the same tree stored with its internal nodes in a
    random order and its leaf slots reversed.  Every tile, chunk, workgroup
    and lane assignment of the climb, the candidate search and the refit
    changes (and the spans get gaps everywhere), so any result that
    depended on scheduling would move; every box and matrix, mapped back,
    must be bit-identical to the original tree's."""
    say(f"[obb_tree] renumbering canary {mesh} {builder}")
    V, F = synth.icosphere(48, seed=11) if mesh == "ico" else synth.hairball(tubes=1500, seed=12)
    if builder == "lbvh":
        nodes, parents, *_ = oracle_lib.lbvh_build(V, F)
    else:
        nodes, parents, *_ = oracle_lib.atrbvh_build(V, F, 7, 2)
    n = F.shape[0]
    rng = np.random.default_rng(n)
    perm = np.concatenate([[0], 1 + rng.permutation(n - 2)])
    lperm = np.arange(n)[::-1].copy()
    nn, npar, old2new = renumber(nodes, parents, perm, lperm)
    Vd = torch.from_numpy(V).cuda()
    Fd = torch.from_numpy(np.ascontiguousarray(F).view(np.int32)).cuda()
    outs = []
    for nd_, pr_ in ((nodes, parents), (nn, npar)):
        o, m = ops.obb_tree(torch.from_numpy(np.ascontiguousarray(nd_).view(np.uint8)).cuda(),
                            torch.from_numpy(np.ascontiguousarray(pr_).view(np.int32)).cuda(), Vd, Fd)
        torch.cuda.synchronize()
        outs.append((o.cpu().numpy(), m.cpu().numpy()))
    (o0, m0), (o1, m1) = outs
    assert np.array_equal(o1[old2new], o0)
    assert np.array_equal(m1[old2new], m0)
    eo, em = oracle_lib.obb_tree(nodes, parents, V, F)
    assert np.array_equal(o0, eo) and np.array_equal(m0, em)


def tied_points(n, seed):
    """n points whose extremes are reached several times: small integers, with the last point a copy of an
    extreme one, and a run of equal points."""
    rng = np.random.default_rng(seed)
    p = rng.integers(-40, 41, (n, 3)).astype(np.float32)
    p[n // 2:n // 2 + n // 5] = p[0]
    p[-1] = p[int(np.argmax(p[:, 0]))]
    return p


# both sides of the batch sizes whose tile table the set-up writes (1024 sets, 16384 tiles), empty sets at either end
@pytest.mark.parametrize("nsets,tile,big", [(1, 0, 40), (64, 0, 40), (1024, 0, 40), (1025, 0, 40), (200, 512, 8340000),
                                            (200, 512, 8350000)])
def test_dito_batch_table_edges(torch, oracle_lib, nsets, tile, big):
    say(f"[dito_batch] table edges {nsets} sets, tile={tile}, {big}")
    rng = np.random.default_rng(nsets + big)
    sizes = rng.integers(0, 60, nsets)
    sizes[[0, -1]] = 0
    sizes[nsets // 2] = big
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    p = rng.standard_normal((int(off[-1]), 3)).astype(np.float32)
    out = ops.dito_batch(*soa(torch, p), torch.from_numpy(off).cuda(), tile_points=tile)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), oracle_lib.points_obb_batch(p, off, threads=8)[0], equal_nan=True)


# host fits on both sides of the size up to which the points go through pinned memory (512 KB); repeated with other points
# in the same buffers, and from device memory
@pytest.mark.parametrize("n", [1, 43690, 43691])
def test_points_obb_staging(torch, oracle_lib, n):
    say(f"[points_obb] n={n}")
    for seed in (1, 2):
        p = synth.gaussian_points(n, seed=seed)
        want = oracle_lib.points_obb(p)
        assert np.array_equal(ops.points_obb(p), want, equal_nan=True)
        d = torch.from_numpy(p).cuda()
        o = ops.lib().kr_cuda_points_obb(ops.C.c_void_p(d.data_ptr()), n, None)
        assert np.array_equal(np.frombuffer(o, np.float32), want, equal_nan=True)


# edges of the single fit's forms: one workgroup (8192 points), tiles of 2048 that wait for each other (up to 128),
# two launches above; of a tile's rows and steps
@pytest.mark.parametrize("n", [1, 255, 1024, 1025, 2049, 8191, 8192, 8193, 10240, 10241, 262144, 262145, 300001])
@pytest.mark.parametrize("kind", ["gaussian", "tied", "nan"])
def test_dito_single_forms(torch, oracle_lib, n, kind):
    say(f"[dito_soa] n={n} {kind}")
    p = tied_points(n, n) if kind == "tied" else synth.gaussian_points(n, seed=n)
    if kind == "nan":
        p[n // 2::7] = np.nan
        p[n // 3, 1] = np.inf
    exp, etr = oracle_lib.points_obb(p, trace=True)
    x, y, z = soa(torch, p)
    ws = torch.full((int(ops.lib().obvh_dito_workspace_size(n)),), 0x5A, dtype=torch.uint8, device="cuda")
    for _ in range(2):  # the second call on what the first left in the workspace
        out, tr = ops.dito(x, y, z, trace=True, workspace=ws)
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), exp, equal_nan=True), (out.cpu().numpy(), exp)
        assert_trace_equal(ops.trace_to_numpy(tr)[0], etr)
    if n <= 262145:
        assert np.array_equal(ops.points_obb(p), oracle_lib.points_obb(p), equal_nan=True)


# tiles of one step and more, remainders of a wave's 512 points, every alignment of a set's first point
@pytest.mark.parametrize("tile", [0, 512, 2048, 32768])
def test_dito_batch_tile_edges(torch, oracle_lib, tile):
    say(f"[dito_batch] tile edges, tile={tile}")
    sizes = np.array([1, 3, 511, 512, 513, 1, 2047, 2048, 2049, 4097, 2, 6145, 32767, 32769, 70001], dtype=np.int64)
    pts = np.concatenate([tied_points(int(n), 5 + k) if k % 2 else synth.gaussian_points(int(n), seed=k)
                          for k, n in enumerate(sizes)])
    pts[600:5000:97, 2] = np.nan
    off = np.concatenate([[0], np.cumsum(sizes)])
    exp, etr = oracle_lib.points_obb_batch(pts, off.astype(np.uint64))
    x, y, z = soa(torch, pts)
    out, tr = ops.dito_batch(x, y, z, torch.from_numpy(off).cuda(), tile_points=tile, trace=True)
    torch.cuda.synchronize()
    gtr = ops.trace_to_numpy(tr)
    for s in range(len(sizes)):
        assert np.array_equal(out[s].cpu().numpy(), exp[s], equal_nan=True), (s, sizes[s])
        assert_trace_equal(gtr[s], etr[s])


def test_dito_batch_overlapping_sets(torch, oracle_lib):
    """Offsets that go back make sets overlap: the sets that fit the tile table keep their boxes, those beyond it and
    the decreasing ones are invalid (NaN, degenerate 4)."""
    say("[dito_batch] overlapping sets")
    n = 5 * 512
    p = synth.gaussian_points(n, seed=3)
    x, y, z = soa(torch, p)
    off = torch.tensor([0, n, 0, n, 0, n, 0, n], dtype=torch.int64).cuda()  # 20 tiles, the table has 13
    out, tr = ops.dito_batch(x, y, z, off, tile_points=512, trace=True)
    torch.cuda.synchronize()
    got, g = out.cpu().numpy(), ops.trace_to_numpy(tr)
    exp = oracle_lib.points_obb(p)
    assert np.array_equal(got[0], exp) and np.array_equal(got[2], exp)
    for s in (1, 3, 4, 5, 6):
        assert np.isnan(got[s]).all() and g[s]["degenerate"] == 4, s


# the sort's forms and tiles (one workgroup up to 4096 faces; 1, 2 and 4 faces per thread), few distinct codes
@pytest.mark.parametrize("nf", [1023, 1024, 1025, 2049, 4096, 4097, 32768, 32769, 70000, 131073])
@pytest.mark.parametrize("cells", [3, 1000])
def test_lbvh_sort_edges(torch, oracle_lib, nf, cells):
    say(f"[lbvh] sort: {nf} faces over {cells} positions per axis")
    rng = np.random.default_rng(nf)
    c = np.floor(rng.uniform(0, 1, (nf, 1, 3)) * cells) / cells
    V = (c + rng.uniform(0, 1e-4, (nf, 3, 3))).reshape(-1, 3).astype(np.float32)
    F = np.zeros((nf, 4), dtype=np.uint32)
    F[:, :3] = np.arange(3 * nf).reshape(nf, 3)
    t = ops.lbvh_build(torch.from_numpy(V).cuda(), torch.from_numpy(F.view(np.int32)).cuda())
    torch.cuda.synchronize()
    nodes, parents, counts, costs, mortons = oracle_lib.lbvh_build(V, F)
    assert np.array_equal(t["mortons"].cpu().numpy().view(np.uint32), mortons)
    assert np.array_equal(t["parents"].cpu().numpy().view(np.uint32), parents)
    assert np.array_equal(ops.nodes_to_numpy(t["nodes"]).view(np.uint8), nodes.view(np.uint8))
    assert np.array_equal(t["counts"].cpu().numpy().view(np.uint32), counts)
    assert np.array_equal(t["costs"].cpu().numpy(), costs)


def test_dito_batch_overlapping_sets_that_just_fit(torch, oracle_lib):
    """Overlapping sets that need exactly as many tiles as the workspace holds (13) keep their boxes; one point more
    needs a 14th and makes the last of them invalid."""
    say("[dito_batch] overlapping sets, a full tile table")
    n = 5 * 512
    p = synth.gaussian_points(n, seed=3)
    x, y, z = soa(torch, p)
    exp = oracle_lib.points_obb(p)
    for last, fits in ((1536, True), (1537, False)):
        off = torch.tensor([0, n, 0, n, 0, last, 0, 0], dtype=torch.int64).cuda()  # 5 + 5 + 3 tiles, or + 4
        out, tr = ops.dito_batch(x, y, z, off, tile_points=512, trace=True)
        torch.cuda.synchronize()
        got, g = out.cpu().numpy(), ops.trace_to_numpy(tr)
        assert np.array_equal(got[0], exp) and np.array_equal(got[2], exp)
        if fits:
            assert np.array_equal(got[4], oracle_lib.points_obb(p[:last]))
        else:
            assert np.isnan(got[4]).all() and g[4]["degenerate"] == 4
        for s in (1, 3, 5):
            assert np.isnan(got[s]).all() and g[s]["degenerate"] == 4, s


def test_dito_batch_overlapping_sets_past_2_to_32_tiles(torch, oracle_lib):
    """Overlapping sets that ask for more than 2^32 tiles in all: those the table holds keep their boxes, all others are
    invalid (the sums of tiles do not wrap)."""
    say("[dito_batch] overlapping sets, 2^32 tiles")
    n = 1 << 22                      # 8192 tiles a set
    pairs = (1 << 19) + 200          # 2^32 tiles and some more
    nsets = 2 * pairs - 1
    p = synth.gaussian_points(n, seed=4)
    x, y, z = soa(torch, p)
    off = torch.tensor([0, n], dtype=torch.int64).repeat(pairs).cuda()
    out = ops.dito_batch(x, y, z, off, tile_points=512).cpu().numpy()
    fit = (n // 512 + nsets + 1) // 8192  # sets that fit the table
    exp = oracle_lib.points_obb(p)
    assert (out[0:2 * fit:2] == exp).all()
    assert np.isnan(out[1:2 * fit:2]).all() and np.isnan(out[2 * fit:]).all()


@pytest.mark.parametrize("nf", [1250000, 1250001])
def test_lbvh_sort_eight_per_thread(torch, oracle_lib, nf):
    """The largest count with four pairs per thread, and the smallest with eight."""
    test_lbvh_sort_edges(torch, oracle_lib, nf, 1000)
