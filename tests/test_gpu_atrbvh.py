"""GPU ATRBVH against the oracle: bit-exact nodes, parents, counts and costs
(topology, leaf order, bounds) for several meshes, treelet sizes and pass
counts, including duplicated geometry (tied codes and distances)."""
import sys

import numpy as np
import pytest

from obvh_amd import ops, synth

pytestmark = pytest.mark.gpu

CI, CT = 1.2, 1.0


@pytest.fixture(scope="module")
def torch():
    import torch as t

    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def mesh(kind):
    if kind == "ico":
        return synth.icosphere(20, seed=2)
    if kind == "hair":
        return synth.hairball(tubes=1500, seed=3)
    if kind == "dup":
        V, F = synth.icosphere(8, seed=4)
        return V, np.concatenate([F, F, F])
    if kind == "tiny":
        return synth.hairball(tubes=1, seed=5)
    if kind == "hair200k":
        return synth.hairball(tubes=5000, seed=6)
    if kind == "flat":  # a jittered grid in the plane z = 0.5: zero-thickness boxes, many tied costs
        n = 50
        rng = np.random.default_rng(7)
        g = np.stack(np.meshgrid(np.arange(n), np.arange(n), indexing="ij"), -1).reshape(-1, 2) + rng.uniform(
            -0.3, 0.3, (n * n, 2))
        V = np.concatenate([g / n, np.full((n * n, 1), 0.5)], 1).astype(np.float32)
        i, j = np.meshgrid(np.arange(n - 1), np.arange(n - 1), indexing="ij")
        a, b = (i * n + j).ravel(), (i * n + j + 1).ravel()
        c, d = ((i + 1) * n + j).ravel(), ((i + 1) * n + j + 1).ravel()
        F = np.concatenate([np.stack([a, b, c], 1), np.stack([b, d, c], 1)])
        return V, np.concatenate([F, np.zeros((len(F), 1), np.int64)], 1).astype(np.uint32)
    raise ValueError(kind)


@pytest.mark.parametrize("kind,ts,its", [("ico", 7, 2), ("hair", 7, 2), ("hair", 9, 2), ("dup", 7, 2),
                                         ("tiny", 7, 2), ("hair", 7, 0), ("hair200k", 7, 2), ("flat", 7, 2)])
def test_atrbvh_matches_oracle(torch, oracle_lib, kind, ts, its):
    say(f"[atrbvh] {kind} treelet={ts} passes={its}")
    V, F = mesh(kind)
    t = ops.atrbvh_build(torch.from_numpy(V).cuda(), torch.from_numpy(np.ascontiguousarray(F).view(np.int32)).cuda(),
                         ts, its, CI, CT)
    torch.cuda.synchronize()
    en, ep, ec, eco = oracle_lib.atrbvh_build(V, F, ts, its, CI, CT)
    nodes = ops.nodes_to_numpy(t["nodes"])
    assert np.array_equal(t["parents"].cpu().numpy().view(np.uint32), ep), "parents differ"
    assert np.array_equal(nodes.view(np.uint8), en.view(np.uint8)), "nodes differ"
    assert np.array_equal(t["counts"].cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(t["costs"].cpu().numpy(), eco)


@pytest.mark.parametrize("kind", ["hair", "flat"])
def test_atrbvh_then_transform_and_collapse(torch, oracle_lib, kind):
    say(f"[atrbvh] transform + collapse on the optimised tree ({kind})")
    V, F = mesh(kind)
    Vd = torch.from_numpy(V).cuda()
    Fd = torch.from_numpy(np.ascontiguousarray(F).view(np.int32)).cuda()
    t = ops.atrbvh_build(Vd, Fd, 7, 2, CI, CT)
    obbs, mats = ops.obb_tree(t["nodes"], t["parents"], Vd, Fd)
    col = ops.collapse(t["nodes"], t["parents"], t["counts"], CI, CT)
    torch.cuda.synchronize()
    nh = ops.nodes_to_numpy(t["nodes"])
    ph = t["parents"].cpu().numpy().view(np.uint32)
    eo, em = oracle_lib.obb_tree(nh, ph, V, F)
    assert np.array_equal(obbs.cpu().numpy(), eo) and np.array_equal(mats.cpu().numpy(), em)
    e = oracle_lib.collapse(nh, ph, t["counts"].cpu().numpy().view(np.uint32), CI, CT)
    assert np.array_equal(col["collapsed"].cpu().numpy(), e["collapsed"].view(np.uint8))


def edge_mesh(nf, kind):
    """nf triangles: small random ones, some stored several times (ties); `huge` scales them past 2^61
    (distances overflow), `flat` puts them in a plane with an integer grid (zero extents, equal areas)."""
    rng = np.random.default_rng(nf)
    c = rng.uniform(-1.0, 1.0, (nf, 1, 3))
    V = c + rng.uniform(-0.02, 0.02, (nf, 3, 3))
    if kind == "flat":
        V = np.round(V * 64.0)
        V[:, :, 2] = -0.0
    V[nf // 3:nf // 3 + nf // 8] = V[0]
    if kind == "huge":
        V = V * 2.0 ** 62
    F = np.zeros((nf, 4), dtype=np.uint32)
    F[:, :3] = np.arange(3 * nf).reshape(nf, 3)
    return V.reshape(-1, 3).astype(np.float32), F


# edges of the phases (512 leaves, one workgroup up to there; the top pass above), the smallest and largest treelets, distances
# past one entry per lane (treelet size 9 and up), boxes that take the general merge
@pytest.mark.parametrize("nf,ts,its,kind", [(1, 3, 1, "plain"), (2, 3, 1, "plain"), (3, 3, 2, "plain"),
                                            (20, 20, 1, "plain"), (512, 8, 2, "plain"), (513, 9, 2, "plain"),
                                            (1500, 20, 2, "plain"), (8193, 12, 3, "plain"), (3000, 3, 3, "flat"),
                                            (3000, 16, 2, "flat"), (2500, 9, 2, "huge"), (2500, 20, 2, "huge")])
def test_atrbvh_edges(torch, oracle_lib, nf, ts, its, kind):
    say(f"[atrbvh] {nf} triangles treelet={ts} passes={its} {kind}")
    V, F = edge_mesh(nf, kind)
    t = ops.atrbvh_build(torch.from_numpy(V).cuda(), torch.from_numpy(F.view(np.int32)).cuda(), ts, its, CI, CT)
    torch.cuda.synchronize()
    en, ep, ec, eco = oracle_lib.atrbvh_build(V, F, ts, its, CI, CT)
    assert np.array_equal(t["parents"].cpu().numpy().view(np.uint32), ep), "parents differ"
    assert np.array_equal(ops.nodes_to_numpy(t["nodes"]).view(np.uint8), en.view(np.uint8)), "nodes differ"
    assert np.array_equal(t["counts"].cpu().numpy().view(np.uint32), ec)
    assert np.array_equal(t["costs"].cpu().numpy(), eco, equal_nan=True)


# the pass between the tiles and the top, from 2^18 leaves on: both sides, several builds alike (the top pass hands nodes
# over between workgroups)
@pytest.mark.parametrize("nf", [262144, 262145])
def test_atrbvh_top_pass(torch, oracle_lib, nf):
    say(f"[atrbvh] top pass, {nf} triangles")
    V, F = edge_mesh(nf, "plain")
    Vd, Fd = torch.from_numpy(V).cuda(), torch.from_numpy(F.view(np.int32)).cuda()
    en, ep, ec, eco = oracle_lib.atrbvh_build(V, F, 7, 2, CI, CT)
    for _ in range(3):
        t = ops.atrbvh_build(Vd, Fd, 7, 2, CI, CT)
        torch.cuda.synchronize()
        assert np.array_equal(t["parents"].cpu().numpy().view(np.uint32), ep), "parents differ"
        assert np.array_equal(ops.nodes_to_numpy(t["nodes"]).view(np.uint8), en.view(np.uint8)), "nodes differ"
        assert np.array_equal(t["counts"].cpu().numpy().view(np.uint32), ec)
        assert np.array_equal(t["costs"].cpu().numpy(), eco)
