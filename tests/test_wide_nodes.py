"""The traversal's wide nodes (four quantised boxes, two levels of the binary
tree) against the binary traversal on the CPU and against the oracle on the
GPU, at the sizes and inputs where they can go wrong."""
import os
import subprocess

import numpy as np
import pytest
import torch

import oracle_lib as orc
from fledge_amd import api

HERE = os.path.dirname(os.path.abspath(__file__))


def test_wide_nodes_host():
    """wide_test: bit-equal hits on wide and binary nodes for 1.9 M rays through
    vertices, along edges and faces, axis-parallel and on box planes."""
    exe = os.path.join(HERE, "cpp", "build", "wide_test")
    if not os.path.exists(exe):
        subprocess.run(["make", "-s", "-C", os.path.join(HERE, "cpp"), "build/wide_test"], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and "ALL PASSED" in r.stdout


def _lattice(n):
    """n x n unit squares in the plane z = 0, two triangles each."""
    y, x = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    x, y = x.ravel(), y.ravel()
    c = np.stack([np.stack([x + a, y + b, 0 * x], 1) for a, b in ((0, 0), (1, 0), (1, 1), (0, 1))], 1)
    ind = 4 * np.arange(n * n)[:, None] + np.array([0, 1, 2, 0, 2, 3])
    return c.reshape(-1).astype(np.float32), ind.reshape(-1).astype(np.int32)


def _rays(v, n, seed):
    rng = np.random.default_rng(seed)
    p = v.reshape(-1, 3)
    lo, ext = p.min(0), np.ptp(p, axis=0)
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = lo + ext * (rng.random((n, 3)) * 1.6 - 0.3)
    d = rng.normal(size=(n, 3))
    k = np.arange(n) % 4
    d[k == 1] = (p[rng.integers(len(p), size=n)] - r[:, 0:3])[k == 1]  # through vertices
    r[k == 2, 0:3] = p[rng.integers(len(p), size=n)][k == 2]  # from vertices
    d[k == 3] *= rng.integers(0, 2, size=(n, 3))[k == 3]  # zeros in the direction
    d[np.linalg.norm(d, axis=1) == 0] = (0, 0, 1)
    r[:, 4:7] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    r[:, 3] = np.where(np.arange(n) % 3 == 0, 0.5 * np.linalg.norm(ext), np.inf)
    return r


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", ["soup2", "soup5", "soup1023", "soup1024", "soup1025", "soup2049", "lattice40",
                                  "far", "huge"])
def test_wide_nodes_gpu(ctx, mesh):
    """Ids and t bit-equal to the oracle: chunk edges of the builder (1024
    leaves), boxes flat in an axis, coordinates where rounding is coarse, and the
    meshes that keep the binary nodes (coordinates beyond 2^40)."""
    print("wide nodes %s" % mesh, flush=True)
    if mesh.startswith("soup"):
        v, i = api.gen_soup(int(mesh[4:]))
    elif mesh.startswith("lattice"):
        v, i = _lattice(int(mesh[7:]))
    else:
        v, i = api.gen_soup(3000)
        if mesh == "far":
            v = (v * np.float32(1e-3) + np.float32(1000.0)).astype(np.float32)
        if mesh == "huge":
            v = (v * np.float32(2.0 ** 42)).astype(np.float32)
    g, o = api.LBVH.build(ctx, torch.from_numpy(v).cuda(), torch.from_numpy(i).cuda()), orc.Lbvh(v, i)
    rays = _rays(v, 20000, 3)
    for n in (1, 63, 20000):
        gid, gt = api.hits_as_numpy(g.trace(torch.from_numpy(rays[:n]).cuda()))
        oid, ot = o.trace(rays[:n])
        assert np.array_equal(gid, oid)
        assert np.array_equal(gt.view(np.uint32), ot.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_unbounded_vertices(ctx, value):
    """Meshes with a vertex that is not finite, alone and in a batch with finite
    ones (each mesh of a batch picks its nodes for itself): ids and t bit-equal to
    the oracle's binary traversal."""
    print("unbounded vertices %r" % value, flush=True)
    sizes, bad = (1500, 700, 2049, 1), (1, 2)
    meshes = [api.gen_soup(n, initseq=60 + k) for k, n in enumerate(sizes)]
    for k in bad:
        meshes[k][0][9 * (sizes[k] // 2) + 4] = value
    up = [(torch.from_numpy(v).cuda(), torch.from_numpy(i).cuda()) for v, i in meshes]
    rays = _rays(meshes[0][0], 8000, 5)
    for k, b in enumerate(api.LBVH.build_batched(ctx, up)):
        alone = api.LBVH.build(ctx, *up[k])
        oid, ot = orc.Lbvh(*meshes[k]).trace(rays)
        for g in (b, alone):
            gid, gt = api.hits_as_numpy(g.trace(torch.from_numpy(rays).cuda()))
            assert np.array_equal(gid, oid)
            assert np.array_equal(gt.view(np.uint32), ot.view(np.uint32))
        assert sizes[k] == 1 or (oid >= 0).any()  # the small triangle lies off every ray


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 1500])
def test_device_bytes(ctx, n):
    """flg_lbvh_info.device_bytes counts every array of the build: 48 bytes of
    triangle and 20 of leaf arrays a triangle; 64 of binary node, 64 of wide node
    and 17 of node arrays a node."""
    v, i = api.gen_soup(n)
    b = api.LBVH.build(ctx, torch.from_numpy(v).cuda(), torch.from_numpy(i).cuda())
    assert b.info().device_bytes == 68 * n + 145 * (n - 1)
