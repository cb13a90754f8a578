"""Structure of the device-built trees at the sizes where the build's steps
change hands: one chunk and several (256 clusters), the last steps in one block
(2048 clusters), chunks of more than 256 (beyond 2048 * 256 clusters), a
frontier of several chunks, and degenerate inputs whose areas all tie."""
import dataclasses
import hashlib

import numpy as np
import pytest

import drawlab_amd
from drawlab_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(n, kind, seed=5):
    rng = np.random.default_rng(seed)
    d = scenes.cornell_box(16, 16)
    if kind == "same":      # every centroid in one Morton cell, every merged area equal
        p = np.tile(np.array([[[0, 0, 0], [1, 0, 0], [0, 1, 0]]], np.float32), (n, 1, 1))
    elif kind == "line":    # a geometric row: merges stay few per step
        x = np.cumsum(np.geomspace(1e-3, 1.0, n))[:, None, None].astype(np.float32)
        p = x * np.array([[[1, 0, 0]]], np.float32) + np.array([[[0, 0, 0], [0, 1e-3, 0], [0, 0, 1e-3]]], np.float32)
    else:
        p = (rng.random((n, 1, 3)) + rng.normal(scale=0.5 / max(1.0, n ** (1 / 3)), size=(n, 3, 3))).astype(np.float32)
    mesh = dataclasses.replace(d.meshes[0], V=np.ascontiguousarray(p.reshape(-1, 3)),
                               F=np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), N=None, UV=None)
    return dataclasses.replace(d, meshes=[mesh]), p


@pytest.mark.parametrize("kind,n", [("soup", 9), ("soup", 255), ("soup", 257), ("soup", 2048), ("soup", 2049),
                                    ("soup", 70_001), ("soup", 524_289), ("same", 3000), ("line", 2500)])
@pytest.mark.parametrize("builder", [drawlab_amd.BUILD_GPU, drawlab_amd.BUILD_GPU_LBVH])
def test_tree_structure(backend, kind, n, builder):
    d, p = _scene(n, kind)
    backend.upload_scene(d)
    st = backend.build_accel(builder)
    nodes, tris = backend.accel_export()
    nodes, tris = nodes.view(np.uint32).reshape(-1, 16), tris.reshape(-1, 12)
    prim = tris.view(np.uint32)[:, 9]
    assert np.array_equal(np.sort(prim), np.arange(n))             # every triangle once
    assert np.array_equal(tris[:, :3], p[prim, 0])
    ref = nodes[:, 12:16].view(np.int32)
    cnt = nodes[:, 10:11].view(np.uint8).reshape(-1, 4).astype(np.int64)
    inner = ref >= 0
    # breadth-first: the children's indices count up from 1 in node order
    assert np.array_equal(ref[inner], np.arange(1, len(nodes)))
    leaf = ~inner & (cnt > 0)
    first = np.where(leaf, ~ref, 0)
    covered = np.zeros(n + 1, np.int64)
    np.add.at(covered, first[leaf], 1)
    np.add.at(covered, first[leaf] + cnt[leaf], -1)
    assert np.array_equal(np.cumsum(covered)[:n], np.ones(n))      # leaves cover the triangles once
    # every child's decoded box holds its triangles, leaves to root
    origin = nodes[:, :3].view(np.float32)
    e = nodes[:, 3]
    step = np.stack([((e >> (8 * a)) & 0xff) << 23 for a in range(3)], 1).astype(np.uint32).view(np.float32)
    q = nodes[:, 4:10].view(np.uint8).reshape(-1, 3, 2, 4).astype(np.float32)
    lo = origin[:, :, None] + q[:, :, 0] * step[:, :, None]        # node, axis, child
    hi = origin[:, :, None] + q[:, :, 1] * step[:, :, None]
    tlo, thi = p[prim].min(axis=1), p[prim].max(axis=1)
    blo = np.full((len(nodes), 4, 3), np.inf, np.float32)
    bhi = np.full((len(nodes), 4, 3), -np.inf, np.float32)
    for k in range(int(cnt[leaf].max())):
        has = leaf & (cnt > k)
        blo[has] = np.minimum(blo[has], tlo[first[has] + k])
        bhi[has] = np.maximum(bhi[has], thi[first[has] + k])
    parent = np.zeros((len(nodes), 2), np.int64)
    parent[ref[inner]] = np.argwhere(inner)
    # parents come before their children: one pass per level from the last
    level = np.zeros(len(nodes), np.int64)
    for i in range(1, len(nodes)):
        level[i] = level[parent[i, 0]] + 1
    assert level.max() + 1 == st["max_depth"]
    for v in range(level.max(), 0, -1):
        at = np.flatnonzero(level == v)
        blo[parent[at, 0], parent[at, 1]] = blo[at].min(axis=1)
        bhi[parent[at, 0], parent[at, 1]] = bhi[at].max(axis=1)
    used = inner | leaf
    assert (lo.transpose(0, 2, 1)[used] <= blo[used]).all() and (hi.transpose(0, 2, 1)[used] >= bhi[used]).all()


# SHA-256 (first 16 digits) of the exported nodes and triangles, PLOC and LBVH,
# of the builders whose steps the host launched one by one with library scans
# between them: fewer and larger launches leave every byte as it was.
TREES = {
    "soup-9": ("0c4a1dc73e0aa9d8", "18ba1b4e7e996ac3"),
    "soup-255": ("4c08e36d1f0fba62", "ca0021fad5de6453"),
    "soup-257": ("685b9e4603452a56", "75fa0e0e8b6003de"),
    "soup-2048": ("b327bc6147fda240", "262c22878552a715"),
    "soup-2049": ("421529b5f4997111", "ddab6fd3cdb1d2c7"),
    "soup-70001": ("c670f20bdedaacb2", "853c65a496d8fcb3"),
    "soup-524289": ("f1edc21f0cc43ede", "4dadf7eea0295b00"),
    "same-3000": ("cfa0f083ca4491e5", "33ce0d44838c222f"),
    "line-2500": ("67d339405b4521f5", "828f32602ca334b6"),
    "sphere-8": ("0276451afcb8e95f", "08e188fd80ee6b6a"),
    "sphere-37": ("b4321f7103d3b854", "d1c520ee51a1eb00"),
    "sphere-200": ("20988c3307dcccff", "f27e261f7e5c5583"),
    "sphere-1024": ("6f8b5b153eed15fe", "5c1bfa94b567bfc7"),
    "zoo": ("5c172e9ced3fefc9", "3238c7d90a93664e"),
}


@pytest.mark.parametrize("name", sorted(TREES))
def test_trees_are_byte_for_byte_the_same(backend, name):
    kind, _, size = name.partition("-")
    if kind == "sphere":
        d = scenes.displaced_sphere(width=16, height=9, grid=int(size), glass_level=2, env_size=(8, 4))
    else:
        d = scenes.material_zoo() if kind == "zoo" else _scene(int(size), kind)[0]
    for builder, want in zip((drawlab_amd.BUILD_GPU, drawlab_amd.BUILD_GPU_LBVH), TREES[name]):
        backend.upload_scene(d)
        backend.build_accel(builder)
        nodes, tris = backend.accel_export()
        assert hashlib.sha256(nodes.tobytes() + tris.tobytes()).hexdigest()[:16] == want, builder
