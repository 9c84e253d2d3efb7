"""The mesh queries' leaf lists (rsg_mesh.h LeafGrid) against the tree walk
they stand in for: the same triangles in the same order for boxes and rays of
every size, inside and outside the mesh and the lists' grid, for vertices on
the query's very boundary, and for non-finite bounds, which the tree serves."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("leaf_lists") / "leaf_lists.so")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                        "-I" + os.path.join(ROOT, "include"), os.path.join(HERE, "cpp", "leaf_lists_host.cpp"),
                        "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    L = C.CDLL(out)
    L.ll_mesh.restype = C.c_void_p
    L.ll_mesh.argtypes = [C.c_char_p, C.c_uint64]
    L.ll_free.argtypes = [C.c_void_p]
    L.ll_bounds.argtypes = [C.c_void_p, C.c_void_p]
    L.ll_has_lists.argtypes = [C.c_void_p]
    for f in (L.ll_boxes, L.ll_rays):
        f.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.POINTER(C.c_long)]
    return L


def _meshes():
    from rocketsim_amd import arena_mesh
    return [("soccar", arena_mesh.soccar_cmf())] + [(f"hoops{i}", c) for i, c in enumerate(arena_mesh.hoops_cmfs())]


@pytest.mark.parametrize("name,cmf", _meshes(), ids=[n for n, _ in _meshes()])
def test_lists_report_what_the_tree_reports(lib, name, cmf):
    m = lib.ll_mesh(cmf, len(cmf))
    assert m
    try:
        assert lib.ll_has_lists(m) == 3
        b = np.zeros(6, np.float32)
        lib.ll_bounds(m, b.ctypes.data)
        nv = int(np.frombuffer(cmf, np.int32, 2)[1])
        verts = np.frombuffer(cmf, np.float32, 3 * nv, len(cmf) - 12 * nv).reshape(-1, 3)
        rng = np.random.default_rng(len(cmf))
        n = 6000
        # starts about the vertices (exactly on one, near one) and anywhere in and around the bounds
        at = verts[rng.integers(0, nv, n)].copy()
        near = rng.random(n) < 0.6
        at[near] += rng.normal(0, 1.5, (near.sum(), 3)).astype(np.float32)
        far = rng.random(n) < 0.15
        at[far] = rng.uniform(b[:3] - 6, b[3:] + 6, (far.sum(), 3))
        # boxes: a point, ordinary ones, the largest the lists serve, larger ones
        size = rng.uniform(0, 3.9, (n, 3)).astype(np.float32)
        size[rng.random(n) < 0.1] = 0
        size[rng.random(n) < 0.1] = 4.25
        size[rng.random(n) < 0.05] = 9.0
        lo = np.where(rng.random((n, 1)) < 0.5, at, at - size).astype(np.float32)
        boxes = np.ascontiguousarray(np.concatenate([lo, lo + size], 1), dtype=np.float32)
        boxes[:4, :] = [[np.nan] * 6, [0, 0, 0, np.inf, 1, 1], [-1e9, 0, 0, -1e9, 1, 1], [1e9, 0, 0, 1e9, 1, 1]]
        hits = C.c_long()
        served = lib.ll_boxes(m, n, boxes.ctypes.data, C.byref(hits))
        assert served >= 0, "a box's triangles differ"
        assert 0.8 * n < served < n and hits.value > n // 4
        # rays: suspension rays through and past the surface, long ones, a point
        d = rng.normal(0, 1, (n, 3))
        d = d / np.linalg.norm(d, axis=1, keepdims=True) * rng.uniform(0, 1.4, (n, 1))
        d[rng.random(n) < 0.2, 2] = 0     # axis-aligned: a zero direction component
        d[rng.random(n) < 0.05] *= 6
        d[rng.random(n) < 0.02] = 0
        rays = np.ascontiguousarray(np.concatenate([at - 0.5 * d, at + 0.5 * d], 1), dtype=np.float32)
        rays[:2, :] = [[np.nan] * 6, [0, 0, 0, 1e9, 0, 0]]
        hits = C.c_long()
        served = lib.ll_rays(m, n, rays.ctypes.data, C.byref(hits))
        assert served >= 0, "a ray's hits differ"
        assert 0.8 * n < served < n and hits.value > n // 20
    finally:
        lib.ll_free(m)
