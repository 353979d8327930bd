"""The vertex finder (csrc/kern_vertex.hip) on made-up tracks against the oracle, at the
counts where its sorts and its storage change: a wavefront's and a workgroup's worth of
tracks, the most that LDS holds and more, hundreds of vertices, pairs of close vertices that
the first fit merges and the split takes apart, outliers.  Vertex ids, degrees of freedom
and order are whole numbers and equal; the sums run in the same order on both sides, so
z, weight, chi2 and sum pt^2 are equal bit for bit."""
import ctypes as C
import os

import numpy as np
import pytest

from conftest import REPO

pytestmark = pytest.mark.gpu
LIB = os.path.join(REPO, "tests", "native", "libpxvertices_selftest.so")


def tracks(nt, vertices, rng):
    """nt tracks around the given number of vertices, a third of those in pairs 0.5 to 1 mm
    apart, a tenth of the tracks with errors too large to count neighbours."""
    zv = rng.uniform(-12, 12, vertices)
    pairs = vertices // 3
    zv[:pairs] = zv[vertices - pairs:] + rng.uniform(0.05, 0.1, pairs)
    ez = rng.uniform(0.003, 0.012, nt)
    z = zv[rng.integers(0, vertices, nt)] + rng.normal(0, 1, nt) * ez
    out = rng.random(nt) < 0.1
    z[out] += rng.normal(0, 0.05, out.sum())
    ez[out] *= 3
    return z.astype(np.float32), (ez * ez).astype(np.float32), rng.uniform(0.5, 5, nt).astype(np.float32)


@pytest.mark.parametrize("algo", [0, 1, 2])
@pytest.mark.parametrize("nt,vertices", [(0, 1), (1, 1), (2, 1), (63, 3), (65, 2), (1023, 30), (1025, 700),
                                         (2049, 40), (8192, 150), (8193, 150), (20000, 400)])
def test_made_up_tracks_match_oracle(oracle, algo, nt, vertices):
    lib = C.CDLL(LIB)
    vp = C.c_void_p
    lib.pxs_vertices.argtypes = [C.c_uint32, vp, vp, vp, C.c_int] + [vp] * 7
    z, ez2, pt = tracks(nt, vertices, np.random.default_rng(nt + vertices))
    if nt:
        o = oracle.vertices(z, ez2, pt * pt, algo)
    else:
        o = {"nv": 0}
    m = max(nt, 1)
    g = {"idv": np.zeros(m, np.int16), "ndof": np.zeros(m, np.int32)}
    for k in ("zv", "wv", "chi2", "ptv2"):
        g[k] = np.zeros(1024, np.float32)
    g["sortInd"] = np.zeros(1024, np.uint16)
    nv = lib.pxs_vertices(nt, z.ctypes.data, ez2.ctypes.data, pt.ctypes.data, algo, *[v.ctypes.data for v in g.values()])
    print(f"algo {algo}, {nt} tracks: {o['nv']} vertices", flush=True)
    assert nv == o["nv"]
    if nv == 0:
        return
    assert np.array_equal(g["idv"][:nt], o["iv"])
    for k in ("ndof", "sortInd"):
        assert np.array_equal(g[k][:nv], o[k]), k
    for k in ("zv", "wv", "chi2", "ptv2"):
        assert np.array_equal(g[k][:nv].view(np.uint32), o[k].view(np.uint32)), k
