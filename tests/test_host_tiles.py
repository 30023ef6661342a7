"""The run-length order of tile lists (nfx_order_tiles_host): the same tiles as nfx_build_tiles_host's, with
descending run lengths, run starts at odd distances and every corner in its node's run at its rank."""

import ctypes

import numpy as np
import pytest


def build(T, N, K):
    from nofluidx3d_amd import _lib

    vp = ctypes.c_void_p
    nT = len(T)
    tets = np.ascontiguousarray(T.reshape(-1, order="F").astype(np.uint32))
    ntiles = -(-nT // K)
    count = np.zeros(ntiles, np.uint32)
    m, mx = ctypes.c_int64(), ctypes.c_int32()
    head = (tets.ctypes.data_as(vp), N, nT, K, ctypes.byref(mx), ctypes.byref(m), count.ctypes.data_as(vp))
    _lib.call("nfx_build_tiles_host", *head, None, None, None, None, None)
    MX = mx.value
    lists = [np.zeros(ntiles * MX, np.uint32), np.zeros(ntiles * MX, np.uint16), np.zeros(4 * K * ntiles, np.uint16),
             np.zeros(ntiles * MX, np.uint32)]
    off = np.zeros(N + 1, np.uint32)
    _lib.call("nfx_build_tiles_host", *head, *[a.ctypes.data_as(vp) for a in lists], off.ctypes.data_as(vp))
    return MX, count, lists


# a full last tile, a last tile of one tetra, a mesh smaller than a tile, and one tetra
@pytest.mark.parametrize("K,keep", [(128, 640), (256, 513), (512, 100), (128, 1)])
def test_ordered_tile_lists(K, keep):
    from nofluidx3d_amd import _lib
    from nofluidx3d_amd.mesh import generate_sphere_mesh
    from nofluidx3d_amd.Simulation import order_tiles

    P, T = generate_sphere_mesh(3.0, 0.6, seed=4)
    T = T[:keep]
    MX, count, plain = build(T, len(P), K)
    lists = [a.copy() for a in plain]
    perm = order_tiles(K, MX, count, lists)
    for c in range(len(count)):
        M, nt = int(count[c]), min(K, len(T) - c * K)
        sl = slice(c * MX, c * MX + M)
        p = perm[c][:M].astype(int)
        assert sorted(p) == list(range(M))
        assert np.array_equal(lists[0][sl], plain[0][sl][p]) and np.array_equal(lists[3][sl], plain[3][sl][p])
        ends = plain[1][sl].astype(int)
        length = np.diff(np.concatenate([[0], ends]))[p]
        assert np.all(np.diff(length) <= 0)
        start = np.concatenate([[0], np.cumsum(length | 1)])[:-1]
        assert np.array_equal(lists[1][sl], start + length)
        assert lists[1][sl].max() <= 4 * K + min(K, 256)  # the corner slots the force pass holds
        # the start of run j from the end of run j - 1 and j's parity, as the force pass takes it
        before = np.concatenate([[0], lists[1][sl][:-1].astype(int)])
        assert np.array_equal(start, before + ((before ^ np.arange(M)) & 1))
        rec, old = lists[2][4 * K * c:4 * K * c + 4 * nt].astype(int), plain[2][4 * K * c:4 * K * c + 4 * nt].astype(int)
        assert np.array_equal(rec >> 8, old >> 8) and np.array_equal(p[rec & 0xFF], old & 0xFF)
        assert len(set(start[rec & 0xFF] + (rec >> 8))) == 4 * nt
    bad = [a.copy() for a in plain]
    bad[2][0] = MX  # a corner of a tile-node that the tile does not have
    vp = ctypes.c_void_p
    assert _lib.lib().nfx_order_tiles_host(len(count), K, MX, count.ctypes.data_as(vp), *[a.ctypes.data_as(vp) for a in bad],
                                           perm.ctypes.data_as(vp)) == -1
