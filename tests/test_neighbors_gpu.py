"""The GPU radius graph (``fsctep_amd.neighbors``, cell list in ``csrc/neighbors.hip``) against the host
list of ``fsctep_amd.synthetic.radius_graph`` (scipy cKDTree, minimum image) and against a brute-force
numpy statement of the reference semantics (utils/graph_utils.py:192-257: every image s in {-1,0,1} on
periodic axes, |pos[j] + s @ cell - pos[i]| < r, no self pair at s = 0).  Integer output: bit-exact, in
the same receiver-sorted order (then by source and image)."""

import ctypes
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gpu(pos, cell, r, pbc=None):
    from fsctep_amd.neighbors import neighbor_csr
    src, dst, sh, dst_ptr = neighbor_csr(torch.tensor(pos, dtype=torch.float64, device=DEV),
                                         r, torch.tensor(np.asarray(cell).reshape(3, 3), dtype=torch.float64), pbc)
    return src.cpu().numpy(), dst.cpu().numpy(), sh.cpu().numpy(), dst_ptr.cpu().numpy()


def _brute(pos, cell, r, pbc):
    """The reference's edge set by brute force over all pairs and images, sorted (dst, src, shift)."""
    cell = np.asarray(cell, np.float64).reshape(3, 3)
    rng = [(-1, 0, 1) if p else (0,) for p in pbc]
    S, D, SH = [], [], []
    for sx in rng[0]:
        for sy in rng[1]:
            for sz in rng[2]:
                s = np.array([sx, sy, sz], np.float64)
                sv = (s[0] * cell[0] + s[1] * cell[1]) + s[2] * cell[2]
                d = (pos[None, :, :] - pos[:, None, :]) + sv          # [i][j] = (pos_j - pos_i) + s.cell
                d2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
                m = d2 < r * r
                if not s.any():
                    np.fill_diagonal(m, False)
                ii, jj = np.nonzero(m)
                S.append(ii)
                D.append(jj)
                SH.append(np.broadcast_to(s, (ii.shape[0], 3)))
    src, dst, sh = np.concatenate(S), np.concatenate(D), np.concatenate(SH)
    o = np.lexsort((sh[:, 2], sh[:, 1], sh[:, 0], src, dst))
    return src[o], dst[o], sh[o]


def _equal(got, want, N):
    src, dst, sh, dst_ptr = got
    np.testing.assert_array_equal(dst, want[1])
    np.testing.assert_array_equal(src, want[0])
    np.testing.assert_array_equal(sh, want[2])
    np.testing.assert_array_equal(dst_ptr, np.concatenate([[0], np.cumsum(np.bincount(want[1], minlength=N))]))


@pytest.mark.parametrize("mode,atoms", [("sparse", 1000), ("sparse", 10000), ("ictd-o3", 4000)])
def test_matches_host_list_of_the_benchmark_systems(mode, atoms):
    import bench
    s = bench._system(mode, atoms, bench.WORKLOADS[mode]["seed"])
    got = _gpu(s.pos, s.cell, 5.0)
    _equal(got, (s.edge_src, s.edge_dst, s.edge_shifts), atoms)
    # the timed rebuild (count pass, edge-count read back, fill pass)
    from fsctep_amd.neighbors import radius_graph_pbc_gpu
    pos = torch.tensor(s.pos, dtype=torch.float64, device=DEV)
    cell = torch.tensor(s.cell, dtype=torch.float64, device=DEV)
    radius_graph_pbc_gpu(pos, 5.0, cell)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(5):
        radius_graph_pbc_gpu(pos, 5.0, cell)
    torch.cuda.synchronize()
    print(f"{mode} {atoms} atoms, {got[0].shape[0]} edges: rebuild {(time.perf_counter() - t0) / 5 * 1e3:.3f} ms")


def test_small_box_many_images_and_open_system():
    from fsctep_amd.synthetic import radius_graph
    rng = np.random.default_rng(3)
    # box 7 A < 2 r: several images of one pair within the cutoff (the host's brute-force branch)
    pos = rng.uniform(0.0, 7.0, (40, 3))
    cell = np.eye(3)[None] * 7.0
    want = radius_graph(pos, cell, True, 5.0)
    _equal(_gpu(pos, cell, 5.0), want, 40)
    _equal(_gpu(pos, cell, 5.0), _brute(pos, cell, 5.0, (1, 1, 1)), 40)
    # open system (kd-tree branch of the host list)
    pos = rng.uniform(0.0, 20.0, (300, 3))
    want = radius_graph(pos, np.eye(3)[None] * 100.0, False, 5.0)
    _equal(_gpu(pos, np.eye(3) * 100.0, 5.0, pbc=False), want, 300)


@pytest.mark.parametrize("pbc", [(1, 1, 1), (1, 1, 0), (0, 0, 0), (0, 1, 0)])
def test_triclinic_partial_pbc_unwrapped_positions(pbc):
    rng = np.random.default_rng(sum(pbc) + 10)
    cell = np.array([[11.0, 0.0, 0.0], [3.1, 10.2, 0.0], [-2.2, 1.7, 12.5]])
    frac = rng.uniform(-0.1, 1.1, (220, 3))                   # some atoms outside the cell
    pos = frac @ cell
    _equal(_gpu(pos, cell, 4.5, pbc), _brute(pos, cell, 4.5, pbc), 220)


def test_degenerate_inputs():
    cell = np.eye(3) * 10.0
    for N in (0, 1):
        src, dst, sh, dst_ptr = _gpu(np.zeros((N, 3)) + 1.0, cell, 5.0)
        assert src.shape == (0,) and sh.shape == (0, 3) and dst_ptr.tolist() == [0] * (N + 1)
    # one atom in a box smaller than the cutoff sees its own images (s != 0), as in the reference
    got = _gpu(np.array([[0.5, 0.5, 0.5]]), np.eye(3) * 4.0, 5.0)
    _equal(got, _brute(np.array([[0.5, 0.5, 0.5]]), np.eye(3) * 4.0, 5.0, (1, 1, 1)), 1)
    assert got[0].shape[0] == 6                               # the 6 face images at 4 A (edge images: 5.66 A)
    # all atoms at one point (no extent): every pair at distance 0
    got = _gpu(np.zeros((5, 3)), cell, 1.0, pbc=False)
    assert got[0].shape[0] == 20


def test_feeds_graph_preparation_unchanged():
    """The list is already receiver-sorted and stable: prepare_graph's order is the identity."""
    import bench
    from fsctep_amd.graph import prepare_graph
    s = bench._system("sparse", 1000, 22)
    src, dst, sh, _ = [torch.as_tensor(a).to(DEV) for a in _gpu(s.pos, s.cell, 5.0)]
    g = prepare_graph(src, dst, sh, 1000)
    assert torch.equal(g.order.cpu(), torch.arange(src.shape[0], dtype=torch.int32))


@pytest.mark.parametrize("n,r", [(513, 9.0), (514, 9.0), (700, 9.0), (700, 3.2)])
def test_receivers_around_the_key_capacity(n, r):
    """512 neighbours rank their keys in LDS, more go through memory; the last case mixes both in one list."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 5.0, (n, 3))
    cell = np.eye(3) * 100.0
    got = _gpu(pos, cell, r, pbc=False)
    _equal(got, _brute(pos, cell, r, (0, 0, 0)), n)
    deg = np.diff(got[3])
    assert deg.max() == n - 1 if r > 8.7 else (deg.max() > 512 and deg.min() < 512)


@pytest.mark.parametrize("n", [769, 1024, 1025, 1026, 1600])
def test_receivers_of_several_key_chunks(n):
    """More than 512 neighbours: keys ranked 256 at a time against chunks of 512, whole and partial ones."""
    pos = np.random.default_rng(n).uniform(0.0, 5.0, (n, 3))
    got = _gpu(pos, np.eye(3) * 100.0, 9.0, pbc=False)
    _equal(got, _brute(pos, np.eye(3) * 100.0, 9.0, (0, 0, 0)), n)
    assert (np.diff(got[3]) == n - 1).all()


def test_fill_stays_within_a_smaller_edge_count():
    """fsc_neighbor_fill with fewer edges than the list has: receivers before the cut are whole, nothing is written
    at or past it (receivers wholly past it have no room at all), also where more than 512 keys are ranked."""
    from fsctep_amd import _lib
    for n, side, r in ((70, 5.0, 9.0), (530, 5.0, 9.0), (90, 12.0, 4.0)):
        pos = torch.tensor(np.random.default_rng(n).uniform(0.0, side, (n, 3)), device=DEV)
        cell = torch.eye(3, dtype=torch.float64, device=DEV) * 100.0
        want = _gpu(pos.cpu().numpy(), cell.cpu().numpy(), r, pbc=False)
        ws_n = ctypes.c_int64()
        _lib.call("fsc_neighbor_workspace", n, ctypes.byref(ws_n))
        ws = torch.empty(ws_n.value, dtype=torch.int32, device=DEV)
        dst_ptr = torch.empty(n + 1, dtype=torch.int32, device=DEV)
        pbc, st = (ctypes.c_int32 * 3)(0, 0, 0), torch.cuda.current_stream().cuda_stream
        _lib.call("fsc_neighbor_count", n, pos.data_ptr(), cell.data_ptr(), pbc, r, dst_ptr.data_ptr(), ws.data_ptr(), st)
        ptr = dst_ptr.cpu().numpy()
        E = int(ptr[n])
        np.testing.assert_array_equal(ptr, want[3])
        for cut in (1, int(ptr[3]), int(ptr[n // 2]) + 1, E - 1, E):
            src = torch.full((E + 1024,), -7, dtype=torch.int64, device=DEV)
            dst, sh = src.clone(), torch.full((E + 1024, 3), -7.0, dtype=torch.float64, device=DEV)
            fill = torch.empty(2 * E, dtype=torch.int32, device=DEV)
            _lib.call("fsc_neighbor_fill", n, cut, pos.data_ptr(), cell.data_ptr(), pbc, r, dst_ptr.data_ptr(),
                      ws.data_ptr(), fill.data_ptr(), src.data_ptr(), dst.data_ptr(), sh.data_ptr(), st)
            whole = int(ptr[np.searchsorted(ptr, cut, side="right") - 1])   # end of the last whole segment
            for got, ref in zip((src, dst, sh), want):
                got = got.cpu().numpy()
                np.testing.assert_array_equal(got[:whole], ref[:whole])
                assert (got[cut:] == -7).all()
