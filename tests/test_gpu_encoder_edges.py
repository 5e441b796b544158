"""The encoder's kernels at the edges of their blocks and trees, bit for bit against the oracle:
assignment for codebook sizes around powers of two (levels of the search tree), ties, infinities
and unaligned inputs; k-means whose sort and scatter blocks, cluster sizes and pairwise trees end
just before, at and just after a boundary."""
import numpy as np
import pytest
import torch

import oracle
from helix_substrate import _hxq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 3, 127, 128, 255, 256, 257, 1000, 4095, 4096])
@pytest.mark.parametrize("offset", [0, 1])
def test_assign_codebook_sizes(dev, k, offset):
    rs = np.random.RandomState(k)
    cb = np.sort(rs.standard_normal(k).astype(np.float32))
    cb[k // 3:k // 2] = cb[k // 3] if k > 2 else cb[k // 3:k // 2]   # a run of equal entries
    mid = ((cb[1:] + cb[:-1]) / 2).astype(np.float32)
    x = np.concatenate([rs.standard_normal(5003).astype(np.float32) * 2, cb, mid,
                        np.float32([np.inf, -np.inf, np.nan, 0.0, -0.0, 3e38, -3e38, 1e-40])])
    print(f"assign k={k} offset={offset} n={x.size}", flush=True)
    buf = torch.zeros(x.size + 4, device=dev)
    buf[offset:offset + x.size] = torch.from_numpy(x).to(dev)   # offset 1: no 16-byte alignment
    got = _hxq.assign_nearest(buf[offset:offset + x.size], torch.from_numpy(cb).to(dev))
    got = got.cpu().numpy().astype(np.int64) & 0xffff
    np.testing.assert_array_equal(got, oracle.assign_nearest_np(x, cb).astype(np.int64))


@pytest.mark.parametrize("n,k", [(1, 1), (7, 3), (2047, 256), (2048, 64), (2049, 256), (4096, 5),
                                 (8192, 1), (8193, 1), (8191 + 129, 2), (70001, 300)])
def test_kmeans_block_edges(dev, n, k):
    rs = np.random.RandomState(n)
    data = rs.standard_normal(n).astype(np.float32)
    if n > 100:
        data[rs.randint(0, n, n // 5)] = np.float32([-0.0, 0.0, 0.5])[rs.randint(0, 3, n // 5)]
    print(f"kmeans n={n} k={k}", flush=True)
    cb, asg, it = _hxq.kmeans_1d(torch.from_numpy(data).to(dev), k, 10, 0.001)
    if cb.numel() <= 256:
        cb_o, asg_o, it_o = oracle.kmeans_np(data, k)
        np.testing.assert_array_equal(asg.cpu().numpy(), asg_o)
        assert it == it_o
    else:   # integer cluster ids (the oracle's are uint8)
        from helix_substrate.hxq_encoder import _simple_kmeans
        cb_o, asg_o = _simple_kmeans(data, k)
        np.testing.assert_array_equal(asg.cpu().numpy().view(np.uint16), asg_o)
    np.testing.assert_array_equal(cb.cpu().numpy(), cb_o)


@pytest.mark.parametrize("sizes", [(63, 64, 65, 127, 128, 129, 130, 255, 256, 257), (8191, 8192, 8193, 16385)])
def test_kmeans_cluster_sizes(dev, sizes):
    """Well separated clusters of given sizes: every shape of the pairwise tree."""
    rs = np.random.RandomState(5)
    data = np.concatenate([10.0 * j + rs.standard_normal(m) for j, m in enumerate(sizes)]).astype(np.float32)
    data = data[rs.permutation(data.size)]
    print(f"kmeans sizes={sizes}", flush=True)
    cb, asg, it = _hxq.kmeans_1d(torch.from_numpy(data).to(dev), len(sizes), 10, 0.001)
    cb_o, asg_o, it_o = oracle.kmeans_np(data, len(sizes))
    np.testing.assert_array_equal(cb.cpu().numpy(), cb_o)
    np.testing.assert_array_equal(asg.cpu().numpy(), asg_o)
    assert it == it_o


@pytest.mark.parametrize("n", [1, 2, 5, 4095, 4096, 4097, 8191, 16389, 262147])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_select_and_outlier_edges(dev, n, offset):
    """Order statistics and outliers around the chunks' and blocks' ends, at every alignment,
    with values that share their upper key bits."""
    rs = np.random.RandomState(n + offset)
    x = rs.standard_normal(n).astype(np.float32)
    x[rs.randint(0, n, max(1, n // 3))] = np.float32(1.0) + rs.randint(0, 4, max(1, n // 3)) * np.float32(2 ** -23)
    x[rs.randint(0, n)] = -np.inf
    print(f"select n={n} offset={offset}", flush=True)
    buf = torch.zeros(n + 4, device=dev)
    buf[offset:offset + n] = torch.from_numpy(x).to(dev)
    d = buf[offset:offset + n]
    ranks = [0, n // 2, min(n - 1, n // 2 + 1), n - 1]
    vals, nans = _hxq.select_f32(d, ranks)
    np.testing.assert_array_equal(vals.cpu().numpy(), np.sort(x)[ranks])
    assert nans == 0
    for lo, hi in ((-1.5, 1.5), (-np.inf, np.inf), (0.0, 0.0)):
        pos, val = _hxq.outliers_f32(d, lo, hi)
        want = np.where((x < np.float32(lo)) | (x > np.float32(hi)))[0]
        np.testing.assert_array_equal(pos.cpu().numpy(), want)
        np.testing.assert_array_equal(val.cpu().numpy(), x[want])


@pytest.mark.parametrize("shift", [0, 4, 1])
def test_outliers_workspace_of_any_alignment(dev, shift):
    n, lib = 9000, _hxq.lib()
    x = torch.randn(n, generator=torch.Generator().manual_seed(2)).to(dev)
    lohi = torch.tensor([-2.0, 2.0], device=dev)
    size = int(lib.hxq_outliers_workspace_bytes(n))
    buf = torch.full((size + 16,), 0x5a, dtype=torch.uint8, device=dev)
    pos = torch.empty(n, dtype=torch.int64, device=dev)
    val, cnt = torch.empty(n, device=dev), torch.empty(1, dtype=torch.int64, device=dev)
    print(f"outliers workspace + {shift}", flush=True)
    rc = lib.hxq_outliers_f32(x.data_ptr(), n, lohi.data_ptr(), n, pos.data_ptr(), val.data_ptr(),
                              cnt.data_ptr(), buf.data_ptr() + shift, size,
                              torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.hxq_last_error()
    want = torch.nonzero(x.abs() > 2.0).ravel()
    m = int(cnt)
    assert torch.equal(pos[:m], want) and torch.equal(val[:m], x[want])
    assert (buf[:shift] == 0x5a).all() and (buf[shift + size:] == 0x5a).all()


@pytest.mark.parametrize("rows,cols,G", [(1, 16, 16), (3, 96, 96), (5, 260, 52), (7, 640, 128), (2, 384, 1)])
def test_affine_fit_edges(dev, rows, cols, G):
    """Group counts that are no multiple of a wave's four, groups below, at and above a wave."""
    rs = np.random.RandomState(G)
    w = rs.standard_normal((rows, cols)).astype(np.float32)
    cb = np.sort(rs.standard_normal(64).astype(np.float32))
    idx = oracle.assign_nearest_np(w.ravel(), cb).reshape(rows, cols).astype(np.uint8)
    ex = np.sort(rs.choice(rows * cols, 7, replace=False)).astype(np.int64)
    print(f"affine rows={rows} cols={cols} G={G}", flush=True)
    s, o = _hxq.affine_fit(torch.from_numpy(w).to(dev), torch.from_numpy(idx).to(dev), torch.from_numpy(cb).to(dev),
                           G, torch.from_numpy(ex).to(dev))
    so, oo = oracle.affine_fit_np(w, idx, cb, G, ex)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
    np.testing.assert_array_equal(o.cpu().numpy(), oo)
