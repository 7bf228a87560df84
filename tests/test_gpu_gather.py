"""The sparse launch's virtual tiles (eight selected 4-cell blocks each, four a split) at the sizes where they can go
wrong: rows of one entry, of a full tile less, exactly and plus one entry, of a full split (32 entries) around its edges
and of the most entries (512 blocks with each tail), an ID repeated in a body, selections whose blocks share a pool tile
in every arrangement, and prompts whose row count sits at the edges of the rule that splits rows. Each against the
oracle's fp64 attention over the selected cells (max-abs 2e-3, test_gpu_sparse.py's and test_gpu_qsp.py's bound)."""
import numpy as np
import pytest

import cases
import fnkv
import oracle as O
import test_gpu_qsa_attend as qsa
import test_gpu_qsp as qsp
import test_gpu_sparse as sparse

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 2e-3


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("fmt", [fnkv.FMT_Q8_0, fnkv.FMT_KV8])
@pytest.mark.parametrize("depth", [1, 3, 4, 26, 30, 31, 34, 126, 127, 130, 254, 2042, 2046, 2047, 2049, 5002])
def test_entries_at_tile_and_split_edges(depth, fmt):
    pool, got, ref, _ = sparse.sparse_case(depth, 1, seed=depth + 900, fmt=fmt)
    assert np.isfinite(got).all()
    assert cases.out_err(got, ref) <= TOL


@pytest.mark.parametrize("T", [1, 4])
def test_repeated_ids_count_once(T):
    # every row's sixth and seventh entries repeat its fifth, the last repeats the one before it
    depth = 6001
    words, offs, _ = O.qsa_body(depth, T, seed=61)
    w = words.view(np.int32).copy()
    cells = []
    for t in range(T):
        o, n_vis = offs[t] // 4, (depth + t + 1) // 4
        ids = w[o + 2:o + 2 + w[o]]
        ids[5] = ids[6] = ids[4]
        ids[-1] = ids[-2]
        b = np.unique(ids).astype(np.int64)
        cells.append(np.concatenate([(4 * b[:, None] + np.arange(4)).reshape(-1), np.arange(4 * n_vis, depth + t + 1)]))
    pool, got, ref, _ = sparse.sparse_case(depth, T, seed=61, body=(w.view(np.uint32), offs, cells))
    assert cases.out_err(got, ref) <= TOL


@pytest.mark.parametrize("blocks_of_tile", [[0], [7], [0, 4], [3, 4], [1, 2, 3], [0, 2, 4, 6], list(range(8))])
def test_blocks_that_share_a_pool_tile(blocks_of_tile):
    # 512 blocks, the same ones of every tile (the last tiles fill up to 512)
    depth, T = 20000, 1
    n_vis = (depth + 1) // 4
    tiles = np.arange(n_vis // 8 - 2)[-(512 // len(blocks_of_tile)):]
    b = (8 * tiles[:, None] + np.array(blocks_of_tile)).reshape(-1)
    b = np.unique(np.concatenate([np.setdiff1d(np.arange(n_vis), b)[:512 - b.size], b]))
    tail = np.arange(4 * n_vis, depth + 1)
    words = np.concatenate([[512, tail.size], b, tail]).astype(np.uint32)
    cells = [np.concatenate([(4 * b[:, None] + np.arange(4)).reshape(-1), tail])]
    pool, got, ref, _ = sparse.sparse_case(depth, T, seed=71,
                                           body=(words, np.array([0, 4 * words.size], np.int32), cells))
    assert cases.out_err(got, ref) <= TOL


# decode rows whose one-tile-a-wave splits are more than the CUs: several tiles a wave (16 pairs of (row, head tile) at 17
# splits: 272; 15: 255, the last with one tile a wave), the new cells written by the launch that prepares its rows, by a
# prepare before it (more than 16 heads a KV head), or appended before it (one row too)
@pytest.mark.parametrize("depth,T,hq,hkv,fmt", [
    (3000, 3, 32, 8, fnkv.FMT_Q8_0), (2045, 5, 32, 8, fnkv.FMT_KV8), (3000, 1, 128, 16, fnkv.FMT_Q8_0),
    (9000, 5, 96, 2, fnkv.FMT_Q8_0), (3000, 5, 12, 3, fnkv.FMT_Q8_0), (600, 5, 64, 16, fnkv.FMT_KV8)])
def test_rows_of_many_kv_heads(depth, T, hq, hkv, fmt):
    pool, got, ref, _ = sparse.sparse_case(depth, T, seed=depth + T + hkv, hq=hq, hkv=hkv, fmt=fmt)
    assert np.isfinite(got).all()
    assert cases.out_err(got, ref) <= TOL


@pytest.mark.parametrize("depth,T,hq,hkv,fmt", [
    (3000, 3, 32, 8, fnkv.FMT_Q8_0), (2044, 5, 32, 8, fnkv.FMT_KV8), (20001, 5, 32, 8, fnkv.FMT_Q8_0),
    (3000, 1, 64, 16, fnkv.FMT_KV8), (2045, 5, 64, 2, fnkv.FMT_Q8_0), (3000, 5, 12, 3, fnkv.FMT_Q8_0)])
def test_prepared_rows_of_many_kv_heads(depth, T, hq, hkv, fmt):
    qsa.run_case(depth, T, hq, hkv, seed=depth + T + hkv, fmt=fmt, planes=True)


# pairs (row, 16-head tile of a KV head) a launch: 17 splits a row up to 30, one split from 257 on (256 CUs, two
# workgroups each)
@pytest.mark.parametrize("rows,hq,h_kv", [(6, 12, 1), (30, 12, 1), (31, 12, 1), (129, 16, 2), (256, 12, 1), (257, 12, 1),
                                          (70, 40, 2)])
def test_prompt_rows_at_the_split_rule(rows, hq, h_kv):
    o16, o32, err, ref = qsp.run_attend(3000, rows, hq, h_kv, seed=rows + hq)
    assert err == 0 and np.isfinite(o32).all()
    assert float(np.abs(o32.astype(np.float64) - ref).max()) <= TOL
    assert np.array_equal(o16.view(np.uint16), o32.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("hq,hkv", [(12, 1), (16, 2), (48, 1)])
def test_prompt_workspace_serves_smaller_chunks(hq, hkv):
    # the bytes for a caller's largest chunk hold every smaller or shallower one's partials
    pool = fnkv.Pool(1, 4, 1, hkv)
    rows = sorted({*range(1, 40), 100, 127, 128, 129, 255, 256, 257, 300, 511, 512, 513, 700, 1000, 2048})
    for a, b in zip(rows, rows[1:]):
        for pos0 in (0, 100, 2000, 40000):
            assert 0 < pool.qsp_ws_bytes(pos0, a, hq) <= pool.qsp_ws_bytes(pos0, b, hq)
            assert pool.qsp_ws_bytes(pos0, a, hq) <= pool.qsp_ws_bytes(pos0 + 1000, a, hq)
    # and no more than the partials that some launch writes: rows of several splits fill two workgroups a CU at most (256
    # CUs), five rows take 17 splits each, and rows of one split write none
    head_tiles = hkv * -(-hq // hkv // 16)
    assert pool.qsp_ws_bytes(40000, 4096, hq) <= max(512 // head_tiles, 5 * 17) * hq * 258 * 4 + 16


@pytest.mark.parametrize("rows,hq,h_kv", [(6, 12, 1), (30, 12, 1), (100, 40, 2), (256, 12, 1), (257, 12, 1)])
def test_prompt_rows_stay_within_their_workspace(rows, hq, h_kv, monkeypatch):
    attend = fnkv.Pool.qsp_attend

    def guarded(pool, slot, layer, pos0, qfull, *more, **kw):
        need = pool.qsp_ws_bytes(pos0, rows, hq)
        buf = torch.full((need + (8 << 20),), 0x5a, dtype=torch.uint8, device="cuda")
        attend(pool, slot, layer, pos0, qfull, *more, ws=buf[:need], **kw)
        assert int((buf[need:] != 0x5a).sum()) == 0

    monkeypatch.setattr(fnkv.Pool, "qsp_attend", guarded)
    _, o32, err, ref = qsp.run_attend(3000, rows, hq, h_kv, seed=rows + hq)
    assert err == 0 and float(np.abs(o32.astype(np.float64) - ref).max()) <= TOL
