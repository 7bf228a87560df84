"""The chunked prefill's key splits at the shapes where their workgroups' layout changes: causal chunks whose first row
blocks see fewer splits than the last (none, one or several short), a chunk that starts a prompt, one row block over many
splits (the four-wave merge), single tiles, last blocks of one token, groups of 1 to 64 query heads. The split launch
against the launch without a workspace (one split a row block) over every row of outputs filled with NaN first, and the
chunk's edge rows against the oracle's fp64 attention (max-abs 2e-3; the two launches then agree within twice that)."""
import numpy as np
import pytest

import cases
import fnkv
import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 2e-3


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("depth,rows,hq,hkv,fmt", [
    (0, 1, 16, 2, fnkv.FMT_Q8_0), (0, 32, 16, 2, fnkv.FMT_Q8_0), (31, 1, 16, 2, fnkv.FMT_Q8_0),
    (0, 33, 16, 1, fnkv.FMT_KV8), (0, 700, 16, 2, fnkv.FMT_Q8_0), (0, 1537, 16, 2, fnkv.FMT_Q8_0),
    (95, 961, 12, 3, fnkv.FMT_Q8_0), (1000, 513, 16, 2, fnkv.FMT_KV8), (3, 1024, 8, 1, fnkv.FMT_Q8_0),
    (9000, 16, 16, 2, fnkv.FMT_Q8_0), (9000, 1, 8, 8, fnkv.FMT_Q8_0), (20000, 65, 64, 1, fnkv.FMT_Q8_0),
    (4000, 257, 1, 1, fnkv.FMT_Q8_0), (6144, 2048, 16, 2, fnkv.FMT_Q8_0)])
def test_splits_cover_every_row(depth, rows, hq, hkv, fmt):
    ctx, seed = depth + rows, depth + 3 * rows + hq
    pool = fnkv.Pool(2, -(-ctx // 256) + 4, 1, hkv, fmt=fmt)
    cases.scatter_ensure(pool, [0], [ctx], seed, churn=0.3)
    k16, v16 = cases.kv_rows(seed, ctx, hkv)
    pool.append(0, 0, 0, torch.from_numpy(k16).cuda(), torch.from_numpy(v16).cuda())
    q16 = cases.queries(seed, (rows, hq, 256))
    q = torch.from_numpy(q16).cuda()
    got, one = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    pool.prefill(0, 0, ctx, q, got)
    pool.prefill(0, 0, ctx, q, one, ws=False)
    torch.cuda.synchronize()
    g, o = got.cpu().numpy().astype(np.float32), one.cpu().numpy().astype(np.float32)
    assert np.isfinite(g).all() and np.isfinite(o).all()
    assert cases.out_err(g, o) <= 2 * TOL
    (_, _, kf), (_, _, vf) = (cases.decoded_kv8 if fmt == fnkv.FMT_KV8 else cases.decoded)(O, k16, v16)
    check = sorted({0, 1, rows // 3, rows // 2, rows - 2, rows - 1} & set(range(rows)))
    ref = O.attn_f64(q16.view(np.uint16), kf, vf, ctx, rows=check)
    assert cases.out_err(got.cpu().numpy()[check], ref) <= TOL
    assert cases.out_err(one.cpu().numpy()[check], ref) <= TOL


@pytest.mark.parametrize("share", [0.2, 0.5, 0.99])
def test_a_workspace_below_the_plans(share):
    # a workspace sized for other chunks: the best splits that it holds, down to one
    depth, rows, hq, hkv = 9000, 65, 16, 2
    ctx = depth + rows
    pool = fnkv.Pool(2, -(-ctx // 256) + 4, 1, hkv)
    cases.scatter_ensure(pool, [0], [ctx], 77, churn=0.3)
    k16, v16 = cases.kv_rows(77, ctx, hkv)
    pool.append(0, 0, 0, torch.from_numpy(k16).cuda(), torch.from_numpy(v16).cuda())
    q16 = cases.queries(77, (rows, hq, 256))
    q = torch.from_numpy(q16).cuda()
    got = torch.full_like(q, float("nan"))
    need = pool.prefill_ws_bytes(ctx, rows, hq)
    held = int(need * share) // 16 * 16
    buf = torch.full((2 * need,), 0x5a, dtype=torch.uint8, device="cuda")  # the bytes behind the workspace stay as they are
    pool.prefill(0, 0, ctx, q, got, ws=buf[:held])
    torch.cuda.synchronize()
    assert int((buf[held:] != 0x5a).sum()) == 0
    (_, _, kf), (_, _, vf) = cases.decoded(O, k16, v16)
    check = [0, 1, 32, 63, 64]
    ref = O.attn_f64(q16.view(np.uint16), kf, vf, ctx, rows=check)
    assert cases.out_err(got.cpu().numpy()[check], ref) <= TOL


@pytest.mark.parametrize("pages", [2047, 2050])
def test_one_split_past_the_page_copy(pages):
    # without a workspace a chunk's keys are one split: up to 2,047 pages its page numbers sit in LDS (2,048 entries),
    # past them the launch reads the device's table
    rows, hq = 5, 8
    ctx = pages * 256 - 100
    pool = fnkv.Pool(2, pages + 4, 1, 1)
    cases.scatter_ensure(pool, [0], [ctx], 91)
    k16, v16 = cases.kv_rows(91, ctx, 1)
    pool.append(0, 0, 0, torch.from_numpy(k16).cuda(), torch.from_numpy(v16).cuda())
    q16 = cases.queries(91, (rows, hq, 256))
    q = torch.from_numpy(q16).cuda()
    got, one = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    pool.prefill(0, 0, ctx, q, got)
    pool.prefill(0, 0, ctx, q, one, ws=False)
    torch.cuda.synchronize()
    (_, _, kf), (_, _, vf) = cases.decoded(O, k16, v16)
    ref = O.attn_f64(q16.view(np.uint16), kf, vf, ctx, rows=[0, 4])
    assert cases.out_err(got.cpu().numpy()[[0, 4]], ref) <= TOL
    assert cases.out_err(one.cpu().numpy()[[0, 4]], ref) <= TOL
    assert cases.out_err(one.cpu().numpy(), got.cpu().numpy()) <= 2 * TOL
