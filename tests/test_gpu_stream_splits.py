"""The dense walk's split sizes at the edges of their rules: the fine splits (128 cells, at most one workgroup a CU: the
last context that takes them, the first that does not, contexts of less than one tile), a workspace too small for the
fine splits (the coarser plan runs in it), and walks past a lane register's 64 tiles (32 KV heads, one context of more
than 16,384 cells). Against the oracle's fp64 attention at the max-abs tolerance of the other decode tests."""
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


def launch(ctxs, T, hq, hkv, seed, dev_slack=0, shrink=0, fmt=fnkv.FMT_Q8_0):
    bound = [c + dev_slack for c in ctxs]
    pool = fnkv.Pool(len(ctxs) + 1, sum(-(-c // 256) for c in bound) + 8, 1, hkv, fmt=fmt)
    cases.scatter_ensure(pool, list(range(len(ctxs))), bound, seed, churn=0.3)
    rows = []
    for s, c in enumerate(ctxs):
        k16, v16 = cases.kv_rows(seed + s, c, hkv)
        pool.append(s, 0, 0, torch.from_numpy(k16).cuda(), torch.from_numpy(v16).cuda())
        rows.append((k16, v16))
    q16 = cases.queries(seed, (len(ctxs), T, hq, 256))
    q = torch.from_numpy(q16).cuda()
    out = torch.full_like(q, float("nan"))
    held = pool.decode_ws_bytes(bound, T, hq) - shrink
    buf = torch.zeros(held + shrink + (1 << 20), dtype=torch.uint8, device="cuda")
    buf[held:] = 0x5a  # the bytes behind the workspace stay as they are
    ws = buf[:held]
    slots = list(range(len(ctxs)))
    if dev_slack:
        err = torch.zeros(1, dtype=torch.int32, device="cuda")
        pool.decode_dev(slots, torch.tensor(ctxs, dtype=torch.int64, device="cuda"), bound, T, 0, q, out, ws, err)
        torch.cuda.synchronize()
        assert int(err.item()) == 0
    else:
        pool.decode(slots, ctxs, T, 0, q, out, ws)
        torch.cuda.synchronize()
    assert int((buf[held:] != 0x5a).sum()) == 0
    return q16, out.cpu().numpy(), rows


def check(q16, got, rows, ctxs, hq, hkv, heads, fmt=fnkv.FMT_Q8_0):
    G = hq // hkv
    dec = cases.decoded_kv8 if fmt == fnkv.FMT_KV8 else cases.decoded
    for i, c in enumerate(ctxs):
        k16, v16 = (np.ascontiguousarray(x[:, heads]) for x in rows[i])
        (_, _, kf), (_, _, vf) = dec(O, k16, v16)
        q_heads = [h * G + g for h in heads for g in range(G)]
        q = np.ascontiguousarray(q16[i][:, q_heads])
        ref = O.attn_f64(q.view(np.uint16), kf, vf, c)
        assert cases.out_err(got[i][:, q_heads], ref) <= TOL


@pytest.mark.parametrize("T", [1, 3, 5])
@pytest.mark.parametrize("ctxs,dev_slack", [
    ([16384], 0), ([16385], 0), ([16000], 384), ([16000], 385), ([6], 0), ([31, 129, 128, 127], 0), ([40], 5000)])
def test_fine_splits(ctxs, dev_slack, T):
    q16, got, rows = launch(ctxs, T, 16, 2, 900 + T, dev_slack)
    check(q16, got, rows, ctxs, 16, 2, [0, 1])


@pytest.mark.parametrize("T", [1, 5])
def test_a_workspace_below_the_fine_plans(T):
    ctxs = [4099]
    for shrink in (257, 8192):  # (the size asked for holds 256 bytes more than the plan: 257 leaves one byte less)
        q16, got, rows = launch(ctxs, T, 16, 2, 920 + T, shrink=shrink)
        check(q16, got, rows, ctxs, 16, 2, [0, 1])
    with pytest.raises(fnkv.FnkvError):  # below the coarser plan's 17 splits as well
        launch(ctxs, T, 16, 2, 920, shrink=17 * 2 * 8 * T * 1032)


@pytest.mark.parametrize("G,T,dev_slack,fmt", [
    (1, 1, 0, fnkv.FMT_Q8_0), (1, 1, 300, fnkv.FMT_KV8), (6, 3, 0, fnkv.FMT_Q8_0), (8, 5, 0, fnkv.FMT_KV8),
    (8, 5, 300, fnkv.FMT_Q8_0)])
def test_walks_past_64_tiles(G, T, dev_slack, fmt):
    ctxs, hkv = [17001], 32
    q16, got, rows = launch(ctxs, T, G * hkv, hkv, 940 + G, dev_slack, fmt=fmt)
    check(q16, got, rows, ctxs, G * hkv, hkv, [0, 13, 31], fmt=fmt)


@pytest.mark.parametrize("deep,T_deep", [([66000], 1), ([140000], 1), ([140000], 5), ([200000], 3),
                                         ([100000, 70000, 3000], 3)])
def test_a_workspace_for_deeper_contexts_serves_shorter_ones(deep, T_deep):
    # the rule's split count falls where larger splits come to fit one round of workgroups: the workspace sized for the
    # deepest contexts and largest step runs every shorter call, as far from fp64 as with its own workspace
    hq, hkv, layers = 16, 2, 1
    pool = fnkv.Pool(len(deep) + 1, sum(-(-c // 256) for c in deep) + 8, layers, hkv)
    for s, c in enumerate(deep):
        assert pool.ensure(s, c)[0] == 0
        g = torch.Generator(device="cuda").manual_seed(970 + s)
        k, v = (torch.randn((c, hkv, 256), generator=g, device="cuda").half() for _ in range(2))
        pool.append(s, 0, 0, k, v)
    held = pool.decode_ws_bytes(deep, T_deep, hq)
    buf = torch.zeros(held + (8 << 20), dtype=torch.uint8, device="cuda")
    buf[held:] = 0x5a  # the bytes behind the workspace stay as they are
    ws = buf[:held]
    calls = [[c] for c in range(T_deep, deep[0], 6007)]
    calls += [[c] for c in (22017, 32768, 33000, 65505, 98305, 131041, 131072, 196577) if c < deep[0]]
    calls += [[max(T_deep, int(c * x)) for c in deep] for x in (0.999, 0.95, 0.7, 0.51, 0.3, 0.1)]
    smaller = 0
    for ctxs in calls:
        for T in {1, T_deep}:
            n = pool.decode_ws_bytes(ctxs, T, hq)
            q = torch.from_numpy(cases.queries(971, (len(ctxs), T, hq, 256))).cuda()
            got, own = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
            slots = list(range(len(ctxs)))
            pool.decode(slots, ctxs, T, 0, q, got, ws)
            pool.decode(slots, ctxs, T, 0, q, own, torch.zeros(n, dtype=torch.uint8, device="cuda"))
            torch.cuda.synchronize()
            smaller += n > held
            assert float((got.float() - own.float()).abs().max()) <= 2 * TOL, (ctxs, T)
    assert int((buf[held:] != 0x5a).sum()) == 0
    print(f"{smaller} of {2 * len(calls)} calls ask for more than the workspace")
    assert smaller > 0


@pytest.mark.parametrize("fmt", [fnkv.FMT_Q8_0, fnkv.FMT_KV8])
def test_long_walks_keep_the_precision(fmt):
    # 16,384 cells take walks of 64 tiles, 17,001 walks of 68, whose weights lie one binary place higher: the part of
    # the error that comes from fp16's floor under the weights (most of it) halves, so the whole falls by a fifth at
    # least; without the lead the longer walks are no closer to 64 bits than the shorter
    hkv, T, heads = 32, 5, [0, 13, 31]
    rel = []
    for c in (16384, 17001):
        q16, got, rows = launch([c], T, 8 * hkv, hkv, 960, fmt=fmt)
        k16, v16 = (np.ascontiguousarray(x[:, heads]) for x in rows[0])
        (_, _, kf), (_, _, vf) = (cases.decoded_kv8 if fmt == fnkv.FMT_KV8 else cases.decoded)(O, k16, v16)
        q_heads = [8 * h + g for h in heads for g in range(8)]
        ref = O.attn_f64(np.ascontiguousarray(q16[0][:, q_heads]).view(np.uint16), kf, vf, c)
        rel.append(np.linalg.norm(got[0][:, q_heads].astype(np.float64) - ref) / np.linalg.norm(ref))
    print(f"relative error: 64 tiles {rel[0]:.3e}, 68 tiles {rel[1]:.3e}")
    assert rel[1] <= 0.8 * rel[0]
