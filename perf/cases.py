"""The work that a user of fnkv has it do, as cases that can be timed and compared: the engine's decode and verify
steps, its sparse (QSA) steps, prompt chunks over both prompt contracts, and the draft block's step row.

A case is a dict of plain values; `kind` names the call:
  dense    one step of `layers` layers: the new cells of every sequence appended and T query tokens attended over the
           sequence's whole context (fnkv_attn_decode; captured: fnkv_attn_decode_dev, the contexts on the device, all
           layers in one HIP graph, as the engine replays them)
  qsa      one step of `layers` layers of attn::attend over selection bodies, with its prepare and gate (fnkv_attend,
           captured in one HIP graph)
  sparse   the same rows without prepare and gate (fnkv_attn_sparse, captured)
  prefill  a prompt chunk: appended, then attended causally (fnkv_q8_append, fnkv_attn_prefill), one layer
  qsp      a prompt chunk under the reference's own contract: fnkv_qsp_kv, then fnkv_qsp_attend over the rows'
           selection bodies (slab layout), one layer
  datc     the draft step row (fnkv_datc_step) of `layers` draft caches, captured in one HIP graph
K and V are N(0, 1) with 4 of the 256 channels x8 (the distribution the repository's tests and benchmark use), page
tables are scattered, selections are either uniformly random or clustered (a sink, a local window and runs)."""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "fnfl-v100_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "fnfl-v100_amd"))

import fnkv  # noqa: E402

D, PAGE, BLOCK, TOP = 256, 256, 4, 512
FORMATS = {"q8_0": fnkv.FMT_Q8_0, "kv8": fnkv.FMT_KV8}


def listed():
    return [
        # one short conversation, one token a step: the smallest step a server takes, launches and latency
        dict(name="decode_4k", kind="dense", ctxs="4096", T=1, layers=12, hq=16, hkv=2, fmt="q8_0", new="f16",
             captured=True),
        # a batch of short conversations of every length, called eagerly with F32 projections, KV8 pool
        dict(name="decode_batch_ragged", kind="dense", ctxs="301,1023,1500,2777,4099,6000,8191,12345", T=1, layers=4,
             hq=16, hkv=2, fmt="kv8", new="f32", captured=False),
        # four conversations of 8K to 64K cells verified at draft depth 2: the benchmark's headline step
        dict(name="verify_8k_64k", kind="dense", ctxs="8192,16384,32768,65536", T=3, layers=4, hq=16, hkv=2,
             fmt="q8_0", new="f16", captured=False),
        # one conversation at the longest context, one token
        dict(name="decode_262k", kind="dense", ctxs="262144", T=1, layers=2, hq=16, hkv=2, fmt="q8_0", new="f16",
             captured=False),
        # the same verified at draft depth 4 through device contexts, an odd length
        dict(name="verify_262k", kind="dense", ctxs="262101", T=5, layers=2, hq=16, hkv=2, fmt="q8_0", new="f16",
             captured=True),
        # the engine's sparse verify step deep in a conversation: 3 rows, 12 heads on one KV head (the reference's card)
        dict(name="qsa_196k", kind="qsa", depth=196605, rows=3, layers=12, hq=12, hkv=1, fmt="q8_0", clustered=False),
        # one sparse decode row early in a conversation, clustered selection, both KV heads, KV8
        dict(name="sparse_9k", kind="sparse", depth=9001, rows=1, layers=12, hq=16, hkv=2, fmt="kv8", clustered=True),
        # a 2,048-token prompt chunk deep in a long prompt
        dict(name="prefill_131k", kind="prefill", ctx=133120, rows=2048, hq=16, hkv=2, fmt="q8_0"),
        # the last, odd chunk of a short prompt
        dict(name="prefill_3k", kind="prefill", ctx=3001, rows=517, hq=16, hkv=2, fmt="q8_0"),
        # a prompt chunk under the reference's contract: sparse rows, prepare and gate
        dict(name="qsp_40k", kind="qsp", pos0=40000, rows=1000, hq=12, hkv=1, fmt="q8_0", clustered=True),
        # the draft block's step row at the deepest point of its own benchmark, and at the shallowest
        dict(name="datc_196k", kind="datc", cells=196608, layers=2),
        dict(name="datc_4k", kind="datc", cells=4096, layers=8),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["dense", "dense", "dense", "qsa", "sparse", "prefill", "qsp", "datc"])
    hq, hkv = rng.choice([(16, 2), (16, 2), (12, 1)])
    fmt = rng.choice(["q8_0", "q8_0", "kv8"])
    if kind == "dense":
        n = log(1, 8)
        T = rng.choice([1, 1, 2, 3, 4] if hkv == 1 else [1, 1, 2, 3, 4, 5, 6])
        ctxs = ",".join(str(log(200, 262144 // n)) for _ in range(n))
        return dict(kind=kind, ctxs=ctxs, T=T, layers=rng.choice([2, 4]), hq=hq, hkv=hkv, fmt=fmt,
                    new=rng.choice(["f16", "f32"]), captured=rng.random() < 0.5)
    if kind in ("qsa", "sparse"):
        return dict(kind=kind, depth=log(100, 196600), rows=rng.randint(1, 5), layers=4, hq=hq, hkv=hkv, fmt=fmt,
                    clustered=rng.random() < 0.5)
    if kind == "prefill":
        rows = log(16, 2048)
        return dict(kind=kind, ctx=rows + log(16, 131072), rows=rows, hq=16, hkv=rng.choice([1, 2]), fmt=fmt)
    if kind == "qsp":
        return dict(kind=kind, pos0=log(64, 131072), rows=log(16, 1500), hq=hq, hkv=hkv, fmt=fmt,
                    clustered=rng.random() < 0.5)
    return dict(kind="datc", cells=log(300, 196608), layers=4)


# ---- inputs, from the seed alone ----

def _gen(seed, *more):
    g = torch.Generator(device="cuda")
    s = int(seed)
    for m in more:
        s = (s * 1000003 + int(m) + 1) % (1 << 62)
    g.manual_seed(s)
    return g


def _uniform(g, shape, lo, hi):
    return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=g)


def _kv(seed, layer, seq, n, hkv):
    """K and V rows, fp16 [n][hkv][256]"""
    g = _gen(seed, 11, layer, seq)
    got = []
    for _ in range(2):
        x = torch.randn((n, hkv, D), generator=g, device="cuda")
        x[:, :, torch.randperm(D, generator=g, device="cuda")[:4]] *= 8.0
        got.append(x.half())
    return got


def _body(rng, q, clustered):
    """One row's selection at position q: (words, cells), the blocks ascending"""
    n_vis = (q + 1) // BLOCK
    k = min(n_vis, TOP)
    if clustered and n_vis > k:
        runs = [np.arange(16), np.arange(max(0, n_vis - 64), n_vis)]
        starts, lengths = rng.integers(0, n_vis, 3 * k // 8), rng.integers(8, 64, 3 * k // 8)
        runs += [np.arange(a, min(n_vis, a + b)) for a, b in zip(starts, lengths)]
        near = np.unique(np.concatenate(runs))
        blocks = near if near.size <= k else rng.choice(near, k, replace=False)
        if blocks.size < k:
            blocks = np.concatenate([blocks, rng.choice(np.setdiff1d(np.arange(n_vis), blocks), k - blocks.size,
                                                        replace=False)])
        blocks = np.sort(blocks)
    else:
        blocks = np.sort(rng.choice(n_vis, k, replace=False)) if k else np.zeros(0, np.int64)
    tail = np.arange(BLOCK * n_vis, q + 1)
    return (np.concatenate([[k, tail.size], blocks, tail]),
            np.concatenate([(BLOCK * blocks[:, None] + np.arange(BLOCK)).reshape(-1), tail]))


def _rows_body(seed, layer, depth, rows, clustered):
    """The packed bodies of rows depth .. depth + rows - 1: int32 words, byte offsets, each row's cells"""
    rng = np.random.default_rng([int(seed) & 0xffffffff, 23, layer])
    got = [_body(rng, depth + t, clustered) for t in range(rows)]
    offsets = np.concatenate([[0], np.cumsum([4 * w.size for w, _ in got])])
    return np.concatenate([w for w, _ in got]).astype(np.int32), offsets.astype(np.int32), [c for _, c in got]


def _slab_body(seed, pos0, rows, clustered):
    """The rows' bodies in slabs of 128 rows: int32 words, offsets [slabs][129], each row's cells. A prompt's
    neighbouring rows select much the same blocks: a row keeps its neighbour's with some of them replaced."""
    rng = np.random.default_rng([int(seed) & 0xffffffff, 29])
    slabs = -(-rows // fnkv.SLAB_ROWS)
    words = np.zeros((slabs, fnkv.SLAB_ROWS * fnkv.ROW_WORDS), np.int32)
    offsets = np.zeros((slabs, fnkv.SLAB_ROWS + 1), np.int32)
    cells, last = [], None
    for t in range(rows):
        q = pos0 + t
        n_vis, k = (q + 1) // BLOCK, min((q + 1) // BLOCK, TOP)
        if last is None or not clustered or n_vis <= TOP or t % 16 == 0:
            w, c = _body(rng, q, clustered)
            last = w[2:2 + k]
        else:
            keep = rng.choice(last, k - 16, replace=False)
            new = rng.integers(0, n_vis, 64)
            new = np.concatenate([[n_vis - 1], new])
            new = new[~np.isin(new, keep)]
            new = new[np.sort(np.unique(new, return_index=True)[1])][:16]
            last = np.sort(np.concatenate([keep, new]))
            tail = np.arange(BLOCK * n_vis, q + 1)
            w = np.concatenate([[k, tail.size], last, tail])
            c = np.concatenate([(BLOCK * last[:, None] + np.arange(BLOCK)).reshape(-1), tail])
        s, i = divmod(t, fnkv.SLAB_ROWS)
        at = offsets[s, i] // 4
        words[s, at:at + w.size] = w
        offsets[s, i + 1:] = 4 * (at + w.size)
        cells.append(c)
    return words, offsets, cells


def _ctxs(case):
    return [max(int(c), case["T"]) for c in case["ctxs"].split(",")]


def _pool(case, cells, layers, seed):
    """A pool whose slots 0 .. n - 1 map `cells` each, grown a page at a time in a random order (scattered tables)"""
    need = [-(-c // PAGE) for c in cells]
    pool = fnkv.Pool(len(cells) + 1, sum(need) + 8, layers, case["hkv"], fmt=FORMATS[case["fmt"]])
    order = np.repeat(np.arange(len(cells)), need)
    rng = np.random.default_rng([int(seed) & 0xffffffff, 31])
    rng.shuffle(order)
    filler, have = len(cells), [0] * len(cells)
    assert pool.ensure(filler, 3 * PAGE)[0] == 0
    for i, s in enumerate(order):
        have[s] += 1
        assert pool.ensure(int(s), have[s] * PAGE)[0] == 0
        if i == len(order) // 2:
            assert pool.trim(filler, 0) == 0
    return pool


def _capture(step):
    """One step as a HIP graph, as the engine captures its layers once and replays them"""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def _dense_q(case, seed):
    shape = (case["layers"], len(_ctxs(case)), case["T"], case["hq"], D)
    return torch.randn(shape, generator=_gen(seed, 41), device="cuda").half()


def _prep_inputs(case, seed, layers, rows):
    """qfull, k, v, the norms of a call that prepares its rows"""
    g = _gen(seed, 43)
    return dict(qfull=_uniform(g, (layers, rows, case["hq"], 2 * D), -3.0, 3.0),
                kv_k=_uniform(g, (layers, rows, case["hkv"], D), -2.0, 2.0),
                kv_v=_uniform(g, (layers, rows, case["hkv"], D), -1.5, 1.5),
                q_norm=_uniform(g, (D,), 0.3, 1.8), k_norm=_uniform(g, (D,), 0.3, 1.8))


def prepare(case, seed):
    return {"dense": _dense, "qsa": _sparse_rows, "sparse": _sparse_rows, "prefill": _prefill, "qsp": _qsp,
            "datc": _datc}[case["kind"]](case, seed)


def run(state):
    return state["run"]()


def _dense(case, seed):
    ctxs, T, layers, hq = _ctxs(case), case["T"], case["layers"], case["hq"]
    # a captured launch serves the steps to come: its bound lies past the contexts
    bound = [c + 300 for c in ctxs] if case["captured"] else ctxs
    pool = _pool(case, bound, layers, seed)
    slots = list(range(len(ctxs)))
    new_k, new_v = [], []
    for layer in range(layers):
        for s, c in zip(slots, ctxs):
            k, v = _kv(seed, layer, s, c, case["hkv"])
            if c > T:
                pool.append(s, layer, 0, k[:c - T].contiguous(), v[:c - T].contiguous())
            new_k.append(k[c - T:])
            new_v.append(v[c - T:])
    dt = torch.float32 if case["new"] == "f32" else torch.float16
    shape = (layers, len(ctxs), T, case["hkv"], D)
    k_new, v_new = torch.stack(new_k).reshape(shape).to(dt), torch.stack(new_v).reshape(shape).to(dt)
    q = _dense_q(case, seed)
    out = torch.zeros_like(q)
    ws = torch.zeros(pool.decode_ws_bytes(bound, T, hq), dtype=torch.uint8, device="cuda")
    if not case["captured"]:
        def step():
            for i in range(layers):
                pool.decode(slots, ctxs, T, i, q[i], out[i], ws, k_new=k_new[i], v_new=v_new[i])
            return out
        return {"run": step}
    ctx_dev = torch.tensor(ctxs, dtype=torch.int64, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")

    def step():
        for i in range(layers):
            pool.decode_dev(slots, ctx_dev, bound, T, i, q[i], out[i], ws, err, k_new=k_new[i], v_new=v_new[i])

    graph = _capture(step)

    def replay():
        graph.replay()
        return out
    return {"run": replay, "keep": (pool, ws, ctx_dev, err, k_new, v_new, q)}


def _sparse_rows(case, seed):
    depth, rows, layers, hq, hkv = case["depth"], case["rows"], case["layers"], case["hq"], case["hkv"]
    pool = _pool(case, [depth + rows + 64], layers, seed)
    for layer in range(layers):
        k, v = _kv(seed, layer, 0, depth, hkv)
        pool.append(0, layer, 0, k, v)
    bodies = []
    for layer in range(layers):
        w, o, _ = _rows_body(seed, layer, depth, rows, case["clustered"])
        bodies.append((torch.from_numpy(w).cuda(), torch.from_numpy(o).cuda()))
    p = _prep_inputs(case, seed, layers, rows)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    depth_dev = torch.tensor([depth], dtype=torch.int32, device="cuda")
    max_cells = depth + rows + 64
    if case["kind"] == "sparse":
        q = torch.randn((layers, rows, hq, D), generator=_gen(seed, 41), device="cuda").half()
        kn, vn = p["kv_k"].half(), p["kv_v"].half()
        out = torch.zeros_like(q)
        ws = torch.empty(pool.sparse_ws_bytes(max_cells - rows, rows, hq), dtype=torch.uint8, device="cuda")

        def step():
            for i in range(layers):
                pool.sparse_dev(0, depth_dev, max_cells, i, q[i], bodies[i][0], bodies[i][1], out[i], ws, err,
                                k_new=kn[i], v_new=vn[i])
        outs = out
        keep = (pool, q, kn, vn, ws)
    else:
        pos = torch.arange(depth, depth + rows, dtype=torch.int32, device="cuda").repeat(4, 1).contiguous()
        out = torch.zeros((layers, rows, hq, D), device="cuda")
        codes = torch.zeros((layers, rows, hq * D), dtype=torch.int8, device="cuda")
        scales = torch.zeros((layers, rows, hq * 8, 2), device="cuda")
        ws = torch.empty(pool.attend_ws_bytes(max_cells, rows, hq), dtype=torch.uint8, device="cuda")
        args = [pool.attend_args(0, i, depth_dev, max_cells, p["qfull"][i], p["kv_k"][i], p["kv_v"][i], p["q_norm"],
                                 p["k_norm"], pos, bodies[i][0], bodies[i][1], out[i], codes[i], scales[i], ws, err)
                for i in range(layers)]

        def step():
            for a in args:
                fnkv.attend(rows, a)
        outs = {"out": out, "codes": codes, "scales": scales}
        keep = (pool, args, p)
    graph = _capture(step)

    def replay():
        graph.replay()
        return outs
    return {"run": replay, "keep": (keep, bodies, err, depth_dev)}


def _prefill(case, seed):
    ctx, rows, hq = case["ctx"], case["rows"], case["hq"]
    before = ctx - rows
    pool = _pool(case, [ctx], 1, seed)
    k, v = _kv(seed, 0, 0, ctx, case["hkv"])
    pool.append(0, 0, 0, k[:before].contiguous(), v[:before].contiguous())
    k, v = k[before:].contiguous(), v[before:].contiguous()
    q = torch.randn((rows, hq, D), generator=_gen(seed, 41), device="cuda").half()
    out = torch.zeros_like(q)
    ws = torch.empty(max(16, pool.prefill_ws_bytes(ctx, rows, hq)), dtype=torch.uint8, device="cuda")

    def step():
        pool.append(0, 0, before, k, v)
        pool.prefill(0, 0, ctx, q, out, ws=ws)
        return out
    return {"run": step}


def _qsp(case, seed):
    pos0, rows, hq, hkv = case["pos0"], case["rows"], case["hq"], case["hkv"]
    pool = _pool(case, [pos0 + rows], 1, seed)
    k, v = _kv(seed, 0, 0, pos0, hkv)
    pool.append(0, 0, 0, k, v)
    w, o, _ = _slab_body(seed, pos0, rows, case["clustered"])
    w, o = torch.from_numpy(w).cuda(), torch.from_numpy(o).cuda()
    p = _prep_inputs(case, seed, 1, rows)
    out16 = torch.zeros((rows, hq, D), dtype=torch.float16, device="cuda")
    out = torch.zeros((rows, hq, D), device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    ws = torch.empty(pool.qsp_ws_bytes(pos0, rows, hq), dtype=torch.uint8, device="cuda")

    def step():
        pool.qsp_kv(0, 0, pos0, p["kv_k"][0], p["kv_v"][0], p["k_norm"])
        pool.qsp_attend(0, 0, pos0, p["qfull"][0], p["q_norm"], w, o, out16, out=out, err=err, ws=ws)
        return {"out": out, "out16": out16}
    return {"run": step}


def _datc_inputs(case, seed):
    n, layers = case["cells"], case["layers"]
    g = _gen(seed, 47)
    return dict(caches=torch.randn((layers, 2, n + 8, D), generator=g, device="cuda").half(),
                qfull=_uniform(g, (layers, fnkv.DATC_HEADS, 2 * D), -3.0, 3.0),
                kv=_uniform(g, (layers, 2, 1, D), -2.0, 2.0), norms=_uniform(g, (2, D), 0.3, 1.8))


def _datc(case, seed):
    n, layers = case["cells"], case["layers"]
    p = _datc_inputs(case, seed)
    caches = p["caches"].view(torch.int16)
    ints = torch.tensor([n - 1, 1], dtype=torch.int32, device="cuda")
    pos = torch.full((4, 1), n - 1, dtype=torch.int32, device="cuda")
    heads = fnkv.DATC_HEADS
    q16 = torch.zeros((layers, heads, D), dtype=torch.int16, device="cuda")
    part = torch.empty(fnkv.datc_part_bytes() // 4, device="cuda")
    out = torch.zeros((layers, heads * D), device="cuda")
    codes = torch.zeros((layers, heads * D), dtype=torch.int8, device="cuda")
    scales = torch.zeros((layers, heads * 8, 2), device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")

    def step():
        for i in range(layers):
            fnkv.datc_step(kv_k=p["kv"][i, 0], kv_v=p["kv"][i, 1], k_norm=p["norms"][1], n_before=ints[0:1], pos=pos,
                           stride=ints[1:2], k_cache=caches[i, 0], v_cache=caches[i, 1], err=err,
                           qfull=p["qfull"][i], q_norm=p["norms"][0], q16=q16[i], part=part, out=out[i],
                           codes=codes[i], scales=scales[i])

    graph = _capture(step)
    outs = {"out": out, "codes": codes, "scales": scales, "k_row": caches[:, 0, n - 1].view(torch.float16)}

    def replay():
        graph.replay()
        return outs
    return {"run": replay, "keep": (p, caches, ints, pos, q16, part, err)}


# ---- what a pass cannot do without ----

def work(case):
    kind = case["kind"]
    if kind == "datc":
        n, layers, h = case["cells"], case["layers"], fnkv.DATC_HEADS
        return {"bytes": layers * (n * 1024 + h * D * (8 + 2 + 5) + h * 64 + 4 * D * 4),
                "flops": layers * 4 * D * h * n}
    hq, hkv = case["hq"], case["hkv"]
    cell = hkv * 2 * (D + 16)
    if kind == "dense":
        ctxs, T, layers = _ctxs(case), case["T"], case["layers"]
        new = T * hkv * 2 * D * (4 if case["new"] == "f32" else 2)
        by = sum(c * cell + T * cell + new + T * hq * D * 4 for c in ctxs)
        pairs = sum(T * (c - T) + T * (T + 1) // 2 for c in ctxs)
        return {"bytes": layers * by, "flops": layers * 4 * D * hq * pairs}
    if kind in ("qsa", "sparse"):
        rows, layers = case["rows"], case["layers"]
        sel = sum(min((q + 1) // BLOCK, TOP) * BLOCK + (q + 1) % BLOCK
                  for q in range(case["depth"], case["depth"] + rows))
        read = min(sel, case["depth"] + rows)
        per = hq * D * (8 + 5) + hq * 64 + hkv * D * 8 if kind == "qsa" else hq * D * 4 + hkv * D * 4
        return {"bytes": layers * (read * cell + rows * (per + cell)), "flops": layers * 4 * D * hq * sel}
    rows = case["rows"]
    if kind == "prefill":
        ctx = case["ctx"]
        pairs = rows * (ctx - rows) + rows * (rows + 1) // 2
        return {"bytes": ctx * cell + rows * (cell + hkv * D * 4 + hq * D * 4), "flops": 4 * D * hq * pairs}
    q = range(case["pos0"], case["pos0"] + rows)
    sel = sum(min((x + 1) // BLOCK, TOP) * BLOCK + (x + 1) % BLOCK for x in q)
    read = min(sel, case["pos0"] + rows)
    return {"bytes": read * cell + rows * (cell + hkv * D * 8 + hq * D * (8 + 4 + 2)), "flops": 4 * D * hq * sel}


# ---- the outputs in 64 bits, without the library ----

def _quantized(x, fmt):
    """Rows through the pool's 8-bit format and back, in 64 bits: Q8_0 (an fp16 scale a 32-value block, codes
    roundf(x / d)) or KV8 (an fp16 scale a 64-value group, codes rint(x / fp16 scale)); the code rules are F32's"""
    x = x.float()
    n = 64 if fmt == "kv8" else 32
    b = x.reshape(*x.shape[:-1], D // n, n)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    if fmt == "kv8":
        s = d.half().float()
        c = torch.where(s > 0, torch.clamp(torch.round(b / s), -127, 127), torch.zeros_like(b))
        return (c.double() * s.double()).reshape(x.shape)
    r = b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    t = torch.trunc(r)
    c = torch.where((r - t).abs() >= 0.5, t + torch.sign(r), t)
    return (c.double() * d.half().double()).reshape(x.shape)


def _theta_scale():
    return np.float32(np.float32(10000000.0) ** np.float32(-2.0 / 64.0))


def _norm_rope(x, g, pos):
    """RMS norm and rotation of rows [rows][heads][256] at positions pos[rows] (every plane), 64 bits over the F32
    angles (the F32 product chain)"""
    x = x.double()
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g.double()
    th = np.asarray(pos, np.float32)[:, None].repeat(32, 1)
    for i in range(1, 32):
        th[:, i] = th[:, i - 1] * _theta_scale()
    a = torch.from_numpy(th.astype(np.float64)).cuda()[:, None, :]
    c, s = torch.cos(a), torch.sin(a)
    lo, hi = y[..., :32].clone(), y[..., 32:64].clone()
    y[..., :32] = lo * c - hi * s
    y[..., 32:64] = lo * s + hi * c
    return y


def _attend(q, k, v, limit=None):
    """q [rows][heads][256], k, v [cells][256], 64 bits; limit[rows]: the cells each row sees"""
    rows, heads = q.shape[:2]
    o = torch.empty_like(q)
    step = max(1, int(2e9 // (8 * k.shape[0] * heads)))
    for a in range(0, rows, step):
        z = q[a:a + step].reshape(-1, D) @ k.t()
        z = z.reshape(-1, heads, k.shape[0]) / 16.0
        if limit is not None:
            hide = torch.arange(k.shape[0], device="cuda")[None, :] >= limit[a:a + step][:, None]
            z.masked_fill_(hide[:, None, :], -math.inf)
        p = torch.softmax(z, -1)
        o[a:a + step] = (p.reshape(-1, k.shape[0]) @ v).reshape(-1, heads, D)
    return o


def _attend_cells(q, k, v, cells, g_heads):
    """q [rows][heads][256] over each row's own cells of k, v [cells][hkv][256], 64 bits"""
    o = torch.empty_like(q)
    for t, c in enumerate(cells):
        at = torch.from_numpy(np.asarray(c, np.int64)).cuda()
        for h in range(k.shape[1]):
            s = slice(h * g_heads, (h + 1) * g_heads)
            p = torch.softmax(q[t, s] @ k[at, h].t() / 16.0, -1)
            o[t, s] = p @ v[at, h]
    return o


def exact(case, seed):
    kind = case["kind"]
    if kind == "datc":
        return _exact_datc(case, seed)
    hq, hkv, fmt = case["hq"], case["hkv"], case["fmt"]
    g = hq // hkv
    if kind == "dense":
        T = case["T"]
        q = _dense_q(case, seed).double()
        o = torch.empty_like(q)
        for layer in range(case["layers"]):
            for s, c in enumerate(_ctxs(case)):
                k, v = (_quantized(x, fmt) for x in _kv(seed, layer, s, c, hkv))
                limit = torch.arange(c - T + 1, c + 1, device="cuda")
                for h in range(hkv):
                    at = slice(h * g, (h + 1) * g)
                    o[layer, s, :, at] = _attend(q[layer, s, :, at].contiguous(), k[:, h].contiguous(),
                                                 v[:, h].contiguous(), limit)
        return o
    if kind == "prefill":
        ctx, rows = case["ctx"], case["rows"]
        k, v = (_quantized(x, fmt) for x in _kv(seed, 0, 0, ctx, hkv))
        q = torch.randn((rows, hq, D), generator=_gen(seed, 41), device="cuda").half().double()
        limit = torch.arange(ctx - rows + 1, ctx + 1, device="cuda")
        o = torch.empty_like(q)
        for h in range(hkv):
            at = slice(h * g, (h + 1) * g)
            o[:, at] = _attend(q[:, at].contiguous(), k[:, h].contiguous(), v[:, h].contiguous(), limit)
        return o
    if kind == "qsp":
        pos0, rows = case["pos0"], case["rows"]
        p = _prep_inputs(case, seed, 1, rows)
        pos = np.arange(pos0, pos0 + rows)
        k, v = _kv(seed, 0, 0, pos0, hkv)
        k = torch.cat([_quantized(k, fmt), _quantized(_norm_rope(p["kv_k"][0], p["k_norm"], pos), fmt)])
        v = torch.cat([_quantized(v, fmt), _quantized(p["kv_v"][0], fmt)])
        q = _norm_rope(p["qfull"][0][..., :D], p["q_norm"], pos)
        cells = _slab_body(seed, pos0, rows, case["clustered"])[2]
        o = _attend_cells(q, k, v, cells, g) * torch.sigmoid(p["qfull"][0][..., D:].double())
        return {"out": o, "out16": o}
    depth, rows, layers = case["depth"], case["rows"], case["layers"]
    p = _prep_inputs(case, seed, layers, rows)
    pos = np.arange(depth, depth + rows)
    o = torch.empty((layers, rows, hq, D), dtype=torch.float64, device="cuda")
    if kind == "sparse":
        q = torch.randn((layers, rows, hq, D), generator=_gen(seed, 41), device="cuda").half().double()
    for layer in range(layers):
        k, v = _kv(seed, layer, 0, depth, hkv)
        if kind == "qsa":
            kn, vn = _norm_rope(p["kv_k"][layer], p["k_norm"], pos), p["kv_v"][layer]
            ql = _norm_rope(p["qfull"][layer][..., :D], p["q_norm"], pos)
        else:
            kn, vn, ql = p["kv_k"][layer].half(), p["kv_v"][layer].half(), q[layer]
        k = torch.cat([_quantized(k, fmt), _quantized(kn, fmt)])
        v = torch.cat([_quantized(v, fmt), _quantized(vn, fmt)])
        o[layer] = _attend_cells(ql, k, v, _rows_body(seed, layer, depth, rows, case["clustered"])[2], g)
        if kind == "qsa":
            o[layer] *= torch.sigmoid(p["qfull"][layer][..., D:].double())
    return {"out": o, "codes": None, "scales": None} if kind == "qsa" else o


def _exact_datc(case, seed):
    n, layers = case["cells"], case["layers"]
    p = _datc_inputs(case, seed)
    at = np.array([n - 1])
    o = torch.empty((layers, fnkv.DATC_HEADS * D), dtype=torch.float64, device="cuda")
    rows = []
    for i in range(layers):
        q = _norm_rope(p["qfull"][i][None, :, :D], p["norms"][0], at)
        k, v = p["caches"][i, 0, :n].double(), p["caches"][i, 1, :n].double()
        row = _norm_rope(p["kv"][i, 0][None], p["norms"][1], at)[0, 0]
        k[n - 1], v[n - 1] = row.half().double(), p["kv"][i, 1, 0].half().double()
        rows.append(row)
        o[i] = (_attend(q, k, v)[0] * torch.sigmoid(p["qfull"][i][:, D:].double())).reshape(-1)
    return {"out": o, "codes": None, "scales": None, "k_row": torch.stack(rows)}


def tolerance(case):
    # About four times the largest distance from exact() that the path showed over these ranges: fp16 outputs alone
    # are 2.5e-4 off; 2e-3 in the deepest dense contexts and 1.1e-3 over 2,051 selected cells, whose weights times V
    # scales reach the bottom of fp16's range; 7e-5 for the F32 attention (a new cell's code one step off counts
    # there). A code of the activation format differs where the value is at a tie.
    return {"dense": {"rel": 8e-3, "max": 0.06}, "prefill": {"rel": 1e-3, "max": 0.02},
            "sparse": {"rel": 4.5e-3, "max": 0.06}, "qsp": {"rel": 4.5e-3, "max": 0.06},
            "qsa": {"rel": 3e-4, "max": 0.01, "differ": 2e-3},
            "datc": {"rel": 1.2e-3, "max": 0.02, "differ": 0.01}}[case["kind"]]
