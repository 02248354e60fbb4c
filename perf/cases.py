"""Workloads of the library's main path, one attention or DeltaNet layer's work a case.

listed() names the cases, draw(rng) makes another one of the same ranges,
prepare(case, seed) builds what a serving program holds before the call (caches,
weights, inputs, descriptors, workspaces) on the GPU, run(state) is one pass through
the public entry points, work(case) its compulsory bytes and operations,
tolerance(case) the error a correct implementation may show, and exact(case, seed)
the results in float64 from plain torch.

Shapes: 2 KV heads of 256 and 16 query heads (the benchmark's configurations) or 24
(the reference's model); q8_0 caches with N(0, 1) rows and 4 outlier channels a head;
48 / 16 DeltaNet value / key heads of 128; QSA blocks of 4 cells, 513 kept, 4 indexer
heads of 128.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qwfn-hybrid_amd"))

import qwfn_kv as K  # noqa: E402
import qwfn_state as S  # noqa: E402

HD, NKV, ROW = 256, 2, 544          # head size, KV heads, bytes of a q8_0 cache row
RATIO, KB, IDX, IDX_H = 4, 513, 128, 4   # QSA: cells a block, blocks kept, indexer key size and heads
N_EMBD = 2560
DN_K, DN_V, DN_D = 16, 48, 128      # DeltaNet key heads, value heads, head size


def listed():
    return [
        # one decoded token after a short prompt: the smallest call, append and attention in one launch
        dict(name="decode_T1_h24_513", kind="decode", T=1, depth=513, heads=24),
        # the benchmark's step: 1 + 2 drafted tokens verified at 16K
        dict(name="verify_T3_h16_16384", kind="decode", T=3, depth=16384, heads=16),
        # the same at the benchmark's long context
        dict(name="verify_T3_h16_65536", kind="decode", T=3, depth=65536, heads=16),
        # the same step at the reference model's 24 heads, an odd depth (its dense path: the MTP head, QSA off)
        dict(name="verify_T3_h24_12295", kind="decode", T=3, depth=12295, heads=24),
        # four conversations of different depths decoded together
        dict(name="batch4_8k_64k", kind="batch", depths="8192,16384,32768,65536", heads=16),
        # the first chunk of a prompt: append of 512 rows, causal attention, output gate
        dict(name="prefill_512_at_0", kind="prefill", T=512, depth=0, heads=16),
        # a late, ragged chunk of a long prompt (the largest case)
        dict(name="prefill_509_at_16387", kind="prefill", T=509, depth=16387, heads=16),
        # one layer of the reference's default verify step (QSA on): inputs and index pooling, block
        # selection, K/V producer, gated attention over each position's cells
        dict(name="qsa_step_T3_73700", kind="qsa_step", T=3, depth=73700, heads=24, bf16=False),
        # the selection side of a QSA-on prefill chunk: block tables, pooled keys, top blocks, visible cells
        dict(name="qsa_chunk_512_at_16384", kind="qsa_chunk", T=512, depth=16384),
        # the attention of that chunk over the lists
        dict(name="qsa_attend_512_at_16384", kind="qsa_attend", T=512, depth=16384, heads=16),
        # the recurrent update of a verify step with its rollback snapshots (36 of the 48 layers)
        dict(name="delta_T3", kind="delta", T=3, snaps=2),
        # the same layer over a prefill chunk
        dict(name="delta_T512", kind="delta", T=512, snaps=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "prefill", "prefill", "qsa_step", "qsa_chunk", "qsa_attend",
                       "delta", "delta"])
    heads = rng.choice([16, 24])
    if kind == "decode":
        return dict(kind=kind, T=rng.randint(1, 4), depth=_log_int(rng, 256, 65536), heads=heads)
    if kind == "batch":
        d = [_log_int(rng, 512, 65536) for _ in range(rng.randint(2, 8))]
        while sum(d) > 131072:
            d[d.index(max(d))] //= 2
        return dict(kind=kind, depths=",".join(str(x) for x in d), heads=heads)
    if kind == "prefill":
        T = _log_int(rng, 64, 512)
        depth = 0 if rng.random() < 0.25 else _log_int(rng, 256, 16387)
        if heads * T > 16 * 509:
            T = 16 * 509 // heads
        return dict(kind=kind, T=T, depth=depth, heads=heads)
    if kind == "qsa_step":
        return dict(kind=kind, T=rng.randint(1, 4), depth=_log_int(rng, 4096, 131072), heads=heads,
                    bf16=rng.random() < 0.5)
    if kind == "qsa_chunk":
        return dict(kind=kind, T=_log_int(rng, 64, 512), depth=4 * _log_int(rng, 1024, 16384))
    if kind == "qsa_attend":
        return dict(kind=kind, T=_log_int(rng, 64, 512), depth=_log_int(rng, 4096, 65536), heads=heads)
    if rng.random() < 0.3:
        T = rng.randint(1, 4)
        return dict(kind="delta", T=T, snaps=T - 1)
    return dict(kind="delta", T=_log_int(rng, 8, 512), snaps=0)


# ---------------------------------------------------------------- inputs

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32)


def _quant(x):
    """F32 rows [n, 32 k] as q8_0 blocks (d = amax / 127 in F16, q = x * (127 / amax) rounded half to
    even): (q int8 [n, k, 32], d F16 [n, k])."""
    b = x.reshape(x.shape[0], -1, 32)
    amax = b.abs().amax(dim=2)
    # quotients rounded once to float32 (a float64 quotient, then float32)
    inv = torch.where(amax > 0, (127.0 / amax.double()).float(), torch.zeros_like(amax))
    return torch.round(b * inv[:, :, None]).to(torch.int8), (amax.double() / 127.0).float().to(torch.float16)


def _pack(x):
    """F32 rows as q8_0 cache bytes [n, 34 k]."""
    q, d = _quant(x)
    n, k = d.shape
    out = torch.empty((n, k, 34), dtype=torch.uint8, device=x.device)
    out[:, :, :2] = d.contiguous().view(torch.uint8).reshape(n, k, 2)
    out[:, :, 2:] = q.view(torch.uint8)
    return out.reshape(n, k * 34)


def _rows(g, n):
    """F32 K or V rows [n, 512]: N(0, 1), 4 channels of each head 8 times larger."""
    x = _randn(g, n, NKV * HD)
    ch = torch.stack([torch.randperm(HD, generator=g, device="cuda")[:4] + h * HD for h in range(NKV)]).reshape(-1)
    x[:, ch] *= 8.0
    return x


def _cache(g, n, room):
    """A q8_0 cache of n + room rows, the first n filled."""
    c = torch.zeros((n + room, ROW), dtype=torch.uint8, device="cuda")
    if n:
        c[:n] = _pack(_rows(g, n))
    return c


def _unpack(cache):
    """Cache bytes [n, 544] as float64 values [n, 2, 256]."""
    b = cache.reshape(cache.shape[0], -1, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).reshape(cache.shape[0], NKV, HD)


def _causal(T, n_kv, depth):
    keys = torch.arange(n_kv, device="cuda")[None, :]
    rows = torch.arange(T, device="cuda")[:, None]
    zero = torch.zeros((), dtype=torch.float16, device="cuda")
    return torch.where(keys <= depth + rows, zero, torch.full_like(zero, float("-inf")))


def _ws(n):
    return torch.empty(max(256, int(n)), dtype=torch.uint8, device="cuda")


def _delta_inputs(case, g):
    T = case["T"]
    conv = _randn(g, T, 2 * DN_K * DN_D + DN_V * DN_D)
    qk = conv[:, :2 * DN_K * DN_D].reshape(T, 2 * DN_K, DN_D)
    conv[:, :2 * DN_K * DN_D] = (qk / qk.norm(dim=2, keepdim=True)).reshape(T, -1)
    # log decay: heads with short and with long memory
    rate = torch.exp(_rand(g, 1, DN_V) * math.log(500.0)) * 0.003
    return dict(conv=conv, g=-_rand(g, T, DN_V) * rate, beta=torch.sigmoid(_randn(g, T, DN_V)),
                state=_randn(g, DN_V, DN_D, DN_D) * 0.05)


def _distinct_lists(g, T, depth, n_kv):
    """Each query's cells as the selection leaves them: 512 whole blocks of 4 and the cells of its own
    block, ascending; the rest of the row zero."""
    width = KB * RATIO
    lists = torch.zeros((T, width), dtype=torch.int32, device="cuda")
    counts = torch.zeros((T,), dtype=torch.int32, device="cuda")
    for t in range(T):
        own = (depth + t) // RATIO
        blk = torch.randperm(own, generator=g, device="cuda")[:KB - 1].sort().values
        cells = (blk[:, None] * RATIO + torch.arange(RATIO, device="cuda")[None, :]).reshape(-1)
        cells = torch.cat([cells, torch.arange(own * RATIO, depth + t + 1, device="cuda")])
        lists[t, :cells.numel()] = cells.to(torch.int32)
        counts[t] = cells.numel()
    return lists, counts


def _qsa_ctx(case):
    return (case["depth"] + case["T"] + 31) // 32 * 32


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    kind, g = case["kind"], _gen(seed)
    if kind == "decode":
        T, d, nh = case["T"], case["depth"], case["heads"]
        return dict(kc=_cache(g, d, T), vc=_cache(g, d, T), k=_rows(g, T), v=_rows(g, T), q=_randn(g, 1, T, nh, HD),
                    mask=_causal(T, d + T, d) if T > 1 else None)
    if kind == "batch":
        depths = [int(x) for x in case["depths"].split(",")]
        n = max(depths)
        kc = torch.zeros((len(depths), n, ROW), dtype=torch.uint8, device="cuda")
        vc = torch.zeros_like(kc)
        for b, d in enumerate(depths):
            kc[b, :d], vc[b, :d] = _cache(g, d, 0), _cache(g, d, 0)
        return dict(depths=depths, kc=kc, vc=vc, q=_randn(g, len(depths), 1, case["heads"], HD))
    if kind == "prefill":
        T, d, nh = case["T"], case["depth"], case["heads"]
        return dict(kc=_cache(g, d, T), vc=_cache(g, d, T), k=_rows(g, T), v=_rows(g, T), q=_randn(g, 1, T, nh, HD),
                    gate=_randn(g, 1, T, nh, HD), mask=_causal(T, d + T, d))
    if kind == "qsa_step":
        T, d, nh, n = case["T"], case["depth"], case["heads"], _qsa_ctx(case)
        wt = torch.bfloat16 if case["bf16"] else torch.float16
        return dict(kc=_cache(g, d, n - d), vc=_cache(g, d, n - d), ic=_randn(g, n, IDX).to(torch.float16),
                    pool=(_randn(g, n // RATIO, IDX)).to(torch.float16), k_raw=_randn(g, T, IDX),
                    knw_idx=_rand(g, IDX) + 0.5, q_idx=_randn(g, T, IDX_H, IDX), cur=_randn(g, T, N_EMBD),
                    wk=(_randn(g, NKV * HD, N_EMBD) * 0.02).to(wt), wv=(_randn(g, NKV * HD, N_EMBD) * 0.02).to(wt),
                    knw=_rand(g, HD) + 0.5, q=_randn(g, 1, T, nh, HD), gate=_randn(g, 1, T, nh, HD))
    if kind == "qsa_chunk":
        T, d = case["T"], case["depth"]
        n_kv = (d + T) // RATIO * RATIO
        return dict(T=n_kv - d, n_kv=n_kv, ic=_randn(g, n_kv, IDX).to(torch.float16), knw_idx=_rand(g, IDX) + 0.5,
                    q_idx=_randn(g, n_kv - d, IDX_H, IDX))
    if kind == "qsa_attend":
        T, d, nh = case["T"], case["depth"], case["heads"]
        lists, counts = _distinct_lists(g, T, d, d + T)
        return dict(kc=_cache(g, d + T, 0), vc=_cache(g, d + T, 0), q=_randn(g, 1, T, nh, HD),
                    gate=_randn(g, 1, T, nh, HD), lists=lists, counts=counts)
    return _delta_inputs(case, g)


def prepare(case, seed):
    K.check(K.load().qwfn_init(0))
    s = _inputs(case, seed)
    kind = s["kind"] = case["kind"]
    s["case"] = case
    if kind in ("decode", "prefill", "qsa_attend"):
        n_kv = case["depth"] + case["T"]
        s["out"] = torch.zeros_like(s["q"])
        s["qv"], s["ov"] = K.q_view(s["q"]), K.out_view(s["out"])
        s["kv"], s["vv"] = K.cache_attn_view(s["kc"], n_kv, NKV), K.cache_attn_view(s["vc"], n_kv, NKV)
        if kind != "qsa_attend":
            s["mv"] = K.mask_view(s["mask"]) if s["mask"] is not None else None
            s["ws"] = _ws(K.fattn_workspace_size(s["qv"], s["kv"], s["vv"], s["mv"]))
    elif kind == "batch":
        B, n = len(s["depths"]), s["kc"].shape[1]
        s["out"] = torch.zeros_like(s["q"])
        s["qv"], s["ov"] = K.q_view(s["q"]), K.out_view(s["out"])
        s["kv"], s["vv"] = (K.cache_attn_view(c, n, NKV, batch=B, batch_stride=n * ROW) for c in (s["kc"], s["vc"]))
        s["ws"] = _ws(K.fattn_workspace_size_seq(s["qv"], s["kv"], s["vv"], None, s["depths"]))
    elif kind == "qsa_step":
        T, d, n = case["T"], case["depth"], _qsa_ctx(case)
        nb = n // RATIO
        s["bias"] = torch.empty((T, nb), dtype=torch.float32, device="cuda")
        s["qds"] = [S.QsaDecodeInputs(RATIO, nb) for _ in range(T)]
        for t in range(T):
            s["qds"][t].bias = s["bias"][t]
        s["qds"][0].rebuild_bias(d)
        s["blk_cells"] = torch.empty(nb * RATIO, dtype=torch.int32, device="cuda")
        S.qsa_tables(s["blk_cells"], RATIO)
        s["pos"] = torch.arange(d, d + T, dtype=torch.int32, device="cuda").repeat(4)
        s["cells"] = torch.zeros((T, KB * RATIO), dtype=torch.int32, device="cuda")
        s["wsel"] = _ws(K.load().qwfn_qsa_select_workspace_size(nb, T))
        s["out"] = torch.zeros_like(s["q"])
        s["qv"], s["ov"] = K.q_view(s["q"]), K.out_view(s["out"])
        s["kv"], s["vv"] = K.cache_attn_view(s["kc"], n, NKV), K.cache_attn_view(s["vc"], n, NKV)
        s["counts"] = [KB * RATIO] * T
        s["ws"] = _ws(K.fattn_workspace_size_query_cells(s["qv"], s["kv"], s["vv"], s["counts"], KB * RATIO))
    elif kind == "qsa_chunk":
        T, nb = s["T"], s["n_kv"] // RATIO
        s["blk_cells"] = torch.empty(nb * RATIO, dtype=torch.int32, device="cuda")
        s["blk_pos"] = torch.empty(4 * nb, dtype=torch.int32, device="cuda")
        s["bias"] = torch.empty((T, nb), dtype=torch.float32, device="cuda")
        s["pool"] = torch.empty((nb, IDX), dtype=torch.float16, device="cuda")
        s["cells"] = torch.zeros((T, KB * RATIO), dtype=torch.int32, device="cuda")
        s["lists"] = torch.zeros((T, KB * RATIO), dtype=torch.int32, device="cuda")
        s["counts"] = torch.zeros((T,), dtype=torch.int32, device="cuda")
        s["wsel"] = _ws(K.load().qwfn_qsa_select_workspace_size(nb, T))
    else:
        T = case["T"]
        s["out"] = torch.zeros((T, DN_V, DN_D), dtype=torch.float32, device="cuda")
        s["snap"] = torch.zeros((case["snaps"], DN_V, DN_D, DN_D), dtype=torch.float32, device="cuda") \
            if case["snaps"] else None
        n = DN_K * DN_D
        s["qkv"] = s["conv"][:, :n], s["conv"][:, n:2 * n], s["conv"][:, 2 * n:]
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "decode":
        K.flash_attn_ext_append(s["qv"], s["kv"], s["vv"], s["mv"], 1 / 16, s["ov"], s["k"], s["v"], case["depth"],
                                ws=s["ws"])
        return dict(out=s["out"], kc=s["kc"], vc=s["vc"])
    if kind == "batch":
        K.flash_attn_ext_seq(s["qv"], s["kv"], s["vv"], None, 1 / 16, s["ov"], s["depths"], ws=s["ws"])
        return dict(out=s["out"])
    if kind == "prefill":
        K.cpy_f32_q8_0_kv(s["k"], s["kc"], s["v"], s["vc"], case["depth"])
        K.flash_attn_ext_gated(s["qv"], s["kv"], s["vv"], s["mv"], 1 / 16, s["ov"], s["gate"], ws=s["ws"])
        return dict(out=s["out"], kc=s["kc"], vc=s["vc"])
    if kind == "qsa_step":
        d = case["depth"]
        S.qsa_decode_prepare_pool_steps(s["qds"], d, s["ic"], s["k_raw"], s["knw_idx"], s["pool"])
        S.qsa_select_cells(s["pool"], s["q_idx"], s["bias"], KB, s["blk_cells"], RATIO, s["cells"], ws=s["wsel"])
        K.kv_produce(s["cur"], s["wk"], s["wv"], s["knw"], s["pos"], s["kc"], s["vc"], d)
        K.flash_attn_ext_query_cells(s["qv"], s["kv"], s["vv"], s["cells"], s["counts"], d, 1 / 16, s["ov"],
                                     gate=s["gate"], ws=s["ws"])
        return dict(out=s["out"], cells=s["cells"], bias=s["bias"], pool=s["pool"], ic=s["ic"], kc=s["kc"], vc=s["vc"])
    if kind == "qsa_chunk":
        d = case["depth"]
        S.qsa_chunk_inputs(d, s["T"], RATIO, None, s["blk_cells"], s["blk_pos"], s["bias"])
        K.qsa_pool_rebuild(s["ic"], s["n_kv"], RATIO, s["knw_idx"], s["pool"])
        S.qsa_select_cells(s["pool"], s["q_idx"], s["bias"], KB, s["blk_cells"], RATIO, s["cells"], ws=s["wsel"])
        S.qsa_visible_cells(s["cells"], s["n_kv"], d, s["lists"], s["counts"])
        return dict(cells=s["cells"], lists=s["lists"], counts=s["counts"], bias=s["bias"], pool=s["pool"],
                    blk_cells=s["blk_cells"], blk_pos=s["blk_pos"])
    if kind == "qsa_attend":
        K.flash_attn_ext_query_cells_dev(s["qv"], s["kv"], s["vv"], s["lists"], s["counts"], case["depth"], 1 / 16,
                                         s["ov"], gate=s["gate"])
        return dict(out=s["out"])
    q, k, v = s["qkv"]
    K.gated_delta_net(q, k, v, s["g"], s["beta"], s["state"], s["out"], DN_K, s["snap"], case["snaps"])
    return dict(out=s["out"], state=s["state"], snap=s["snap"])


# ---------------------------------------------------------------- pricing

def work(case):
    kind = case["kind"]
    T = case.get("T", 1)
    qo = 2 * T * case.get("heads", 0) * HD * 4
    if kind == "decode":
        n = case["depth"] + T
        pairs = T * case["depth"] + T * (T + 1) // 2
        return dict(bytes=n * 2 * ROW + T * 2 * (2048 + ROW) + qo + (2 * T * n if T > 1 else 0),
                    flops=4 * case["heads"] * HD * pairs)
    if kind == "batch":
        d = [int(x) for x in case["depths"].split(",")]
        return dict(bytes=sum(d) * 2 * ROW + 2 * len(d) * case["heads"] * HD * 4, flops=4 * case["heads"] * HD * sum(d))
    if kind == "prefill":
        n = case["depth"] + T
        pairs = T * case["depth"] + T * (T + 1) // 2
        return dict(bytes=n * 2 * ROW + T * 2 * (2048 + ROW) + qo * 3 // 2 + 2 * T * n,
                    flops=4 * case["heads"] * HD * pairs)
    if kind == "qsa_step":
        nb = _qsa_ctx(case) // RATIO
        seen = min(case["depth"], T * KB * RATIO)
        return dict(bytes=nb * IDX * 2 + T * nb * 8 + 2 * NKV * HD * N_EMBD * 2 + seen * 2 * ROW + qo * 3 // 2,
                    flops=2 * T * nb * IDX_H * IDX + 4 * T * NKV * HD * N_EMBD + 4 * case["heads"] * HD * T * KB * RATIO)
    if kind == "qsa_chunk":
        n_kv = (case["depth"] + T) // RATIO * RATIO
        T, nb = n_kv - case["depth"], n_kv // RATIO
        return dict(bytes=n_kv * IDX * 2 + nb * (IDX * 2 + 4 * RATIO + 16) + T * (nb * 4 + IDX_H * IDX * 4 + 2 * KB * RATIO * 4),
                    flops=2 * T * nb * IDX_H * IDX)
    if kind == "qsa_attend":
        return dict(bytes=(case["depth"] + T) * 2 * ROW + qo * 3 // 2 + T * KB * RATIO * 4,
                    flops=4 * case["heads"] * HD * T * (KB - 1) * RATIO)
    state = DN_V * DN_D * DN_D
    return dict(bytes=4 * (state * (2 + case["snaps"]) + T * (2 * DN_K * DN_D + 2 * DN_V * DN_D + 2 * DN_V)),
                flops=7 * T * state)


def tolerance(case):
    """About four times the error against float64 of the float32-accumulating kernels over the ranges of
    draw(): attention 2e-6 .. 8e-6 (float32 scores through exp), DeltaNet 5e-8 .. 7e-7, the F16 pooled
    keys 6e-6 (single roundings of an F16 step). Scores that agree to a rounding exchange places in the
    selection: 5e-4 of a chunk's cells, and one exchange moves up to 1/3 of a short chunk's list."""
    kind = case["kind"]
    if kind == "delta":
        return {"rel": 3e-6}
    if kind == "qsa_chunk":
        return {"rel": 2.5e-5, "differ": 5e-3}
    if kind == "qsa_step":
        return {"rel": 3e-5, "differ": 3e-3}
    if kind == "decode":
        return {"rel": 2e-5, "differ": 1e-6}
    return {"rel": 3e-5, "differ": 1e-6}


# ---------------------------------------------------------------- float64 results

def _attend64(q, k, v, visible=None):
    """q [n, 256] quantised to q8_0 as the op defines it, k and v [keys, 256] float64, visible [n, keys]."""
    qq, qd = _quant(q.reshape(-1, HD))
    qf = (qq.double() * qd.double()[:, :, None]).reshape(-1, HD)
    s = qf @ k.t() / 16
    if visible is not None:
        s = torch.where(visible, s, torch.full_like(s[:1, :1], float("-inf")))
    return torch.softmax(s, dim=1) @ v


def _attend_layer64(q, kc, vc, depth):
    """Causal attention of q [1, T, heads, 256] at depth over the caches."""
    _, T, nh, _ = q.shape
    k, v, g = _unpack(kc), _unpack(vc), nh // NKV
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    vis = torch.arange(kc.shape[0], device=q.device)[None, :] <= depth + torch.arange(T, device=q.device)[:, None]
    for h in range(nh):
        out[0, :, h] = _attend64(q[0, :, h].contiguous(), k[:, h // g], v[:, h // g], vis)
    return out


def _rope64(x, pos):
    """IMROPE of [n, dims] at equal positions [n]: pairs (i, i + 32), the angle the running float32
    product ggml forms."""
    step = torch.tensor(1e7, dtype=torch.float32).pow(torch.tensor(-2.0 / 64, dtype=torch.float32)).to(x.device)
    th = pos.to(torch.float32)
    y = x.clone()
    for i in range(32):
        c, s = torch.cos(th.double()), torch.sin(th.double())
        y[:, i], y[:, i + 32] = x[:, i] * c - x[:, i + 32] * s, x[:, i] * s + x[:, i + 32] * c
        th = th * step
    return y


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-6) * w.double()


def _pool64(ic, blocks, knw):
    members = blocks[:, None] * RATIO + torch.arange(RATIO, device=ic.device)[None, :]
    return _rope64(_norm64(ic[members].double().mean(dim=1), knw), blocks * RATIO).to(torch.float16)


def _top64(pool, q_idx, bias):
    """The kept blocks, best first, ties to the lower block."""
    score = torch.zeros((q_idx.shape[0], pool.shape[0]), dtype=torch.float64, device=pool.device)
    for h in range(IDX_H):
        score += torch.relu(q_idx[:, h].to(torch.float16).double() @ pool.double().t())
    score = score.to(torch.float32) + bias
    return torch.sort(score, dim=1, descending=True, stable=True).indices[:, :KB]


def _cells(top):
    return (top[:, :, None] * RATIO + torch.arange(RATIO, device=top.device)).reshape(top.shape[0], -1)


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    dev = "cuda"
    if kind in ("decode", "prefill"):
        d, T = case["depth"], case["T"]
        s["kc"][d:], s["vc"][d:] = _pack(s["k"]), _pack(s["v"])
        out = _attend_layer64(s["q"], s["kc"], s["vc"], d)
        if kind == "prefill":
            out = out * torch.sigmoid(s["gate"].double())
        return dict(out=out, kc=s["kc"], vc=s["vc"])
    if kind == "batch":
        outs = [_attend_layer64(s["q"][b:b + 1], s["kc"][b, :d], s["vc"][b, :d], d)
                for b, d in enumerate(s["depths"])]
        return dict(out=torch.cat(outs))
    if kind == "qsa_step":
        T, d, nh = case["T"], case["depth"], case["heads"]
        nb = _qsa_ctx(case) // RATIO
        pos = torch.arange(d, d + T, device=dev)
        s["ic"][d:d + T] = s["k_raw"].to(torch.float16)
        bias = torch.empty((T, nb), dtype=torch.float32, device=dev)
        blk = torch.arange(nb, device=dev)
        for t in range(T):
            bias[t] = torch.where(blk < (d + t + 1) // RATIO, 0.0, torch.where(blk == (d + t) // RATIO, 1e9, -math.inf))
        # a block's pooled key as the last of the step's positions in it leaves it
        own = torch.unique(pos // RATIO)
        s["pool"][own] = _pool64(s["ic"], own, s["knw_idx"])
        cells = _cells(_top64(s["pool"], s["q_idx"], bias))
        cur = s["cur"].to(s["wk"].dtype).double()
        k, v = cur @ s["wk"].double().t(), cur @ s["wv"].double().t()
        for h in range(NKV):
            c = slice(h * HD, (h + 1) * HD)
            k[:, c] = _rope64(_norm64(k[:, c], s["knw"]), pos)
        s["kc"][d:d + T], s["vc"][d:d + T] = _pack(k.float()), _pack(v.float())
        kd, vd, g = _unpack(s["kc"]), _unpack(s["vc"]), nh // NKV
        out = torch.empty(s["q"].shape, dtype=torch.float64, device=dev)
        for t in range(T):
            c = cells[t][cells[t] <= d + t]
            for h in range(NKV):
                hs = slice(h * g, (h + 1) * g)
                out[0, t, hs] = _attend64(s["q"][0, t, hs].contiguous(), kd[c, h], vd[c, h])
        out = out * torch.sigmoid(s["gate"].double())
        return dict(out=out, cells=cells.to(torch.int32), bias=bias, pool=s["pool"], ic=s["ic"], kc=s["kc"], vc=s["vc"])
    if kind == "qsa_chunk":
        T, d, n_kv = s["T"], case["depth"], s["n_kv"]
        nb = n_kv // RATIO
        blk = torch.arange(nb, device=dev)
        p = d + torch.arange(T, device=dev)[:, None]
        bias = torch.where(blk < (p + 1) // RATIO, 0.0, torch.where(blk * RATIO <= p, 1e9, -1e9)).float()
        pool = _pool64(s["ic"], blk, s["knw_idx"])
        cells = _cells(_top64(pool, s["q_idx"], bias))
        lists, counts = torch.zeros_like(cells), torch.zeros((T,), dtype=torch.int32, device=dev)
        for t in range(T):
            c = cells[t][cells[t] <= d + t].sort().values
            lists[t, :c.numel()], counts[t] = c, c.numel()
        return dict(cells=cells.to(torch.int32), lists=lists.to(torch.int32), counts=counts, bias=bias, pool=pool,
                    blk_cells=torch.arange(n_kv, dtype=torch.int32, device=dev),
                    blk_pos=(blk * RATIO).to(torch.int32).repeat(4))
    if kind == "qsa_attend":
        nh = case["heads"]
        kd, vd, g = _unpack(s["kc"]), _unpack(s["vc"]), nh // NKV
        out = torch.empty(s["q"].shape, dtype=torch.float64, device=dev)
        counts = s["counts"].tolist()
        for t in range(case["T"]):
            c = s["lists"][t, :counts[t]].long()
            for h in range(NKV):
                hs = slice(h * g, (h + 1) * g)
                out[0, t, hs] = _attend64(s["q"][0, t, hs].contiguous(), kd[c, h], vd[c, h])
        return dict(out=out * torch.sigmoid(s["gate"].double()))
    T = case["T"]
    n, rep = DN_K * DN_D, DN_V // DN_K
    conv = s["conv"].double()
    q = conv[:, :n].reshape(T, DN_K, DN_D).repeat_interleave(rep, dim=1)
    k = conv[:, n:2 * n].reshape(T, DN_K, DN_D).repeat_interleave(rep, dim=1)
    v = conv[:, 2 * n:].reshape(T, DN_V, DN_D)
    st, e, beta = s["state"].double(), torch.exp(s["g"].double()), s["beta"].double()
    out, snaps = torch.empty((T, DN_V, DN_D), dtype=torch.float64, device=dev), []
    for t in range(T):
        st = st * e[t][:, None, None]
        dv = (v[t] - (st * k[t][:, :, None]).sum(dim=1)) * beta[t][:, None]
        st = st + k[t][:, :, None] * dv[:, None, :]
        out[t] = (st * q[t][:, :, None]).sum(dim=1) / math.sqrt(DN_D)
        snaps.append(st)
    snap = torch.stack([snaps[T - 1 - i] for i in range(1, case["snaps"] + 1)]) if case["snaps"] else None
    return dict(out=out, state=st, snap=snap)
