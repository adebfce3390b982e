"""The work that a user of this framework has it do, as cases that can be timed and compared.

Every case is one pass through the public entry points (the C ABI of include/dspark.h, through the binding's library
handle, or the binding's Engine), over the range of sizes that speculative decoding gives them:

  attn      verify attention of a model's attention layers over fp16 K/V pages (1 to 64 tokens, hundreds to 128k keys)
  rec       the same over the int8 K/V records (16/4/128 heads, up to 16 tokens)
  mlp       the gated FFN of a model's layers on int8 weights: row scales, per-128-column scales, or those with int8 x
  head      a vocabulary projection and its greedy tokens: the int8 LM head with the penalised argmax, or the fp16 crop head
  kv        K/V rows of prompt positions appended to the page (or record) pools of a model's attention layers
  project   the drafter's context seeded at prefill: taps captured and projected into the drafter's rings
  round     one whole speculative round (context, drafter, drafts, verify, accept, commit) through a launch

Sizes are those of the 16-layer configuration (hidden 2048, FFN 8192, 32/8/64 heads, vocabulary 65536) and of the
reference geometry (hidden 2048, FFN 7680, 16/4/128 heads, vocabulary 128000), and others around them.
"""
import importlib.util
import math
import os
import sys
import zlib

import torch

PAGE = 32
DEV = "cuda"


def _host():
    """The binding (its folder's name is not a Python identifier)."""
    name = "dspark_amd_host"
    if name not in sys.modules:
        path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lfm3-1.7b-mi50_amd", "dspark.py")
        spec = importlib.util.spec_from_file_location(name, path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest calls: a few verified tokens early in a conversation, the wide-head geometry, ragged length
        {"name": "attn_short", "kind": "attn", "q_heads": 16, "kv_heads": 4, "head_dim": 128, "ctx": 1001, "tokens": 8,
         "layers": 6, "window": 0, "gate": True},
        # a 16-token block at 32k keys: every attention layer of the 16-layer configuration
        {"name": "attn_32k", "kind": "attn", "q_heads": 32, "kv_heads": 8, "head_dim": 64, "ctx": 32768, "tokens": 16,
         "layers": 6, "window": 0, "gate": True},
        # the widest block of the configurations at the longest context (two of its layers)
        {"name": "attn_128k_wide", "kind": "attn", "q_heads": 32, "kv_heads": 8, "head_dim": 64, "ctx": 131072,
         "tokens": 33, "layers": 2, "window": 0, "gate": False},
        # the reference geometry's own cache format, at its usual draft length, mid-context: six full layers
        {"name": "rec_32k", "kind": "rec", "ctx": 32771, "tokens": 8, "layers": 6, "window": 0, "gate": True},
        # a verify block through the FFNs of four layers, one scale per row
        {"name": "mlp_16", "kind": "mlp", "format": "row", "tokens": 16, "hidden": 2048, "ffn": 8192, "layers": 4},
        # the most tokens a State holds
        {"name": "mlp_64", "kind": "mlp", "format": "row", "tokens": 64, "hidden": 2048, "ffn": 8192, "layers": 4},
        # the reference's shipped weight and activation formats at its verify width
        {"name": "mlp_x8", "kind": "mlp", "format": "x8", "tokens": 8, "hidden": 2048, "ffn": 7680, "layers": 4},
        # the LM head of the verify pass with its greedy tokens
        {"name": "lm_head", "kind": "head", "head": "lm", "tokens": 16, "hidden": 2048, "vocab": 65536},
        # prefill: a chunk of a prompt into the K/V pages of six layers, not page-aligned
        {"name": "kv_prefill", "kind": "kv", "format": "f16", "kv_heads": 8, "head_dim": 64, "pos0": 1003,
         "positions": 8192, "layers": 6},
        # the whole drafter window seeded once per request
        {"name": "project_2k", "kind": "project", "model": "c4", "positions": 2048, "first": 1001},
        # whole rounds: the 16-layer configuration in a 32k conversation, the reference geometry in a short one
        {"name": "round_c4_32k", "kind": "round", "model": "c4", "ctx": 32768, "block": 16, "drafts": 15},
        {"name": "round_ref_1k", "kind": "round", "model": "ref", "ctx": 1003, "block": 9, "drafts": 7},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "rec", "mlp", "head", "kv", "project", "round"])
    if kind == "attn":
        q_heads, kv_heads, dim = rng.choice([(32, 8, 64), (16, 4, 128)])
        return {"kind": kind, "q_heads": q_heads, "kv_heads": kv_heads, "head_dim": dim, "ctx": _log(rng, 200, 131072),
                "tokens": rng.choice([1, 4, 8, 9, 16, 33, rng.randint(1, 64)]), "layers": rng.randint(1, 3),
                "window": rng.choice([0, 0, 256]), "gate": rng.random() < 0.5}
    if kind == "rec":
        return {"kind": kind, "ctx": _log(rng, 200, 131072), "tokens": rng.choice([1, 4, 8, 9, rng.randint(1, 16)]),
                "layers": rng.randint(1, 6), "window": rng.choice([0, 0, 256]), "gate": rng.random() < 0.5}
    if kind == "mlp":
        fmt = rng.choice(["row", "row", "g128", "x8"])
        return {"kind": kind, "format": fmt, "tokens": rng.randint(1, 64 if fmt == "row" else 16),
                "hidden": rng.choice([2048, 256 * rng.randint(2, 10)]),
                "ffn": rng.choice([8192, 7680, 128 * rng.randint(4, 64)]), "layers": 4}
    if kind == "head":
        return {"kind": kind, "head": rng.choice(["lm", "crop"]), "tokens": rng.randint(1, 64), "hidden": 2048,
                "vocab": 16 * _log(rng, 1024, 8000)}
    if kind == "kv":
        fmt, (kv_heads, dim) = rng.choice(["f16", "rec"]), rng.choice([(8, 64), (4, 128)])
        return {"kind": kind, "format": fmt, "kv_heads": 4 if fmt == "rec" else kv_heads,
                "head_dim": 128 if fmt == "rec" else dim, "pos0": rng.randint(0, 40000),
                "positions": _log(rng, 1, 8192), "layers": rng.randint(1, 6)}
    if kind == "project":
        n = _log(rng, 16, 2047)
        return {"kind": kind, "model": rng.choice(["c4", "ref"]), "positions": n, "first": rng.randint(0, 2000)}
    model = rng.choice(["c4", "ref"])
    block = 9 if model == "ref" else rng.choice([9, 16, rng.randint(4, 16)])
    return {"kind": kind, "model": model, "ctx": _log(rng, 300, 32768), "block": block,
            "drafts": rng.choice([3, min(7, block - 1)])}


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) << 32) ^ zlib.crc32(name.encode()))
    return g


def _randn(seed, name, shape, std=1.0, dtype=torch.float16):
    return torch.randn(shape, generator=_gen(seed, name), device=DEV).mul_(std).to(dtype)


def _rand(seed, name, shape, lo, hi, dtype=torch.float16):
    return torch.rand(shape, generator=_gen(seed, name), device=DEV).mul_(hi - lo).add_(lo).to(dtype)


def _u8(seed, name, shape):
    """Biased int8 weights, uniform in [-127, 127]."""
    return torch.randint(1, 256, shape, generator=_gen(seed, name), device=DEV, dtype=torch.uint8)


def _wscale(seed, name, shape, k):
    """Weight scales under which a row of K int8 weights keeps the size of its input."""
    return _rand(seed, name, shape, 0.75 / (73.3 * math.sqrt(k)), 1.25 / (73.3 * math.sqrt(k)))


def _table(seed, name, n_pages):
    """A block table as a long-running cache has it: the logical pages anywhere in the pool."""
    return torch.randperm(n_pages, generator=_gen(seed, name), device=DEV).to(torch.int32)


def _records(k, v):
    """int8 records [n][KVH][264] of fp32 rows [n][KVH][128] (symmetric, one scale per row of K and of V)."""
    n, h, _ = k.shape
    rec = torch.empty((n, h, 264), dtype=torch.int8, device=DEV)
    for x, at in ((k, 0), (v, 132)):
        s = (x.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-6)
        rec[:, :, at:at + 128] = (x / s).round().clamp(-128, 127).to(torch.int8)
        rec[:, :, at + 128:at + 132] = s.float().view(torch.int8)
    return rec.view(torch.uint8)


def _record_values(rec):
    """K and V in fp64 of records [...][264]."""
    def part(at):
        s = rec[..., at + 128:at + 132].contiguous().view(torch.float32).double()
        return rec[..., at:at + 128].contiguous().view(torch.int8).double() * s
    return part(0), part(132)


def _pages(ctx, tokens):
    return (ctx + tokens + PAGE - 1) // PAGE


# ------------------------------------------------------------------------------------------------ engines
class _Mem:
    """Memory of an engine, which a tensor over it keeps alive."""

    def __init__(self, eng, ptr, shape, typestr):
        self.eng = eng
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "version": 2,
                                         "strides": None}


_TYPES = {"u8": "|u1", "f16": "<f2", "f32": "<f4", "i32": "<i4"}


def _view(eng, name, dtype, shape=None):
    """An engine tensor as a torch tensor over the engine's own memory."""
    ptr, nbytes = eng.tensor(name)
    size = {"u8": 1, "f16": 2, "f32": 4, "i32": 4}[dtype]
    t = torch.as_tensor(_Mem(eng, ptr, (nbytes // size,), _TYPES[dtype]), device=DEV)
    return t if shape is None else t[:math.prod(shape)].view(shape)


def _desc(case):
    h = _host()
    if case["model"] == "c4":
        return h.c4_desc(block=case.get("block", 16))
    if case["kind"] == "project":  # fp16 rings, so that the projected rows can be compared as numbers
        return h.ref_desc(kv_format=0)
    return h.ref_desc(block=case["block"], max_drafts=case["block"] - 2)


def _mix_rows(d, i):
    rows = d.q_heads * d.head_dim + 2 * d.kv_heads * d.head_dim + d.q_heads
    return 3 * d.hidden if d.layer_kind[i] == 0 else (rows + 15) // 16 * 16


def _gemm_shapes(d):
    """Every int8 weight of a model: name -> (rows, columns)."""
    H, out = d.hidden, {}
    for i in range(d.n_layers):
        out[f"L{i}.mix"] = (_mix_rows(d, i), H)
        out[f"L{i}.out"] = (H, H)
        out[f"L{i}.w13"], out[f"L{i}.w2"] = (2 * d.ffn, H), (H, d.ffn)
    rows = d.q_heads * d.head_dim + 2 * d.kv_heads * d.head_dim
    for j in range(d.draft_layers):
        out[f"D{j}.mix"] = ((rows + 15) // 16 * 16, H)
        out[f"D{j}.out"] = (H, H)
        out[f"D{j}.w13"], out[f"D{j}.w2"] = (2 * d.draft_ffn, H), (H, d.draft_ffn)
    out["head"] = (d.vocab, H)
    out["crop"] = ((d.crop_rows + 1 + 15) // 16 * 16, H)
    out["fc"] = (H, d.n_taps * H)
    out["ckv"] = (d.draft_layers * 2 * d.kv_heads * d.head_dim, H)
    return out


def _weight(d, seed, name):
    rows, cols = _gemm_shapes(d)[name]
    shape = (cols // 128, rows) if d.weight_format else (rows,)
    return _u8(seed, name + ".w", (rows, cols)), _wscale(seed, name + ".s", shape, cols)


def _vector(d, seed, name):
    """Norm weights (around 1) and conv taps."""
    H, D = d.hidden, d.head_dim
    if name.endswith("conv.w"):
        return _randn(seed, name, (H, d.conv_kernel), 1 / math.sqrt(d.conv_kernel))
    shape = (d.n_taps, H) if name == "tap_norms" else (D,) if name.endswith(("q_norm", "k_norm")) else (H,)
    return _rand(seed, name, shape, 0.8, 1.2)


def _embed(d, seed):
    return _randn(seed, "embed", (d.vocab, d.hidden))


def _fill(eng, d, seed, caches):
    """A loaded model: every weight, and with `caches` the K/V, ring and conv history of an earlier conversation."""
    for name in _gemm_shapes(d):
        w, s = _weight(d, seed, name)
        _view(eng, name + ".w", "u8", w.shape).copy_(w)
        _view(eng, name + ".s", "f16", s.shape).copy_(s)
    _view(eng, "embed", "f16", (d.vocab, d.hidden)).copy_(_embed(d, seed))
    for name in eng.names():
        if name.endswith(("norm", "norms", "conv.w")):
            x = _vector(d, seed, name)
            _view(eng, name, "f16", x.shape).copy_(x)
    _view(eng, "crop_ids", "i32").copy_(torch.randperm(d.vocab, generator=_gen(seed, "crop_ids"), device=DEV)[:d.crop_rows])
    for name in ("markov.w2q", "markov.w1q"):
        v = _view(eng, name, "u8")
        v.copy_(_u8(seed, name, v.shape) ^ 0x80)
    for name, lo, hi in (("markov.w2s", 0.5, 1.5), ("markov.w1s", 1, 1)):
        v = _view(eng, name, "f32")
        v.copy_(_rand(seed, name, v.shape, lo / (73.3 * (16 if lo < 1 else 1)), hi / (73.3 * (16 if lo < 1 else 1)),
                      torch.float32))
    v = _view(eng, "conf_c2", "f32")
    v.copy_(_rand(seed, "conf_c2", v.shape, -0.1, 0.1, torch.float32))
    if caches:
        for name in eng.names():
            if name.startswith(("kv.", "ring.D", "conv.L")):
                rec = name.endswith(".rec")
                v = _view(eng, name, "u8" if rec else "f16")
                v.copy_(_cache(seed, name, v.numel(), rec))


def _cache(seed, name, n, rec):
    if not rec:
        return _randn(seed, name, (n,))
    rows = n // 264
    return _records(_randn(seed, name + "k", (rows, 1, 128), dtype=torch.float32),
                    _randn(seed, name + "v", (rows, 1, 128), dtype=torch.float32)).view(-1)


# ------------------------------------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    return {"attn": _prep_attn, "rec": _prep_attn, "mlp": _prep_mlp, "head": _prep_head, "kv": _prep_kv,
            "project": _prep_project, "round": _prep_round}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _heads(case):
    return (16, 4, 128) if case["kind"] == "rec" else (case["q_heads"], case["kv_heads"], case["head_dim"])


def _attn_inputs(case, seed, layer):
    """q, the layer's pools, gate and block table."""
    QH, KVH, D = _heads(case)
    M, n = case["tokens"], _pages(case["ctx"], case["tokens"])
    q = _randn(seed, f"q{layer}", (M, QH, D))
    gate = _randn(seed, f"gate{layer}", (M, QH), dtype=torch.float32) if case["gate"] else None
    if case["kind"] == "rec":
        rows = [_randn(seed, f"{x}{layer}", (n * PAGE, KVH, D), dtype=torch.float32) for x in "kv"]
        pools = [_records(*rows).view(n, PAGE, KVH, 264)]
    else:
        pools = [_randn(seed, f"k{layer}", (n, KVH, PAGE, D)), _randn(seed, f"v{layer}", (n, KVH, D, PAGE))]
    return q, pools, gate, _table(seed, "table", n)


def _prep_attn(case, seed):
    h, calls, keep, outs = _host(), [], [], []
    rec = case["kind"] == "rec"
    ws = h.Workspace(DEV)
    a, w = case["ctx"], case["window"]
    start = max(0, a - w + 1) if w else 0
    for i in range(case["layers"]):
        q, pools, gate, table = _attn_inputs(case, seed, i)
        out = torch.empty_like(q)
        make = h.rec_attn_args if rec else h.attn_args
        args = make(q, *pools, a, start=start, window=w, out=out, gate=gate, block_table=table)
        calls.append(args)
        keep.append((q, pools, gate, table))
        outs.append(out)
    lib = h.lib()
    size = lib.dspark_verify_attention_rec_workspace if rec else lib.dspark_verify_attention_workspace
    buf = ws.get(size(calls[0]))
    for args in calls:
        args.workspace, args.workspace_bytes = buf.data_ptr(), buf.numel()
    return {"run": _run_attn, "host": h, "fn": lib.dspark_verify_attention_rec if rec else lib.dspark_verify_attention,
            "calls": calls, "outs": outs, "keep": (keep, buf)}


def _run_attn(s):
    stream, fn, check = s["host"].stream_handle(), s["fn"], s["host"].check
    for args in s["calls"]:
        check(fn(args, stream), "verify attention")
    return s["outs"]


def _mlp_inputs(case, seed, layer):
    H, F = case["hidden"], case["ffn"]
    group = case["format"] != "row"
    up, down = _u8(seed, f"up{layer}", (2 * F, H)), _u8(seed, f"down{layer}", (H, F))
    up_s = _wscale(seed, f"up_s{layer}", (H // 128, 2 * F) if group else (2 * F,), H)
    down_s = _wscale(seed, f"down_s{layer}", (F // 128, H) if group else (H,), F)
    return _randn(seed, f"x{layer}", (case["tokens"], H)), up, up_s, down, down_s


def _prep_mlp(case, seed):
    h = _host()
    layers = [_mlp_inputs(case, seed, i) for i in range(case["layers"])]
    mid = [torch.empty((case["tokens"], case["ffn"]), dtype=torch.float16, device=DEV) for _ in layers]
    out = [torch.empty((case["tokens"], case["hidden"]), dtype=torch.float32, device=DEV) for _ in layers]
    need = 256
    for n, k in ((2 * case["ffn"], case["hidden"]), (case["hidden"], case["ffn"])):
        need = max(need, h.lib().dspark_gemm_i8_workspace(case["tokens"], n, k))
    ws = h.Workspace(DEV)
    ws.get(need)
    return {"run": _run_mlp, "host": h, "format": case["format"], "layers": layers, "mid": mid, "out": out, "ws": ws}


def _run_mlp(s):
    h, ws = s["host"], s["ws"]
    for (x, up, up_s, down, down_s), mid, out in zip(s["layers"], s["mid"], s["out"]):
        if s["format"] == "row":
            h.gemm_i8(x, up, up_s, epilogue=1, y_f16=mid, workspace=ws)
            h.gemm_i8(mid, down, down_s, y_f32=out, workspace=ws)
        else:
            f = h.gemm_i8_g128 if s["format"] == "g128" else h.gemm_i8_g128_x8
            f(x, up, up_s, epilogue=1, y_f16=mid)
            f(mid, down, down_s, y_f32=out)
    return {"mid": s["mid"], "out": s["out"]}


REP = 1.05


def _head_inputs(case, seed):
    M, H, V = case["tokens"], case["hidden"], case["vocab"]
    x = _randn(seed, "x", (M, H))
    if case["head"] == "crop":
        return x, _randn(seed, "w", (V, H), 1 / math.sqrt(H)), None, None
    seen = (torch.rand(((V + 31) // 32, 32), generator=_gen(seed, "seen"), device=DEV) < 0.01).long()
    seen = (seen << torch.arange(32, device=DEV)).sum(-1)
    seen = torch.where(seen >= 1 << 31, seen - (1 << 32), seen).to(torch.int32)
    return x, _u8(seed, "w", (V, H)), _wscale(seed, "s", (V,), H), seen


def _prep_head(case, seed):
    h = _host()
    M, V = case["tokens"], case["vocab"]
    x, w, s, seen = _head_inputs(case, seed)
    tokens = torch.randint(0, V, (64,), generator=_gen(seed, "tokens"), device=DEV).tolist()
    st = h.state_tensor(a=1000, anchor=tokens[0], tokens=tokens, run=1, rounds_left=32, budget=512, eos=-1)
    ws, ws_keys = h.Workspace(DEV), h.Workspace(DEV)
    ws.get(max(h.lib().dspark_gemm_i8_workspace(M, V, case["hidden"]), h.lib().dspark_head_argmax_workspace(M, V)))
    ws_keys.get(h.lib().dspark_verify_argmax_workspace(M, V))
    return {"run": _run_head, "host": h, "head": case["head"], "x": x, "w": w, "s": s, "seen": seen, "st": st, "ws": ws,
            "ws_keys": ws_keys, "logits": torch.empty((M, V), dtype=torch.float32, device=DEV),
            "best": torch.empty(M, dtype=torch.int64, device=DEV)}


def _run_head(s):
    h = s["host"]
    if s["head"] == "crop":
        h.head_argmax(s["x"], s["w"], y_f32=s["logits"], best=s["best"], workspace=s["ws"])
    else:
        h.gemm_i8(s["x"], s["w"], s["s"], y_f32=s["logits"], workspace=s["ws"])
        h.verify_argmax(s["logits"], s["seen"], s["st"], rep=REP, inv_rep=1 / REP, best=s["best"], workspace=s["ws_keys"])
    # a key is (value, token): its low word is the token, the value is among the logits
    return {"logits": s["logits"], "tokens": s["best"].view(torch.int32)[::2]}


def _kv_inputs(case, seed, layer):
    """K and V of a prompt chunk, as they lie in the rows of a q | k | v projection."""
    KVH, D, n = case["kv_heads"], case["head_dim"], case["positions"]
    dtype = torch.float32 if case["format"] == "rec" else torch.float16
    rows = _randn(seed, f"rows{layer}", (n, 6 * KVH * D), dtype=dtype)
    return rows[:, 4 * KVH * D:5 * KVH * D], rows[:, 5 * KVH * D:]


def _prep_kv(case, seed):
    h, KVH, D = _host(), case["kv_heads"], case["head_dim"]
    n = _pages(case["pos0"], case["positions"])
    rec = case["format"] == "rec"
    pools = [(h.rec_pages_alloc(n, KVH),) if rec else h.kv_pages_alloc(n, KVH, D) for _ in range(case["layers"])]
    return {"run": _run_kv, "host": h, "write": h.kv_write_rec if rec else h.kv_write, "pos0": case["pos0"],
            "rows": [_kv_inputs(case, seed, i) for i in range(case["layers"])], "pools": pools,
            "table": _table(seed, "table", n)}


def _run_kv(s):
    for (k, v), pools in zip(s["rows"], s["pools"]):
        s["write"](k, v, *pools, s["pos0"], block_table=s["table"])
    return s["pools"]


def _taps(case, seed, d):
    return [_randn(seed, f"tap{b}", (case["positions"], d.hidden)) for b in range(d.n_taps)]


def _prep_project(case, seed):
    h, d = _host(), _desc(case)
    eng = h.Engine(d, 4096)
    _fill(eng, d, seed, False)
    eng.prepare()
    rings = [(_view(eng, f"ring.D{j}.k", "f16"), _view(eng, f"ring.D{j}.v", "f16")) for j in range(d.draft_layers)]
    return {"run": _run_project, "eng": eng, "taps": _taps(case, seed, d), "rings": rings, "first": case["first"],
            "end": case["first"] + case["positions"]}


def _run_project(s):
    for slot, rows in enumerate(s["taps"]):
        s["eng"].capture_tap(slot, rows, s["first"], s["first"])
    s["eng"].project_prompt(s["first"], s["end"])
    return s["rings"]


def _round_tokens(case, seed, d):
    """The anchor, then the tokens that the round verifies."""
    return torch.randint(0, d.vocab, (1 + case["drafts"],), generator=_gen(seed, "tokens"), device=DEV).tolist()


def _prep_round(case, seed):
    h, d, a = _host(), _desc(case), case["ctx"]
    eng = h.Engine(d, a + 256)
    _fill(eng, d, seed, True)
    eng.prepare()
    tokens = _round_tokens(case, seed, d)
    _view(eng, "plant", "i32")[a + 1:a + len(tokens)] = torch.tensor(tokens[1:], dtype=torch.int32, device=DEV)
    eng.init_seen(tokens)
    return {"run": _run_round, "eng": eng, "a": a, "anchor": tokens[0], "drafts": case["drafts"],
            "lo": max(0, a - d.draft_window), "base": _view(eng, "base", "f32"),
            "logits": _view(eng, "logits", "f32", (1 + case["drafts"], d.vocab))}


def _run_round(s):
    # One round per launch, the first after a prefill (nothing new to project), its drafts from the plant: the whole
    # round runs, and which tokens it verifies doesn't hang on near ties of a random model, so its logits can be compared.
    s["eng"].launch(s["a"], s["anchor"], rounds=1, ctx_new=0, ctx_pos=s["a"], ctx_lo=s["lo"], force_m=-1,
                    max_drafts=s["drafts"])
    return {"base": s["base"], "logits": s["logits"]}


# ------------------------------------------------------------------------------------------------ work and tolerance
def _gemm_work(m, rows, cols, group=False):
    return rows * cols + 2 * rows * (cols // 128 if group else 1), 2 * m * rows * cols


def work(case):
    kind, m, layers = case["kind"], case.get("tokens", 0), case.get("layers", 1)
    nbytes = flops = 0
    if kind in ("attn", "rec"):
        QH, KVH, D = _heads(case)
        keys = m + (min(case["window"] + m, case["ctx"]) if case["window"] else case["ctx"])
        nbytes = keys * KVH * (264 if kind == "rec" else 4 * D) + 4 * m * QH * D + (4 * m * QH if case["gate"] else 0)
        flops = 4 * m * QH * D * keys
    elif kind == "mlp":
        H, F, group = case["hidden"], case["ffn"], case["format"] != "row"
        for rows, cols in ((2 * F, H), (H, F)):
            b, f = _gemm_work(m, rows, cols, group)
            nbytes, flops = nbytes + b, flops + f
        nbytes += m * (2 * H + 4 * F + 4 * H)
    elif kind == "head":
        H, V = case["hidden"], case["vocab"]
        nbytes = V * H * (2 if case["head"] == "crop" else 1) + 2 * m * H + 4 * m * V + (2 * V if case["head"] == "lm" else 0)
        flops = 2 * m * V * H
    elif kind == "kv":
        n = case["positions"] * case["kv_heads"]
        nbytes = n * (1024 + 264) if case["format"] == "rec" else n * case["head_dim"] * 8
    elif kind == "project":
        d, n = _desc(case), case["positions"]
        H = d.hidden
        rows = d.draft_layers * 2 * d.kv_heads * d.head_dim
        for r, c in ((H, d.n_taps * H), (rows, H)):
            b, f = _gemm_work(n, r, c, d.weight_format)
            nbytes, flops = nbytes + b, flops + f
        nbytes += n * d.n_taps * H * 2 + n * rows * 2
    else:
        d, a, mv = _desc(case), case["ctx"], 1 + case["drafts"]
        for name, (r, c) in _gemm_shapes(d).items():
            b, f = _gemm_work(mv if name.startswith("L") or name == "head" else d.block, r, c, d.weight_format)
            nbytes, flops = nbytes + b, flops + f
        row = d.kv_heads * (264 if d.kv_format else 4 * d.head_dim)
        for k in d.layer_kind[:d.n_layers]:
            nbytes += ((a if k == 1 else min(a, d.window)) + mv) * row if k else 0
        nbytes += d.draft_layers * (min(a, d.draft_window) + d.block) * row
        nbytes += 4 * (mv * d.vocab + d.block * d.crop_rows)
    return {"bytes": nbytes * layers, "flops": flops * layers}


def tolerance(case):
    # About four times what these paths show against fp64 (whole rounds: the rounding of every layer travels on).
    kind = case["kind"]
    if kind == "kv":
        return "exact"
    if kind in ("attn", "rec", "project"):
        return {"rel": 2e-3, "max": 2e-2}
    if kind == "mlp":
        return {"rel": 6e-3, "max": 0.1} if case["format"] == "x8" else {"rel": 1e-3, "max": 1e-2}
    if kind == "head":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.01}
    return {"rel": 9e-3, "max": 0.1} if case["model"] == "c4" else {"rel": 2.8e-2, "max": 0.3}


# ------------------------------------------------------------------------------------------------ fp64
def exact(case, seed):
    with torch.no_grad():
        return {"attn": _exact_attn, "rec": _exact_attn, "mlp": _exact_mlp, "head": _exact_head, "kv": _exact_kv,
                "project": _exact_project, "round": _exact_round}[case["kind"]](case, seed)


def _k_index(D):
    """Where K[key][d] lies in a (page, KV head) block: the operand order of include/dspark.h, as [PAGE * D]."""
    key, d = torch.arange(PAGE, device=DEV)[:, None], torch.arange(D, device=DEV)[None, :]
    n = 4 * (key // 8) + key % 4
    return ((((key // 4) % 2 * (D // 32) + d // 32) * 64 + n + 16 * ((d % 32) // 8)) * 8 + d % 8).reshape(-1)


def _logical(kp, vp, table, D):
    """K and V by position, [positions][KVH][D] in fp64, of page pools."""
    kp, vp = kp[table.long()].double(), vp[table.long()].double()
    n, KVH = kp.shape[0], kp.shape[1]
    k = kp.reshape(n, KVH, PAGE * D)[:, :, _k_index(D)].view(n, KVH, PAGE, D)
    return k.transpose(1, 2).reshape(n * PAGE, KVH, D), vp.view(n, KVH, D, PAGE).permute(0, 3, 1, 2).reshape(n * PAGE, KVH, D)


def _quantize_q(q):
    """The record path's q: int8 per 32 dimensions."""
    g = q.float().reshape(*q.shape[:-1], q.shape[-1] // 32, 32)
    s = (g.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-20)
    return ((g * (1 / s)).round() * s).double().view(q.shape)


def _softmax_attention(q, k, v, a, start, window, causal):
    """q [M][QH][D], k and v [positions][KVH][D] with the block's rows at a ..."""
    M, QH, D = q.shape
    KVH = k.shape[1]
    pos, t = torch.arange(a + M, device=DEV)[None, :], torch.arange(M, device=DEV)[:, None]
    seen = (pos < a) & (pos >= start) & ((pos > a + t - window) if window else True)
    seen = seen | ((pos >= a) & ((pos <= a + t) if causal else True))
    out = torch.empty_like(q)
    lo = start if not window else min(start, max(0, a - window))
    for h in range(QH):
        kh, vh = k[lo:a + M, h * KVH // QH], v[lo:a + M, h * KVH // QH]
        s = (q[:, h] @ kh.T / math.sqrt(D)).masked_fill(~seen[:, lo:], -math.inf)
        out[:, h] = torch.softmax(s, -1) @ vh
    return out


def _exact_attn(case, seed):
    outs, (QH, KVH, D) = [], _heads(case)
    a, w = case["ctx"], case["window"]
    for i in range(case["layers"]):
        q, pools, gate, table = _attn_inputs(case, seed, i)
        if case["kind"] == "rec":
            k, v = _record_values(pools[0][table.long()].reshape(-1, KVH, 264))
            q = _quantize_q(q)
        else:
            k, v = _logical(*pools, table, D)
        o = _softmax_attention(q.double(), k, v, a, max(0, a - w + 1) if w else 0, w, True)
        outs.append(o * torch.sigmoid(gate.double())[:, :, None] if case["gate"] else o)
    return outs


def _x8(x):
    """int8 activations: one scale per 16 columns."""
    g = x.float().reshape(x.shape[0], -1, 16)
    s = (g.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-20)
    return ((g * (1 / s)).round().double() * s.double()).view(x.shape)


def _mm(x, w, s, x8=False):
    """x [m][K] times int8 weights [N][K] with row scales [N] or group scales [K / 128][N]."""
    x, out = _x8(x) if x8 else x, []
    for r in range(0, w.shape[0], 16384):
        q = w[r:r + 16384].double() - 128
        if s.dim() == 2:
            q = (q.view(q.shape[0], -1, 128) * s[:, r:r + 16384].double().T[:, :, None]).view(q.shape)
            out.append(x @ q.T)
        else:
            out.append(x @ q.T * s[r:r + 16384].double())
    return torch.cat(out, 1)


def _gated(y):
    return torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]


def _exact_mlp(case, seed):
    mid, out, x8 = [], [], case["format"] == "x8"
    for i in range(case["layers"]):
        x, up, up_s, down, down_s = _mlp_inputs(case, seed, i)
        mid.append(_gated(_mm(x.double(), up, up_s, x8)))
        out.append(_mm(mid[-1].half().double(), down, down_s, x8))
    return {"mid": mid, "out": out}


def _exact_head(case, seed):
    x, w, s, _ = _head_inputs(case, seed)
    if case["head"] == "crop":
        y = torch.cat([x.double() @ w[r:r + 16384].double().T for r in range(0, w.shape[0], 16384)], 1)
    else:
        y = _mm(x.double(), w, s)
    return {"logits": y, "tokens": None}


def _scatter_pages(k, v, pos, n_pages, table):
    """Page pools in fp64 with rows k, v [n][KVH][D] at positions pos, zeros elsewhere."""
    n, KVH, D = k.shape
    kp = torch.zeros((n_pages, KVH, PAGE * D), dtype=torch.float64, device=DEV)
    vp = torch.zeros((n_pages, KVH, D, PAGE), dtype=torch.float64, device=DEV)
    page, slot = table.long()[pos // PAGE], pos % PAGE
    at = _k_index(D).view(PAGE, D)[slot]
    h = torch.arange(KVH, device=DEV)
    kp[page[:, None, None], h[None, :, None], at[:, None, :]] = k
    vp[page[:, None, None], h[None, :, None], torch.arange(D, device=DEV)[None, None, :], slot[:, None, None]] = v
    return kp.view(n_pages, KVH, PAGE, D), vp


def _exact_kv(case, seed):
    if case["format"] == "rec":  # whole numbers
        return None
    n, KVH, D = case["positions"], case["kv_heads"], case["head_dim"]
    n_pages, pos = _pages(case["pos0"], n), case["pos0"] + torch.arange(n, device=DEV)
    out = []
    for i in range(case["layers"]):
        k, v = (x.double().reshape(n, KVH, D) for x in _kv_inputs(case, seed, i))
        out.append(_scatter_pages(k, v, pos, n_pages, _table(seed, "table", n_pages)))
    return out


def _norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, base, pairs):
    """x [n][heads][D] rotated in pairs (i, i + D / 2), i < pairs; the angles in fp32, the table in fp16."""
    D = x.shape[-1]
    ex = [float(torch.tensor(2 * i / D, dtype=torch.float32)) for i in range(pairs)]
    inv = torch.tensor([math.pow(base, e) for e in ex], dtype=torch.float32).reciprocal().to(DEV)
    f = (pos.float()[:, None] * inv).double()[:, None, :]
    c, s = f.cos().half().double(), f.sin().half().double()
    y, half = x.clone(), D // 2
    y[..., :pairs] = x[..., :pairs] * c - x[..., half:half + pairs] * s
    y[..., half:half + pairs] = x[..., half:half + pairs] * c + x[..., :pairs] * s
    return y


def _exact_project(case, seed):
    d = _desc(case)
    n, KVH, D = case["positions"], d.kv_heads, d.head_dim
    norms = _vector(d, seed, "tap_norms")
    x = torch.cat([_norm(t.double(), norms[b], d.eps) for b, t in enumerate(_taps(case, seed, d))], 1)
    x = _norm(_mm(x, *_weight(d, seed, "fc")), _vector(d, seed, "hidden_norm"), d.eps)
    kv = _mm(x, *_weight(d, seed, "ckv")).view(n, d.draft_layers, 2, KVH, D)
    pos = case["first"] + torch.arange(n, device=DEV)
    pages = d.ring_positions // PAGE
    table, out = torch.arange(4096 // PAGE + 64, device=DEV) % pages, []
    for j in range(d.draft_layers):
        k = _rope(_norm(kv[:, j, 0], _vector(d, seed, f"D{j}.k_norm"), d.eps), pos, d.rope_base, d.rope_pairs)
        kp, vp = _scatter_pages(k, kv[:, j, 1], pos, pages, table)
        out.append((kp.view(-1), vp.view(-1)))
    return out


def _cached(d, seed, name, table, lo, hi):
    """K and V of cache positions lo .. hi - 1 (their whole pages), by position from lo's page on, and that position."""
    p0, p1 = lo // PAGE, (hi + PAGE - 1) // PAGE
    at, KVH, D = table[p0:p1].long(), d.kv_heads, d.head_dim
    n = d.pages
    if d.kv_format:
        rec = _cache(seed, name + ".rec", n * PAGE * KVH * 264, True).view(n, PAGE, KVH, 264)
        k, v = _record_values(rec[at].reshape(-1, KVH, 264))
    else:
        pools = [_cache(seed, f"{name}.{x}", n * KVH * PAGE * D, False) for x in "kv"]
        k, v = _logical(pools[0].view(n, KVH, PAGE, D), pools[1].view(n, KVH, D, PAGE), at, D)
    return k, v, p0 * PAGE


def _exact_attention(d, seed, pre, mix, a, window, draft, rope):
    """The block's attention in fp64 from its q | k | v (| gate) rows; ungated heads [M][QH * D]."""
    M, QH, KVH, D = mix.shape[0], d.q_heads, d.kv_heads, d.head_dim
    pos = a + torch.arange(M, device=DEV)
    q, k, v = (mix[:, i * D:j * D].reshape(M, j - i, D) for i, j in ((0, QH), (QH, QH + KVH), (QH + KVH, QH + 2 * KVH)))
    q = _rope(_norm(q, _vector(d, seed, pre + "q_norm"), d.eps), pos, *rope).half().double()
    k = _rope(_norm(k, _vector(d, seed, pre + "k_norm"), d.eps), pos, *rope)
    if d.kv_format:
        k, v = _record_values(_records(k.float(), v.float()))
        q = _quantize_q(q)
    else:
        k, v = k.half().double(), v.half().double()
    lo = max(0, a - d.draft_window) if draft else max(0, a - window + 1) if window else 0
    if draft:
        d.pages = d.ring_positions // PAGE
        table = torch.arange((a + 256 + d.block) // PAGE + 2, device=DEV) % d.pages
        ck, cv, at = _cached(d, seed, "ring." + pre[:-1], table, lo, a)
    else:
        d.pages = (a + 256 + d.block + PAGE - 1) // PAGE + 1
        ck, cv, at = _cached(d, seed, "kv." + pre[:-1], torch.arange(d.pages, device=DEV), lo, a)
    k, v = torch.cat([ck[:a - at], k]), torch.cat([cv[:a - at], v])
    return _softmax_attention(q, k, v, a - at, lo - at, 0 if draft else window, not draft).reshape(M, QH * D)


def _exact_conv(d, seed, i, mix, a):
    bx = (mix[:, 0::3] * mix[:, 2::3]).half().double()
    ring, K = _cache(seed, f"conv.L{i}", 128 * d.hidden, False).view(128, d.hidden).double(), d.conv_kernel
    hist = torch.cat([ring[(a - K + 1 + torch.arange(K - 1, device=DEV)) % 128], bx])
    w = _vector(d, seed, f"L{i}.conv.w").double()
    return mix[:, 1::3] * sum(w[:, k] * hist[k:k + bx.shape[0]] for k in range(K))


def _exact_round(case, seed):
    d, a = _desc(case), case["ctx"]
    H, QH, KVH, D = d.hidden, d.q_heads, d.kv_heads, d.head_dim
    tokens, embed = _round_tokens(case, seed, d), _embed(d, seed)
    mm = lambda x, name: _mm(x, *_weight(d, seed, name), bool(d.x_format))  # noqa: E731
    vec = lambda name: _vector(d, seed, name).double()  # noqa: E731
    full, swa = (d.rope_base, d.rope_pairs), (d.rope_base_swa, d.rope_pairs_swa)
    h = embed[[tokens[0]] + [d.mask_token] * (d.block - 1)].double()
    for j in range(d.draft_layers):
        pre = f"D{j}."
        y = _exact_attention(d, seed, pre, mm(_norm(h, vec(pre + "op_norm"), d.eps), pre + "mix"), a, 0, True, full)
        h = h + mm(y, pre + "out")
        h = h + mm(_gated(mm(_norm(h, vec(pre + "ffn_norm"), d.eps), pre + "w13")), pre + "w2")
    base = mm(_norm(h, vec("draft_norm"), d.eps), "crop")
    h = embed[tokens].double()
    for i in range(d.n_layers):
        pre, kind = f"L{i}.", d.layer_kind[i]
        mix = mm(_norm(h, vec(pre + "op_norm"), d.eps), pre + "mix")
        if kind == 0:
            y = _exact_conv(d, seed, i, mix, a)
        else:
            y = _exact_attention(d, seed, pre, mix, a, d.window if kind == 2 else 0, False,
                                 swa if kind == 2 and d.rope_base_swa > 0 else full)
            gate = mix[:, (QH + 2 * KVH) * D:(QH + 2 * KVH) * D + QH]
            y = (y.view(-1, QH, D) * torch.sigmoid(gate)[:, :, None]).view(-1, QH * D)
        h = h + _norm(mm(y, pre + "out"), vec(pre + "post_op_norm"), d.eps)
        v = mm(_gated(mm(_norm(h, vec(pre + "ffn_norm"), d.eps), pre + "w13")), pre + "w2")
        h = h + _norm(v, vec(pre + "post_ffn_norm"), d.eps)
    return {"base": base.reshape(-1), "logits": mm(_norm(h, vec("final_norm"), d.eps), "head")}
