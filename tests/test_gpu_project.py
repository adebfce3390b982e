"""The drafter's prompt projection over many positions in one pass (dspark_engine_project_prompt past one block):
captured taps -> fc -> hidden norm -> ckv -> k norm + RoPE -> ring rows, on the many-token GEMM's two tile sizes with row
and group scales, at position counts around the tiles' edges, against fp64 from the same weights.

Bar: the ring holds fp16 of values whose inputs the GPU and the check round to fp16 at the same points (the captured taps,
the hidden norm's output), so a value differs by its own rounding and by what last-bit flips of those inputs carry
through a dot product: two fp16 steps at the largest magnitude, the bar of the blockwise projection's test. A record holds
a row of K or V in steps of its largest magnitude / 127: half a step more."""
import numpy as np
import pytest

from conftest import load_host, rope_numpy
from test_gpu_engine import REF_REC, REF_SMALL, SMALL, make_weights
from test_gpu_fullsize import ring_rows
from test_gpu_launch import ulp16

pytestmark = pytest.mark.gpu

# 64-token tiles, K in bands (2 taps x 256 columns: 8 chunks), 2 drafter layers
NARROW = dict(SMALL, draft_window=700, ring_positions=1024)
# group scales, head_dim 128
GROUPS = dict(REF_SMALL, draft_window=700, ring_positions=1024, weight_format=1)
# 128-token tiles for fc (16 x 13 tiles at 1537 positions), 64-token ones for ckv, an odd number of chunks per band
WIDE = dict(SMALL, hidden=2048, q_heads=32, kv_heads=8, ffn=256, draft_ffn=256, n_taps=1, tap_layer=[1],
            draft_window=1600, ring_positions=2048)
WIDE_GROUPS = dict(WIDE, weight_format=1, n_taps=3, tap_layer=[0, 1, 2])
CASES = [(NARROW, n, first) for n, first in ((9, 0), (63, 5), (64, 31), (65, 7), (128, 0), (200, 500), (700, 330))]
CASES += [(GROUPS, n, 33) for n in (10, 64, 129, 511)]
CASES += [(WIDE, 1537, 700), (WIDE_GROUPS, 1537, 1), (WIDE_GROUPS, 1600, 0)]
# int8 K/V records: blocks of 9, the two position counts around a block, page edges, 64- and 128-token tiles
RECORDS = dict(REF_REC, draft_window=700, ring_positions=1024)
RECORDS_ROWS = dict(RECORDS, weight_format=0)
# fc in 16, 8 and 4 bands (128 chunks of K; one, two and four token tiles of 64), and in 4 of 15 chunks (16 and a short last
# one with group scales)
BANDS = dict(WIDE, n_taps=4, tap_layer=[0, 1, 2, 3])
BANDS_GROUPS = dict(BANDS, weight_format=1)
UNEVEN = dict(WIDE, hidden=1280, q_heads=20, kv_heads=5, n_taps=3, tap_layer=[0, 1, 2])
UNEVEN_GROUPS = dict(UNEVEN, weight_format=1)
CASES += [(geom, n, 9) for geom in (BANDS, BANDS_GROUPS) for n in (17, 64, 65, 200)]
CASES += [(geom, n, 31) for geom in (UNEVEN, UNEVEN_GROUPS) for n in (10, 40)]
CASES += [(RECORDS, n, first) for n, first in ((9, 3), (10, 0), (31, 1), (33, 31), (64, 32), (600, 77))]
CASES += [(RECORDS_ROWS, 10, 23), (RECORDS_ROWS, 417, 5)]


@pytest.mark.parametrize("geom,n,first", CASES)
def test_many_positions(geom, n, first):
    import torch
    from oracle import round as rnd
    host = load_host()
    desc = host.model_desc(**geom)
    H, KVH, D = desc.hidden, desc.kv_heads, desc.head_dim
    print(f"case hidden={H} n={n} first={first} weight_format={desc.weight_format}", flush=True)
    eng = host.Engine(desc, 2560)
    W = rnd.Weights(desc, make_weights(eng, desc, 7))
    rng = np.random.default_rng(n)
    taps = rng.standard_normal((desc.n_taps, n, H)).astype(np.float16)
    rec = desc.kv_format == 1
    names = ["rec"] if rec else ["k", "v"]
    before = {}
    for name in (f"ring.D{j}.{x}" for j in range(desc.draft_layers) for x in names):  # any bits: no slot starts as zeros
        before[name] = rng.integers(0, 1 << 16, eng.tensor(name)[1] // 2).astype(np.uint16)
        eng.upload(name, before[name])
    for slot in range(desc.n_taps):
        eng.capture_tap(slot, torch.from_numpy(taps[slot]).cuda(), first, first)
    eng.project_prompt(first, first + n)
    torch.cuda.synchronize()

    x = np.concatenate([rnd.tap_rows(W, taps[b].astype(np.float64), b) for b in range(desc.n_taps)], axis=1)
    c = rnd.gemm(x, *W.gemm_w("fc", H, desc.n_taps * H))
    _, x = rnd.resnorm(None, c, None, W.f16("hidden_norm"), 0, desc.eps)
    kv = rnd.gemm(x, *W.gemm_w("ckv", desc.draft_layers * 2 * KVH * D, H)).reshape(n, desc.draft_layers, 2, KVH, D)
    rope = rnd.h2f(rope_numpy(desc.rope_base, desc.rope_pairs, D, first + n))[first:][:, None, :]
    cos, sin, half, p = rope[..., :D // 2], rope[..., D // 2:], D // 2, desc.rope_pairs
    bt = eng.download("ring_table", np.int32)
    for j in range(desc.draft_layers):
        k = kv[:, j, 0]
        k = k / np.sqrt((k * k).mean(-1, keepdims=True) + desc.eps) * W.f16(f"D{j}.k_norm")
        wk = k.copy()
        wk[..., :p] = k[..., :p] * cos[..., :p] - k[..., half:half + p] * sin[..., :p]
        wk[..., half:half + p] = k[..., half:half + p] * cos[..., :p] + k[..., :p] * sin[..., :p]
        gk, gv = ring_rows(eng, desc, j, range(first, first + n))
        kerr, verr = np.abs(gk - wk), np.abs(gv - kv[:, j, 1])
        print(f"layer {j}: K max-abs {np.max(kerr):.2e}, V max-abs {np.max(verr):.2e}", flush=True)
        for err, want in ((kerr, wk), (verr, kv[:, j, 1])):
            bar = 2 * ulp16(np.max(np.abs(want)))
            if rec:  # half a code, of a scale whose own row differs by the bar
                bar = bar + 0.5 * (np.max(np.abs(want), -1, keepdims=True) + bar) / 127
            assert np.all(err <= bar), np.max(err - bar)
        # every slot of the ring outside [first, first + n) holds the bits it held
        at = np.arange(first, first + n)
        pages, slots = bt[at // 32], at % 32
        for x in names:
            now, was = eng.download(f"ring.D{j}.{x}", np.uint16), before[f"ring.D{j}.{x}"]
            if rec:
                now, was = (b.view(np.uint8).reshape(-1, 32, KVH * 264) for b in (now, was))
                now[pages, slots] = was[pages, slots] = 0
            elif x == "k":  # [page][head][keys in operand order][dims]
                index = np.asarray(host.k_page_index(D))
                now, was = (b.reshape(-1, KVH, 32 * D) for b in (now, was))
                for pg, sl in zip(pages, slots):
                    now[pg][:, index[sl]] = was[pg][:, index[sl]] = 0
            else:  # [page][head][dims][keys]
                now, was = (b.reshape(-1, KVH, D, 32) for b in (now, was))
                now[pages, :, :, slots] = was[pages, :, :, slots] = 0
            assert np.array_equal(now, was), x
    eng.close()


def test_long_window_memory():
    """A drafter window beyond what the one-pass projection takes (taps of 2 GiB) holds no projection buffers for the rest
    of it; ranges that it does take are projected as ever."""
    import torch
    host = load_host()
    desc = host.model_desc(**dict(WIDE, n_taps=3, tap_layer=[0, 1, 2], draft_window=400000, ring_positions=400064))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    eng = host.Engine(desc, 401000)
    extra = free - torch.cuda.mem_get_info()[0] - sum(eng.tensor(n)[1] for n in eng.names())
    print(f"case window 400000: {extra / 2**30:.2f} GiB beside the named tensors", flush=True)
    # 174762 rows of 2 bands x 2048 fp32 and 2048 fp16, the weights' tiles, allocation granularity
    assert extra < 174762 * 2048 * 10 + 2**30, extra
    make_weights(eng, desc, 7)
    rows = torch.randn((64, desc.hidden), device="cuda").to(torch.float16)
    for slot in range(desc.n_taps):
        eng.capture_tap(slot, rows, 390000, 390000)
    eng.project_prompt(390000, 390064)
    torch.cuda.synchronize()
    assert np.any(eng.download("ring.D0.k", np.uint16))
    eng.close()
