"""The GEMMs over row-major operands (streamed tiles; few rows with group scales) through the C ABI at the edges of their
tiles, ranges and rings, against fp64.

Bar: every product of an int8 weight (or an fp16 one) and an fp16 x is exact in fp32 and K of them are added in fp32 in
some order, so an output is within (K + groups) 2^-24 of the sum of its terms' magnitudes (the scales' products add one
rounding each); fp16 outputs add half an fp16 step of the value. int8 x (quantized on load): 1e-3 of the largest output,
where a product next to a code midpoint takes the neighbouring code (tests/test_gpu_gemm_x8.py)."""
import numpy as np
import pytest

from conftest import load_host

pytestmark = pytest.mark.gpu


def operands(M, N, K, seed, wide=False):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((M, K)).astype(np.float16)
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16) if wide else rng.integers(1, 256, (N, K), dtype=np.uint8)
    return rng, x, w


def at_offset(torch, a, nbytes):
    """A device copy of `a` that starts `nbytes` past a 256-byte boundary."""
    raw = torch.zeros(a.nbytes + nbytes, dtype=torch.uint8, device="cuda")
    raw[nbytes:] = torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).cuda()
    return raw[nbytes:].view(torch.float16 if a.dtype == np.float16 else torch.uint8).view(a.shape)


def check(got, want, terms, K, half=False):
    bar = (K + K // 128 + 2) * 2.0 ** -24 * terms + (np.abs(want) * 2.0 ** -10 + 2.0 ** -24 if half else 0)
    assert np.all(np.abs(got.astype(np.float64) - want) <= bar), float(np.max(np.abs(got - want) / bar))


SHAPES = [(1, 16, 128), (16, 80, 256), (17, 64, 1152), (32, 4096, 128), (33, 208, 2048), (48, 16464, 1024), (49, 32784, 512),
          (64, 2048, 8192), (64, 144, 4224), (64, 16, 128), (49, 2064, 1152), (8, 16448, 1024), (5, 40000, 256), (64, 40000, 512), (9, 2064, 1088)]


@pytest.mark.parametrize("off", [0, 8])  # off a 16-byte boundary: the general kernels
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8_rows(M, N, K, off):
    import torch
    host = load_host()
    print(f"case int8 M={M} N={N} K={K} off={off}", flush=True)
    rng, x, w = operands(M, N, K, N + K + M)
    s = (rng.uniform(0.5, 1.5, N) / (73.3 * np.sqrt(K))).astype(np.float16)
    xd, wd, sd = at_offset(torch, x, off), at_offset(torch, w, off), torch.from_numpy(s).cuda()
    q = w.astype(np.float64) - 128
    want = x.astype(np.float64) @ q.T * s.astype(np.float64)
    terms = np.abs(x.astype(np.float64)) @ np.abs(q).T * s.astype(np.float64)
    ws = host.Workspace()
    y32, y16 = torch.empty((M, N), device="cuda"), torch.empty((M, N), dtype=torch.float16, device="cuda")
    for _ in range(2):  # the second call finds the counters as the first left them
        host.gemm_i8(xd, wd, sd, y_f32=y32, y_f16=y16, workspace=ws)
        first = y32.clone()
        check(y32.cpu().numpy(), want, terms, K)
        check(y16.cpu().numpy(), want, terms, K, half=True)
    assert torch.equal(first, y32)
    h = host.gemm_i8(xd, wd, sd, epilogue=1, workspace=ws).cpu().numpy()
    g, u = want[:, 0::2], want[:, 1::2]
    ref = g / (1 + np.exp(-g)) * u
    assert np.max(np.abs(h - ref)) <= 2e-3 * max(1.0, np.max(np.abs(ref)))


@pytest.mark.parametrize("off", [0, 8])
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (16, 16464, 512), (17, 80, 192), (33, 4112, 1024), (48, 16, 2048), (64, 32768, 256),
                                   (64, 208, 576)])
def test_head_rows(M, N, K, off):
    import torch
    host = load_host()
    print(f"case head M={M} N={N} K={K} off={off}", flush=True)
    _, x, w = operands(M, N, K, N + K + M, wide=True)
    y = torch.empty((M, N), device="cuda")
    best = host.head_argmax(at_offset(torch, x, off), at_offset(torch, w, off), y_f32=y)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    got = y.cpu().numpy()
    check(got, want, np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T, K)
    assert np.array_equal(host.keys_to_tokens(best).cpu().numpy(), np.argmax(got, 1))


GROUPS = [(1, 16, 128), (8, 48, 256), (9, 2064, 640), (16, 4096, 1920), (7, 2048, 2304), (16, 2048, 7680), (9, 4112, 4096),
          (16, 8256, 1024), (3, 15360, 2048), (16, 16464, 384), (9, 9984, 640), (8, 8192, 1792),
          (8, 20480, 768), (5, 17424, 1024), (3, 2064, 1152), (4, 2064, 1152), (16, 4096, 1152)]


@pytest.mark.parametrize("x8", [False, True])
@pytest.mark.parametrize("M,N,K", GROUPS)
def test_group_scales(M, N, K, x8):
    import torch
    from oracle import oracle as orc
    host = load_host()
    print(f"case groups M={M} N={N} K={K} x8={x8}", flush=True)
    rng, x, w = operands(M, N, K, N + K + M)
    gs = (rng.uniform(0.5, 1.5, (K // 128, N)) / (73.3 * np.sqrt(K))).astype(np.float16)
    scale = np.repeat(gs.astype(np.float64), 128, axis=0).T * (w.astype(np.float64) - 128)
    v = x.astype(np.float64)
    if x8:
        c, s = orc.quantize_x16(x.astype(np.float32))
        v = c.astype(np.float64) * np.repeat(s.astype(np.float64), 16, axis=1)
    want = v @ scale.T
    for off in (0, 8):
        f = host.gemm_i8_g128_x8 if x8 else host.gemm_i8_g128
        a = (at_offset(torch, x, off), at_offset(torch, w, off), torch.from_numpy(gs).cuda())
        y, _ = f(*a)
        if x8:
            assert np.max(np.abs(y.cpu().numpy() - want)) <= 1e-3 * np.max(np.abs(want))
        else:
            check(y.cpu().numpy(), want, np.abs(v) @ np.abs(scale).T, K)
        assert torch.equal(f(*a)[0], y)
        h = torch.empty((M, N // 2), dtype=torch.float16, device="cuda")
        f(*a, epilogue=1, y_f16=h)
        g, u = want[:, 0::2], want[:, 1::2]
        ref = g / (1 + np.exp(-g)) * u
        assert np.max(np.abs(h.cpu().numpy() - ref)) <= 3e-3 * max(1.0, np.max(np.abs(ref)))
