"""2:4 sparse ternary linear on the GPU against the oracle's restatement of
the WGSL 2:4 kernel (kernels/sparse_ternary.rs:321-360), in the GPU 5-bit
layout. Same tolerances as the dense path."""
import json
import os

import numpy as np
import pytest
import torch

import ferrisres_amd as frx
import oracle
from ferrisres_amd import synth
from _gpu import assert_bf16_within_1ulp, assert_close_f32, dev_bf16, dev_f32, dev_u32, host

pytestmark = pytest.mark.gpu
KATS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "reference_kats.json")))


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a gfx950 device"
    c = frx.Context(0)
    yield c
    c.close()


def _run(ctx, meta, s, xf, xb, xt, yt):
    M, K = xf.shape
    N = meta.shape[0]
    x = dev_bf16(xb) if xt == "bf16" else dev_f32(xf)
    y = torch.empty((M, N), dtype=torch.bfloat16 if yt == "bf16" else torch.float32, device="cuda:0")
    ctx.sparse24_ternary_linear(dev_u32(meta), dev_f32(s), x, y)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("kat", KATS["sparse24_gpu"], ids=lambda k: k["source"].split()[-1])
def test_reference_kats_on_gpu(ctx, kat):
    w = np.array(kat["weights"], np.int8).reshape(kat["rows"], kat["cols"])
    meta, sc = frx.pack_sparse24_gpu(w, with_scales=True)
    x = np.array(kat["input"], np.float32).reshape(kat["seq"], kat["cols"])
    y = host(_run(ctx, meta, sc, x, None, "f32", "f32"))
    np.testing.assert_allclose(y.ravel(), kat["expected"], atol=kat["tol"], rtol=0)


@pytest.mark.parametrize("M,K,N", [(1, 96, 8), (4, 1024, 100), (16, 2048, 64), (1, 4100, 37), (33, 512, 130),
                                   (128, 4096, 256)])
@pytest.mark.parametrize("xt,yt", [("bf16", "f32"), ("f32", "f32"), ("bf16", "bf16")])
def test_sparse_parity_random(ctx, M, K, N, xt, yt):
    name = f"sp24/{M}x{K}x{N}"
    t = synth.sparse24_uniform(name, "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    s = synth.row_scales(name, "s", N, samples=256)
    xf, xb = synth.activations(name, "x", M, K)
    if xt == "f32":
        xf = synth.normal(7, M * K).reshape(M, K)
    ref = oracle.sparse24_gpu_matmul(meta, s, xf, M, K, N)
    y = _run(ctx, meta, s, xf, xb, xt, yt)
    if yt == "f32":
        assert_close_f32(host(y), ref)
    else:
        assert_bf16_within_1ulp(y.view(torch.int16).cpu().numpy().view(np.uint16), ref)


@pytest.mark.parametrize("M,K,N,xt", [(1, 100, 12, "bf16"), (2, 388, 260, "bf16"), (1, 4100, 1028, "bf16"),
                                      (2, 6004, 516, "bf16"), (1, 388, 260, "f32"), (3, 4100, 8196, "f32"),
                                      (4, 8188, 4100, "f32"),
                                      (1, 388, 8196, "bf16"), (1, 100, 8192, "f32"), (1, 4100, 8192, "bf16"),
                                      (1, 4100, 8196, "f32"), (1, 4612, 8192, "f32"), (1, 6004, 8708, "bf16"),
                                      (1, 4612, 6148, "f32"), (1, 4100, 7684, "bf16"), (1, 5124, 7172, "f32")])
@pytest.mark.parametrize("yt", ["f32", "bf16"])
def test_sparse_decode_gemv_ragged(ctx, M, K, N, xt, yt):
    """Few tokens on ragged shapes, in the row tiles (fewer than 8192 rows, or
    more than one token) and in the table GEMV (one token, 8192 rows and more):
    rows whose word count is not a multiple of 4 (a row's last 16-byte metadata
    load runs into the next row, whose words are cleared), a last chunk shorter
    than 16 words, a last row block shorter than 256 rows, row blocks that are
    and are not a multiple of 8 (both block orders), and chunk counts on both
    sides of the fused reduction's limit (4612 and 6004 columns: 13 and 16
    chunks, added by the separate launch)."""
    name = f"sp24/gemv/{M}x{K}x{N}"
    t = synth.sparse24_uniform(name, "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    s = synth.row_scales(name, "s", N, samples=256)
    xf, xb = synth.activations(name, "x", M, K)
    if xt == "f32":
        xf = synth.normal(11, M * K).reshape(M, K)
    ref = oracle.sparse24_gpu_matmul(meta, s, xf, M, K, N)
    y = _run(ctx, meta, s, xf, xb, xt, yt)
    if yt == "f32":
        assert_close_f32(host(y), ref)
    else:
        assert_bf16_within_1ulp(y.view(torch.int16).cpu().numpy().view(np.uint16), ref)


@pytest.mark.parametrize("M,K,N,xt", [(1, 100, 12, "bf16"), (2, 4, 1, "f32"), (8, 4100, 129, "f32"), (9, 396, 131, "f32"),
                                      (16, 388, 260, "bf16"), (17, 1540, 514, "bf16"), (24, 6004, 255, "f32"),
                                      (32, 772, 8196, "bf16"), (3, 14340, 127, "bf16"), (1, 5000, 8196, "f32")])
@pytest.mark.parametrize("yt", ["f32", "bf16"])
def test_sparse_row_tiles_ragged(ctx, M, K, N, xt, yt):
    """The decode-batch row tiles at their edges: rows that end inside a
    16-byte metadata load or a chunk, K % 8 == 4 (half an activation load past
    the row), N not a multiple of 4, partly filled column sets, every chunk
    count of a slice; twice (the arrival counters are left at zero)."""
    name = f"sp24/rows/{M}x{K}x{N}"
    t = synth.sparse24_uniform(name, "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    s = synth.row_scales(name, "s", N, samples=min(K, 256))
    xf, xb = synth.activations(name, "x", M, K)
    if xt == "f32":
        xf = synth.normal(13, M * K).reshape(M, K)
    ref = oracle.sparse24_gpu_matmul(meta, s, xf, M, K, N)
    for _ in range(2):
        y = _run(ctx, meta, s, xf, xb, xt, yt)
        if yt == "f32":
            assert_close_f32(host(y), ref)
        else:
            assert_bf16_within_1ulp(y.view(torch.int16).cpu().numpy().view(np.uint16), ref)


@pytest.mark.parametrize("M,K,N", [(2048, 4096, 4096), (2048, 4096, 11008), (16, 4096, 11008), (64, 11008, 512)])
def test_sparse_bit_exact_on_dyadic(ctx, M, K, N):
    """Whole output, bit for bit (dyadic x, power-of-two scales: every
    partial sum exact), including the full 2048 x 4096 x 11008 prefill."""
    rng = np.random.default_rng(M + N)
    t = synth.sparse24_uniform(f"dy/{M}", "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    x = (rng.integers(-64, 65, size=(M, K)) / 8.0).astype(np.float32)
    s = (2.0 ** rng.integers(-4, 2, size=N)).astype(np.float32)
    ref = (x @ t.T.astype(np.float32)) * s[None, :]
    y = host(_run(ctx, meta, s, x, synth.f32_to_bf16_bits(x), "bf16", "f32"))
    np.testing.assert_array_equal(y, ref)


def test_cpu_layout_through_transcoder(ctx):
    rows, cols = 64, 512
    t = synth.sparse24_uniform("tc", "w", rows, cols)
    p, sg = oracle.sparse24_cpu_from_ternary(t, rows, cols)
    meta = frx.sparse24_cpu_to_gpu(p, sg, rows, cols)
    x = synth.normal(3, 8 * cols).reshape(8, cols)
    s = np.full(rows, 0.03, np.float32)
    ref = oracle.sparse24_cpu_matmul(p, sg, 0.03, rows, cols, x, 8).reshape(8, rows)
    assert_close_f32(host(_run(ctx, meta, s, x, None, "f32", "f32")), ref)


def test_sparse_raw_metadata_patterns_6_7(ctx):
    """Raw metadata words: every 5-bit code including patterns 6 and 7
    (read as 5 by the reference) and set bits 30-31 (not part of any
    group). The prefill path (bf16, K % 64 == 0) against the oracle."""
    M, K, N = 64, 512, 256
    rng = np.random.default_rng(67)
    wpr = (K // 4 + 5) // 6
    meta = rng.integers(0, 2**32, size=(N, wpr), dtype=np.uint64).astype(np.uint32)
    s = (rng.random(N) * 0.05 + 0.01).astype(np.float32)
    xf, xb = synth.activations("sp24/raw", "x", M, K)
    xw = synth.bf16_bits_to_f32(xb)
    ref = oracle.sparse24_gpu_matmul(meta, s, xw, M, K, N)
    y = _run(ctx, meta, s, xf, xb, "bf16", "f32")
    assert_close_f32(host(y), ref)


def test_sparse_prefill_11008_sampled(ctx):
    """2:4 prefill at X[2048, 4096] x W[11008, 4096]: every output row of
    eight sampled tokens against the oracle (each row depends only on its
    token)."""
    M, K, N = 2048, 4096, 11008
    name = "sp24/prefill11008"
    t = synth.sparse24_uniform(name, "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    s = synth.row_scales(name, "s", N, samples=256)
    xf, xb = synth.activations(name, "x", M, K)
    y = host(_run(ctx, meta, s, xf, xb, "bf16", "f32"))
    rows = np.array([0, 1, 127, 128, 1000, 1919, 2046, 2047])
    xw = synth.bf16_bits_to_f32(xb)[rows]
    ref = oracle.sparse24_gpu_matmul(meta, s, np.ascontiguousarray(xw), len(rows), K, N)
    assert_close_f32(y[rows], ref.reshape(len(rows), N))


@pytest.mark.parametrize("M,K,N", [(1, 4096, 11008), (5, 11008, 4096), (16, 4096, 11008), (17, 11008, 4096),
                                   (200, 4096, 4096), (3, 2048, 300), (1600, 16384, 2048), (2, 4100, 1000),
                                   (4, 11008, 4096)])
def test_sparse_split_k_bit_exact_on_dyadic(ctx, M, K, N):
    """Decode and small prefill, where 64-token tiles leave compute units
    idle: K is split into parts of whole 64-column steps (each reading its
    own metadata windows) whose fp32 partials are added in part order. Dyadic
    inputs: every sum exact, the same bits in split mode NEVER (the unsplit
    kernels; one and two tokens work in K chunks there too) and as the dense
    product, f32 and bf16 outputs."""
    rng = np.random.default_rng(5 * M + K + N)
    t = synth.sparse24_uniform(f"dysk/{M}x{K}x{N}", "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    x = (rng.integers(-64, 65, size=(M, K)) / 8.0).astype(np.float32)
    s = (2.0 ** rng.integers(-4, 2, size=N)).astype(np.float32)
    ref = (x @ t.T.astype(np.float32)) * s[None, :]
    xb = synth.f32_to_bf16_bits(x)
    np.testing.assert_array_equal(host(_run(ctx, meta, s, x, xb, "bf16", "f32")), ref)
    yb = _run(ctx, meta, s, x, xb, "bf16", "bf16")
    np.testing.assert_array_equal(yb.view(torch.int16).cpu().numpy().view(np.uint16), synth.f32_to_bf16_bits(ref))
    ctx.set_gemv_split(frx.GEMV_SPLIT_NEVER)
    try:
        y0 = host(_run(ctx, meta, s, x, xb, "bf16", "f32"))
    finally:
        ctx.set_gemv_split(frx.GEMV_SPLIT_AUTO)
    np.testing.assert_array_equal(y0, ref)


@pytest.mark.parametrize("M,K,N", [(1, 4096, 512), (2, 4100, 512), (7, 4096, 512), (48, 4096, 512),
                                   (600, 4096, 512), (1024, 1024, 4096)])
def test_sparse_split_k_raw_metadata(ctx, M, K, N):
    """Raw metadata words (patterns 6 and 7, stray bits 30-31) through the
    split path (windows that straddle words at every step phase) and, from
    512 tokens, the prepared form (split and whole-K), against the oracle."""
    rng = np.random.default_rng(91 + M)
    wpr = (K // 4 + 5) // 6
    meta = rng.integers(0, 2**32, size=(N, wpr), dtype=np.uint64).astype(np.uint32)
    s = (rng.random(N) * 0.05 + 0.01).astype(np.float32)
    xf, xb = synth.activations(f"sp24/rawsk{M}", "x", M, K)
    ref = oracle.sparse24_gpu_matmul(meta, s, synth.bf16_bits_to_f32(xb), M, K, N)
    assert_close_f32(host(_run(ctx, meta, s, xf, xb, "bf16", "f32")), ref)


@pytest.mark.parametrize("M,K,N,xt,prepared", [(3, 4096, 4096, "bf16", False), (4, 11008, 4096, "bf16", False),
                                               (16, 4096, 512, "f32", False), (1, 4096, 4096, "bf16", True),
                                               (4, 4096, 11008, "bf16", True), (24, 2048, 1024, "bf16", True)])
def test_sparse_never_runs_whole_k(M, K, N, xt, prepared):
    """Split mode NEVER: no K parts. Seen by the fp32 partials' room, which a call in
    that mode does not allocate (and does in AUTO); the outputs agree within
    f32 sums."""
    g = torch.Generator(device="cuda:0").manual_seed(M + K + N)
    meta = _random_meta(g, N, K)
    s = 0.02 + 0.01 * torch.rand(N, generator=g, device="cuda:0")
    x = torch.randn((M, K), generator=g, device="cuda:0").to(torch.bfloat16 if xt == "bf16" else torch.float32)
    c = frx.Context(0)
    try:
        prep = torch.empty((N, K // 16), dtype=torch.int32, device="cuda:0")
        c.sparse24_prepare(meta, K, prep)
        live, out = [], []
        for mode in (frx.GEMV_SPLIT_NEVER, frx.GEMV_SPLIT_AUTO):
            c.set_gemv_split(mode)
            y = torch.full((M, N), float("nan"), device="cuda:0")
            if prepared:
                c.sparse24_prepared_linear(prep, s, x, y)
            else:
                c.sparse24_ternary_linear(meta, s, x, y)
            torch.cuda.synchronize()
            live.append(c.workspace_stats()[0])
            out.append(y.double())
    finally:
        c.close()
    planes = (M * K * 4 + 255) // 256 * 256 if xt == "f32" else 0  # f32 x as bf16 hi | lo rows
    assert live[0] == planes and live[1] > planes
    err = (torch.linalg.norm(out[0] - out[1]) / torch.linalg.norm(out[1])).item()
    assert err < (2.0 ** -20 if xt == "bf16" else 2.0 ** -16)


def _prepare(ctx, meta, K):
    N = meta.shape[0]
    prep = torch.empty((N, K // 16), dtype=torch.int32, device="cuda:0")
    ctx.sparse24_prepare(dev_u32(meta), K, prep)
    return prep


@pytest.mark.parametrize("M,K,N", [(1, 4096, 11008), (16, 1024, 300), (64, 4096, 4096), (700, 2048, 1000),
                                   (2048, 4096, 4096)])
def test_prepared_linear_bit_exact_on_dyadic(ctx, M, K, N):
    """frx_sparse24_prepare + frx_sparse24_prepared_linear: dyadic inputs give
    the exact product, and the same bits as frx_sparse24_ternary_linear,
    bf16 and f32 outputs."""
    rng = np.random.default_rng(7 * M + K + N)
    t = synth.sparse24_uniform(f"prep/{M}x{K}x{N}", "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    x = (rng.integers(-64, 65, size=(M, K)) / 8.0).astype(np.float32)
    s = (2.0 ** rng.integers(-4, 2, size=N)).astype(np.float32)
    ref = (x @ t.T.astype(np.float32)) * s[None, :]
    xb = dev_bf16(synth.f32_to_bf16_bits(x))
    prep = _prepare(ctx, meta, K)
    y = torch.empty((M, N), dtype=torch.float32, device="cuda:0")
    ctx.sparse24_prepared_linear(prep, dev_f32(s), xb, y)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(host(y), ref)
    yb = torch.empty((M, N), dtype=torch.bfloat16, device="cuda:0")
    ctx.sparse24_prepared_linear(prep, dev_f32(s), xb, yb)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(yb.view(torch.int16).cpu().numpy().view(np.uint16), synth.f32_to_bf16_bits(ref))


@pytest.mark.parametrize("M", [3, 130, 1024])
def test_prepared_linear_raw_metadata(ctx, M):
    """Raw metadata words (patterns 6 and 7, stray bits 30-31) through the
    prepared form, against the oracle and against the 5-bit entry."""
    K, N = 2048, 768
    rng = np.random.default_rng(5 + M)
    wpr = (K // 4 + 5) // 6
    meta = rng.integers(0, 2**32, size=(N, wpr), dtype=np.uint64).astype(np.uint32)
    s = (rng.random(N) * 0.05 + 0.01).astype(np.float32)
    xf, xb = synth.activations(f"sp24/prepraw{M}", "x", M, K)
    ref = oracle.sparse24_gpu_matmul(meta, s, synth.bf16_bits_to_f32(xb), M, K, N)
    prep = _prepare(ctx, meta, K)
    y = torch.empty((M, N), dtype=torch.float32, device="cuda:0")
    ctx.sparse24_prepared_linear(prep, dev_f32(s), dev_bf16(xb), y)
    torch.cuda.synchronize()
    assert_close_f32(host(y), ref)
    y5 = host(_run(ctx, meta, s, xf, xb, "bf16", "f32"))
    if M > 16:
        np.testing.assert_array_equal(host(y), y5)


@pytest.mark.parametrize("M,K,N", [(33, 4096, 4096), (48, 11008, 512), (160, 1024, 14336), (256, 4096, 11008),
                                   (517, 2048, 1000), (1024, 512, 8192)])
def test_prepared_linear_same_bits_above_32_tokens(ctx, M, K, N):
    """Random activations, whose sums depend on their order: above 32 tokens both
    forms give the same bits, split over K and in whole-K tiles, f32 and bf16
    outputs; at 32 and below they agree within f32 sums."""
    g = torch.Generator(device="cuda:0").manual_seed(M + K)
    meta = _random_meta(g, N, K)
    s = 0.02 + 0.01 * torch.rand(N, generator=g, device="cuda:0")
    prep = torch.empty((N, K // 16), dtype=torch.int32, device="cuda:0")
    ctx.sparse24_prepare(meta, K, prep)
    x = torch.randn((M, K), generator=g, device="cuda:0").to(torch.bfloat16)
    for rows, same in ((M, True), (32, False), (17, False), (2, False)):
        for dt in (torch.float32, torch.bfloat16):
            y5, yp = (torch.full((rows, N), float("nan"), dtype=dt, device="cuda:0") for _ in range(2))
            ctx.sparse24_ternary_linear(meta, s, x[:rows], y5)
            ctx.sparse24_prepared_linear(prep, s, x[:rows], yp)
            torch.cuda.synchronize()
            if same:
                assert torch.equal(y5, yp)
            else:
                err = torch.linalg.norm(y5.double() - yp.double()) / torch.linalg.norm(yp.double())
                assert err.item() < (2.0 ** -20 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("M,K,N", [(17, 512, 300), (24, 1920, 7296), (32, 2752, 8250), (25, 1024, 1025), (32, 4096, 7300),
                                   (20, 448, 4), (28, 2048, 1024)])
@pytest.mark.parametrize("yt", ["f32", "bf16"])
def test_prepared_17_to_32_tokens(ctx, M, K, N, yt):
    """17-32 tokens over prepared rows, in the row tiles and, past 24 tokens in
    many short slices (2752 x 8250, 4096 x 7300), in the tile engine, ragged rows,
    against fp64; twice (the arrival counters are left at zero). f32 sums of
    exact products: below 2^-20 of the norm; bf16 outputs one rounding."""
    g = torch.Generator(device="cuda:0").manual_seed(M + K + N)
    meta = _random_meta(g, N, K)
    s = 0.02 + 0.01 * torch.rand(N, generator=g, device="cuda:0")
    prep = torch.empty((N, K // 16), dtype=torch.int32, device="cuda:0")
    ctx.sparse24_prepare(meta, K, prep)
    x = torch.randn((M, K), generator=g, device="cuda:0").to(torch.bfloat16)
    ref = (x.double() @ _dense64(meta, K).t()) * s.double()
    for _ in range(2):
        y = torch.full((M, N), float("nan"), dtype=torch.float32 if yt == "f32" else torch.bfloat16, device="cuda:0")
        ctx.sparse24_prepared_linear(prep, s, x, y)
        torch.cuda.synchronize()
        err = (torch.linalg.norm(y.double() - ref) / torch.linalg.norm(ref)).item()
        assert err < (2.0 ** -20 if yt == "f32" else 2.0 ** -8)


def test_prepared_entry_errors(ctx):
    """K % 64 != 0 and f32 activations are refused with a status, before any
    launch; the context stays usable."""
    N, K = 64, 256
    t = synth.sparse24_uniform("prep/err", "w", N, K)
    meta = dev_u32(frx.pack_sparse24_gpu(t))
    bad = torch.empty((N, 96 // 16), dtype=torch.int32, device="cuda:0")
    with pytest.raises(frx.FrxError) as e:
        ctx.sparse24_prepare(dev_u32(frx.pack_sparse24_gpu(synth.sparse24_uniform("prep/err96", "w", N, 96))), 96,
                             bad)
    assert e.value.kind == "Shape"
    prep = _prepare(ctx, frx.pack_sparse24_gpu(t), K)
    s = dev_f32(np.full(N, 0.5, np.float32))
    y = torch.empty((2, N), dtype=torch.float32, device="cuda:0")
    with pytest.raises(frx.FrxError) as e:
        ctx.sparse24_prepared_linear(prep, s, torch.zeros((2, K), dtype=torch.float32, device="cuda:0"), y)
    assert e.value.kind == "Unsupported"
    ctx.sparse24_prepared_linear(prep, s, torch.zeros((2, K), dtype=torch.bfloat16, device="cuda:0"), y)
    torch.cuda.synchronize()
    assert float(y.abs().max()) == 0.0
    del meta


@pytest.mark.parametrize("M,K,N", [(1, 4096, 11008), (7, 2048, 1000), (130, 4096, 512), (700, 1024, 2048),
                                   (300, 1024, 11008), (2048, 1024, 2048), (4, 4096, 11008), (3, 11008, 4096)])
def test_sparse_f32_activations_bit_exact_on_dyadic(ctx, M, K, N):
    """f32 activations (the reference's dtype) as bf16 planes on the sparse pipe
    (one token over 8192 rows and more: in the table GEMV), in the row tiles,
    split over K, whole-K, and over the prepared form. Dyadic x lies in the hi
    plane: exact products and sums, f32 and bf16 outputs (what the other planes
    hold is test_sparse_f32_few_tokens_keep_every_bit's and
    test_sparse_f32_planes_error's)."""
    rng = np.random.default_rng(3 * M + K + N)
    t = synth.sparse24_uniform(f"f32sp/{M}x{K}x{N}", "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    x = (rng.integers(-64, 65, size=(M, K)) / 8.0).astype(np.float32)
    s = (2.0 ** rng.integers(-4, 2, size=N)).astype(np.float32)
    ref = (x @ t.T.astype(np.float32)) * s[None, :]
    np.testing.assert_array_equal(host(_run(ctx, meta, s, x, None, "f32", "f32")), ref)
    yb = _run(ctx, meta, s, x, None, "f32", "bf16")
    np.testing.assert_array_equal(yb.view(torch.int16).cpu().numpy().view(np.uint16), synth.f32_to_bf16_bits(ref))


@pytest.mark.parametrize("M,K,N", [(3, 4096, 4096), (64, 2048, 3000), (600, 2048, 1024), (4, 4096, 11008),
                                   (1, 4100, 1000)])
def test_sparse_f32_activations_random_parity(ctx, M, K, N):
    """Genuine f32 activations (the lo half matters) against the oracle's
    sequential f32 sums, f32 and bf16 outputs."""
    name = f"sp24f32/{M}x{K}x{N}"
    t = synth.sparse24_uniform(name, "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    s = synth.row_scales(name, "s", N, samples=256)
    xf = synth.normal(synth.seed_of(name, "xf32"), M * K).reshape(M, K)
    ref = oracle.sparse24_gpu_matmul(meta, s, xf, M, K, N)
    assert_close_f32(host(_run(ctx, meta, s, xf, None, "f32", "f32")), ref)
    yb = _run(ctx, meta, s, xf, None, "f32", "bf16")
    assert_bf16_within_1ulp(yb.view(torch.int16).cpu().numpy().view(np.uint16), ref)


def _dense64(meta, K):
    """The signed 2:4 matrix of 5-bit metadata as float64 (patterns above 5 read as 5)."""
    n, words = meta.shape
    sh = torch.arange(0, 30, 5, device=meta.device, dtype=torch.int32)
    v = ((meta[:, :, None] >> sh) & 31).view(n, words * 6)[:, :K // 4]
    pairs = torch.tensor([(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)], device=meta.device)
    pos = pairs[(v & 7).clamp(max=5).long()]
    full = torch.zeros((n, K // 4, 4), dtype=torch.float64, device=meta.device)
    for j in range(2):
        full.scatter_(2, pos[:, :, j:j + 1], (1 - 2 * ((v >> (3 + j)) & 1)).double()[:, :, None])
    return full.view(n, K)


def _random_meta(g, N, K):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, (N, (K // 4 + 5) // 6), generator=g, device="cuda:0", dtype=torch.int32)


@pytest.mark.parametrize("M,K,N", [(1, 100, 12), (1, 4096, 4096), (1, 4096, 8192), (1, 11008, 8196), (2, 1040, 1000),
                                   (2, 4096, 11008), (3, 4100, 8196), (3, 4096, 512), (4, 14336, 130), (4, 8188, 4100)])
def test_sparse_f32_few_tokens_keep_every_bit(ctx, M, K, N):
    """1-4 f32 tokens multiply all 24 bits of x. One nonzero activation per token:
    every output is 0 or +- that value, whatever the order of the sums (two
    bf16 planes would miss it by up to 2^-17). And random x against fp64: f32
    sums of exact products, below 2^-20 of the result's norm where two planes
    are 2^-18.6 off."""
    g = torch.Generator(device="cuda:0").manual_seed(M + K + N)
    meta = _random_meta(g, N, K)
    w = _dense64(meta, K)
    one = torch.ones(N, device="cuda:0")
    x = torch.zeros((M, K), device="cuda:0")
    cols = torch.randint(0, K, (M,), generator=g, device="cuda:0")
    odd = 2 * torch.randint(0, 2 ** 22, (M,), generator=g, device="cuda:0") + 1  # the last of 24 bits set
    x[torch.arange(M, device="cuda:0"), cols] = 1.0 + odd.float() * 2.0 ** -23
    y = torch.full((M, N), float("nan"), device="cuda:0")
    ctx.sparse24_ternary_linear(meta, one, x, y)
    torch.cuda.synchronize()
    assert torch.equal(y.double(), x.double() @ w.t())
    x = torch.randn((M, K), generator=g, device="cuda:0")
    ctx.sparse24_ternary_linear(meta, one, x, y)
    torch.cuda.synchronize()
    ref = x.double() @ w.t()
    assert (torch.linalg.norm(y.double() - ref) / torch.linalg.norm(ref)).item() < 2.0 ** -20


@pytest.mark.parametrize("M,K,N", [(5, 4096, 1000), (8, 1040, 516), (16, 11008, 300), (24, 4100, 130), (25, 1024, 512),
                                   (64, 2048, 1024)])
def test_sparse_f32_planes_error(ctx, M, K, N):
    """More f32 tokens travel as bf16 hi and lo: within 2^-16 of the result's
    norm (2^-17 an element), which a wrong or missing lo plane (2^-9) is not."""
    g = torch.Generator(device="cuda:0").manual_seed(M + K + N)
    meta = _random_meta(g, N, K)
    x = torch.randn((M, K), generator=g, device="cuda:0")
    s = 0.02 + 0.01 * torch.rand(N, generator=g, device="cuda:0")
    y = torch.full((M, N), float("nan"), device="cuda:0")
    ctx.sparse24_ternary_linear(meta, s, x, y)
    torch.cuda.synchronize()
    ref = (x.double() @ _dense64(meta, K).t()) * s.double()
    assert (torch.linalg.norm(y.double() - ref) / torch.linalg.norm(ref)).item() < 2.0 ** -16


def test_sparse_decode_paths_repeat_and_graph(ctx):
    """The decode GEMV (chunk sums added by the last-arriving chunk, its
    arrival counters left zero by every launch; and with a separate
    reduction over long rows) and the split-K engine: back-to-back launches
    of different shapes, then replays of captured launches with eager
    launches between, every result equal to its first eager run bit for
    bit."""
    shapes = [(1, 4096, 11008), (1, 11008, 4096), (2, 4096, 4096), (16, 4096, 4096)]
    cases = []
    for M, K, N in shapes:
        name = f"sp24/graph/{M}x{K}x{N}"
        t = synth.sparse24_uniform(name, "w", N, K)
        meta = dev_u32(frx.pack_sparse24_gpu(t))
        s = dev_f32(synth.row_scales(name, "s", N, samples=256))
        _, xb = synth.activations(name, "x", M, K)
        cases.append((meta, s, dev_bf16(xb), torch.empty((M, N), dtype=torch.float32, device="cuda:0")))

    def call(i):
        meta, s, x, y = cases[i]
        ctx.sparse24_ternary_linear(meta, s, x, y)

    for i in range(len(cases)):
        call(i)
    torch.cuda.synchronize()
    refs = [host(c[3]).copy() for c in cases]
    for rep in range(12):
        call(rep % len(cases))
    torch.cuda.synchronize()
    for i, c in enumerate(cases):
        np.testing.assert_array_equal(host(c[3]), refs[i])
    st = torch.cuda.Stream()
    ctx.set_stream(st)
    try:
        graphs = []
        for i in range(3):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=st):
                call(i)
            graphs.append(g)
        torch.cuda.synchronize()
        for rep in range(4):
            for i, g in enumerate(graphs):
                cases[i][3].fill_(float("nan"))
                with torch.cuda.stream(st):
                    g.replay()
                    call(3)  # an eager launch between replays
            torch.cuda.synchronize()
            ctx.synchronize()
            for i in range(4):
                np.testing.assert_array_equal(host(cases[i][3]), refs[i])
    finally:
        ctx.set_stream(None)


@pytest.mark.parametrize("M,K,N,xt", [(160, 1024, 11008, "bf16"), (333, 512, 11004, "f32"), (680, 512, 11008, "bf16"),
                                      (1000, 576, 5632, "bf16"), (333, 1088, 8192, "bf16"), (1400, 256, 4096, "f32")])
def test_sparse_gemm_tile_heights(ctx, M, K, N, xt):
    """2:4 tiles of 64, 96 and 128 tokens, and metadata prepared per call from 160
    tokens in whole-K tiles: dyadic activations give the exact product."""
    t = synth.sparse24_uniform(f"sp/th/{M}x{K}x{N}", "w", N, K)
    meta = frx.pack_sparse24_gpu(t)
    g = torch.Generator(device="cuda:0").manual_seed(M)
    x = (torch.randint(-8, 9, (M, K), generator=g, device="cuda:0").float() / 4)
    s = 2.0 ** torch.randint(-4, 1, (N,), generator=g, device="cuda:0").float()
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda:0")
    ctx.sparse24_ternary_linear(dev_u32(meta), s, x.to(torch.bfloat16) if xt == "bf16" else x, y)
    torch.cuda.synchronize()
    w = torch.from_numpy(np.asarray(t, np.float32).reshape(N, K)).to("cuda:0")
    assert torch.equal(y.double(), (x.double() @ w.double().t()) * s.double())


@pytest.mark.parametrize("M,K,N,xt,prepares", [(256, 1024, 14336, "bf16", False), (200, 3072, 11008, "bf16", False),
                                               (256, 512, 14336, "f32", False), (160, 4096, 11008, "bf16", True),
                                               (443, 3328, 5312, "bf16", True), (400, 768, 8192, "f32", True),
                                               (200, 1024, 11008, "f32", True), (512, 512, 14336, "bf16", True)])
def test_sparse_prepares_where_it_pays(M, K, N, xt, prepares):
    """160 to 511 tokens in whole-K tiles decode the metadata into its prepared
    form only over long rows (over 1024 columns the pass cost 17% of the call):
    seen by the room it takes in the context, N K / 4 bytes. The output is the
    same either way."""
    g = torch.Generator(device="cuda:0").manual_seed(M + K)
    meta = _random_meta(g, N, K)
    s = 2.0 ** torch.randint(-4, 1, (N,), generator=g, device="cuda:0").float()
    x = torch.randint(-8, 9, (M, K), generator=g, device="cuda:0").float() / 4
    y = torch.full((M, N), float("nan"), device="cuda:0")
    c = frx.Context(0)
    try:
        c.sparse24_ternary_linear(meta, s, x.to(torch.bfloat16) if xt == "bf16" else x, y)
        torch.cuda.synchronize()
        live = c.workspace_stats()[0] - (M * K * 4 if xt == "f32" else 0)  # f32 x as planes
        assert (live >= N * K // 4) == prepares and (prepares or live < 4096)
    finally:
        c.close()
    assert torch.equal(y.double(), (x.double() @ _dense64(meta, K).t()) * s.double())
