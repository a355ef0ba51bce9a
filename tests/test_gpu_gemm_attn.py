"""GPU parity of the step-time kernels (Linear GEMM with bf16 or Q8_0
weights, attention) and the Q8_0 quantiser against the oracle, through the C
ABI.

Bars: the GEMM with fp32 output is held to |d| <= 1e-5 * max(|ref|, 1) (its
products of bf16 inputs are exact in fp32 and only the accumulation order
differs from the oracle's); bf16 outputs to the bf16 bar (rel L2 <= 1e-2,
cos >= 0.9999) plus one bf16 ulp for a single rounding.  Attention rounds its
softmax weights to bf16 before the PV product, so both of its output types are
held to the bf16 bar.  The quantiser is bit-exact."""
import numpy as np
import pytest
import torch

import dit_hip
from conftest import assert_bf16, assert_fp32, bf16_metrics
from test_gpu_fused import SEED, as_input, check, dev_tensor, host

pytestmark = pytest.mark.gpu


# ---------------------------------------------------------------- quantiser --
def _quant_rows(orc):
    x = orc.randn(SEED + 200, (61, 3072), std=0.02)
    x[0] = 0.0                                            # d = 0 -> id = 0
    x[1] = orc.randn(SEED + 201, (3072,), std=1e-6)       # subnormal fp16 d
    x[2] = orc.randn(SEED + 202, (3072,), std=300.0)
    # exact halves: amax 127 -> d = 1, so x * id = x and roundf rounds away from 0
    x[3] = np.tile(np.array([127.0, 0.5, 1.5, -2.5, -0.5, 2.5, 126.5, -126.5], np.float32), 384)
    return x


def test_quantize_q8_0_bit_exact(orc, dev):
    print("quantize_q8_0 61x3072", flush=True)
    x = _quant_rows(orc)
    got = dit_hip.quantize_q8_0(dev_tensor(x, torch.float32))
    torch.cuda.synchronize()
    want = orc.quantize(x, 8).reshape(x.shape[0], -1)
    g = got.cpu().numpy()
    assert g.shape == want.shape
    bad = np.argwhere(g != want)
    assert bad.size == 0, f"{len(bad)} bytes differ, first at {bad[0]}"


def test_quantize_q8_0_strided_rows(orc, dev):
    x = orc.randn(SEED + 203, (33, 1024), std=0.02)
    big = dev_tensor(np.concatenate([x, np.zeros((33, 64), np.float32)], axis=1), torch.float32)
    out = torch.zeros((33, 1024 // 32 * 34 + 6), dtype=torch.uint8, device="cuda")
    dit_hip.quantize_q8_0(big[:, :1024], out=out)
    torch.cuda.synchronize()
    o = out.cpu().numpy()
    assert np.array_equal(o[:, :1088], orc.quantize(x, 8).reshape(33, -1))
    assert not o[:, 1088:].any(), "wrote past the row"


# --------------------------------------------------------------------- GEMM --
GEMM_SHAPES = [(1, 64, 64), (130, 200, 320), (256, 256, 3072), (513, 1000, 128), (64, 33, 192)]


@pytest.mark.parametrize("config", [-1, 0, 1, 2, 5, 6, 8])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", GEMM_SHAPES)
def test_gemm(orc, dev, M, N, K, out_dtype, config):
    print(f"gemm M={M} N={N} K={K} {out_dtype} config={config}", flush=True)
    a = orc.randn(SEED + 210, (M, K))
    b = orc.randn(SEED + 211, (N, K), std=0.02)
    y = dit_hip.gemm(dev_tensor(a, torch.bfloat16), dev_tensor(b, torch.bfloat16), out_dtype=out_dtype,
                     config=config)
    torch.cuda.synchronize()
    ref = orc.linear(orc.round_bf16(a), orc.round_bf16(b))
    check(host(y), ref, out_dtype, f"gemm {M}x{N}x{K}")


@pytest.mark.parametrize("config", [0, 1, 2, 5, 6, 8])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_gemm_strided_bias_addend(orc, dev, out_dtype, config):
    M, N, K = 300, 384, 512
    big_a = orc.randn(SEED + 212, (M, K + 128))
    b = orc.randn(SEED + 213, (N, K), std=0.02)
    bias = orc.randn(SEED + 214, (N,), std=0.1)
    add = orc.randn(SEED + 215, (M, N + 8))
    ad = dev_tensor(big_a, torch.bfloat16)[:, 64:64 + K]           # lda = K + 128
    addd = dev_tensor(add, out_dtype)[:, :N]                        # ldd = N + 8
    out = torch.zeros((M, N + 16), dtype=out_dtype, device="cuda")
    dit_hip.gemm(ad, dev_tensor(b, torch.bfloat16), bias=dev_tensor(bias, torch.float32),
                 addend=addd, out=out[:, :N], config=config)
    torch.cuda.synchronize()
    lin = orc.linear(orc.round_bf16(big_a[:, 64:64 + K]), orc.round_bf16(b), bias)
    ref = lin + as_input(add[:, :N], out_dtype)
    got = host(out)
    check(got[:, :N], ref, out_dtype, "gemm strided+bias+addend")
    assert not got[:, N:].any(), "wrote past N"


def test_gemm_in_place_addend(orc, dev):
    """C aliasing the addend: y += x W^T, the accumulate form of the
    attention-plus-MLP output projection."""
    M, N, K = 200, 256, 256
    a, b = orc.randn(SEED + 216, (M, K)), orc.randn(SEED + 217, (N, K), std=0.02)
    c0 = orc.randn(SEED + 218, (M, N))
    c = dev_tensor(c0, torch.float32)
    dit_hip.gemm(dev_tensor(a, torch.bfloat16), dev_tensor(b, torch.bfloat16), addend=c, out=c)
    torch.cuda.synchronize()
    assert_fp32(host(c), orc.linear(orc.round_bf16(a), orc.round_bf16(b)) + c0, what="gemm in-place")


@pytest.mark.parametrize("config", [0, 1, 2, 5, 6, 8])
def test_gemm_large_sampled_rows(orc, dev, config):
    """4608 x 3072 x 3072 (a Flux2 block's attention projection); 88 rows
    spread over every row tile are checked against the oracle."""
    M, N, K = 4608, 3072, 3072
    a = orc.randn(SEED + 219, (M, K))
    b = orc.randn(SEED + 220, (N, K), std=0.02)
    y = dit_hip.gemm(dev_tensor(a, torch.bfloat16), dev_tensor(b, torch.bfloat16), out_dtype=torch.float32,
                     config=config)
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(0, M, 53), [M - 1]]))
    ref = orc.linear(orc.round_bf16(a[rows]), orc.round_bf16(b))
    assert_fp32(host(y)[rows], ref, what="gemm 4608x3072x3072")


@pytest.mark.parametrize("config", [-1, 0, 1, 2, 5, 6, 8])
def test_gemm_grouped(orc, dev, config):
    """Five GEMMs of different N and K (and an empty one) in one launch, each
    against the oracle: the q/k/v/gate/up pattern plus ragged edges."""
    shapes = [(300, 256, 256), (300, 384, 256), (300, 136, 320), (300, 520, 128), (0, 64, 64), (47, 72, 64)]
    items, refs = [], []
    for i, (M, N, K) in enumerate(shapes):
        a = orc.randn(SEED + 240 + i, (M, K))
        b = orc.randn(SEED + 250 + i, (N, K), std=0.02)
        items.append((dev_tensor(a, torch.bfloat16), dev_tensor(b, torch.bfloat16),
                      torch.zeros((M, N), dtype=torch.float32, device="cuda")))
        refs.append(orc.linear(orc.round_bf16(a), orc.round_bf16(b)) if M else np.zeros((0, N), np.float32))
    outs = dit_hip.gemm_grouped(items, config=config)
    torch.cuda.synchronize()
    for (M, N, K), o, r in zip(shapes, outs, refs):
        assert_fp32(host(o), r, what=f"grouped gemm {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,lda_pad", [(64, 48, 16, 0), (300, 136, 40, 0), (33, 20, 3, 0), (129, 257, 200, 0),
                                           (70, 96, 64, 3), (1, 1, 1, 0)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_gemm_any_shape(orc, dev, M, N, K, lda_pad, out_dtype):
    """Shapes the tiled kernels do not take (ggml's mul_mat takes any K): K
    not a multiple of 64, a leading dimension that breaks 16-byte rows
    (lda = K + 3), single elements.  They run the masked kernel, against the
    oracle; an explicit tiled configuration refuses them."""
    print(f"gemm any M={M} N={N} K={K} lda=K+{lda_pad} {out_dtype}", flush=True)
    a = orc.randn(SEED + 230, (M, K + lda_pad))
    b = orc.randn(SEED + 231, (N, K), std=0.02)
    y = dit_hip.gemm(dev_tensor(a, torch.bfloat16)[:, :K], dev_tensor(b, torch.bfloat16), out_dtype=out_dtype)
    torch.cuda.synchronize()
    check(host(y), orc.linear(orc.round_bf16(a[:, :K]), orc.round_bf16(b)), out_dtype, f"gemm any {M}x{N}x{K}")
    y4 = dit_hip.gemm(dev_tensor(a, torch.bfloat16)[:, :K], dev_tensor(b, torch.bfloat16), out_dtype=out_dtype,
                      config=4)
    torch.cuda.synchronize()
    assert torch.equal(y4.view(torch.int16 if out_dtype == torch.bfloat16 else torch.int32),
                       y.view(torch.int16 if out_dtype == torch.bfloat16 else torch.int32))
    with pytest.raises(RuntimeError, match="K % 64 == 0"):
        dit_hip.gemm(dev_tensor(a, torch.bfloat16)[:, :K], dev_tensor(b, torch.bfloat16), config=0)


def test_gemm_any_shape_equals_tiled_on_tiled_shapes(orc, dev):
    """On a shape every kernel takes, the masked kernel accumulates k in the
    same order as the tiled ones (k-steps of 16, ascending): bit-identical C."""
    M, N, K = 200, 192, 256
    a = dev_tensor(orc.randn(SEED + 232, (M, K)), torch.bfloat16)
    b = dev_tensor(orc.randn(SEED + 233, (N, K), std=0.02), torch.bfloat16)
    outs = [dit_hip.gemm(a, b, out_dtype=torch.float32, config=c) for c in (0, 1, 2, 4, 5, 6, 8)]
    torch.cuda.synchronize()
    for c, o in zip((1, 2, 4, 5, 6, 8), outs[1:]):
        assert torch.equal(o.view(torch.int32), outs[0].view(torch.int32)), f"config {c}"
    z = torch.zeros((0, 64), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((8, 64), dtype=torch.bfloat16, device="cuda")
    assert dit_hip.gemm(z, w).shape == (0, 8)


# ------------------------------------------------------- Q8_0 weight GEMM --
def _q8_weight(orc, seed, N, K):
    """Q8_0 blocks of N(0, 0.02) weights (the device quantiser), their split
    layout and their bf16 dequantisation."""
    w = orc.randn(seed, (N, K), std=0.02)
    blocks = dit_hip.quantize_q8_0(dev_tensor(w, torch.float32))
    return blocks, dit_hip.q8_0_split(blocks, N, K), dit_hip.dequant(blocks, dit_hip.Q8_0, N, K)


def test_q8_0_split_layout(orc, dev):
    """codes = q + 128 as uint8 and scales = fp32(d) transposed, decoded from
    the block bytes on the host."""
    N, K = 37 * 4, 320
    blocks, q8, _ = _q8_weight(orc, SEED + 260, N, K)
    torch.cuda.synchronize()
    raw = blocks.cpu().numpy().reshape(N, K // 32, 34)
    d = raw[:, :, :2].copy().view(np.float16)[:, :, 0].astype(np.float32)
    qs = raw[:, :, 2:].view(np.int8).reshape(N, K)
    assert np.array_equal(q8.codes.cpu().numpy(), (qs.astype(np.int16) + 128).astype(np.uint8))
    assert np.array_equal(q8.scales.cpu().numpy(), d.T)


Q8_SHAPES = [(1, 64, 64), (130, 200, 320), (256, 256, 3072), (513, 1000, 128), (64, 33, 192), (300, 522, 256),
             (77, 130, 96), (40, 64, 32)]  # the last two: K % 64 == 32, the masked kernel


@pytest.mark.parametrize("config", [-1, 1, 3, 7, 9])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", Q8_SHAPES)
def test_gemm_q8_0_equals_dequant_then_gemm(orc, dev, M, N, K, out_dtype, config):
    """Dequantising in the GEMM's load path (config 3: 256 x 256 tiles in
    eight waves, converted after the LDS read; configs 7 and 9: the K = 64
    kernel's 256 x 256 tiles in four or eight waves and config 1: 128 x 128
    tiles, converted as they are staged; -1: picked by shape) gives the bf16 weights dt_dequant
    writes and the same fp32 accumulation order, so C is bit-identical to
    dt_dequant followed by the bf16 GEMM; and within the bar of the oracle on
    the dequantised weights."""
    if config != -1 and K % 64:
        pytest.skip("K % 64 == 32 runs the masked kernel only")
    print(f"gemm_q8_0 M={M} N={N} K={K} {out_dtype} config={config}", flush=True)
    a = orc.randn(SEED + 261, (M, K))
    _, q8, wd = _q8_weight(orc, SEED + 262, N, K)
    ad = dev_tensor(a, torch.bfloat16)
    if config == -1:
        y = dit_hip.gemm_q8_0(ad, q8, out_dtype=out_dtype)
    else:
        y = torch.empty((M, N), dtype=out_dtype, device="cuda")
        dit_hip.gemm_grouped([(ad, q8, y)], config=config)
    y_ref = dit_hip.gemm(ad, wd, out_dtype=out_dtype)
    torch.cuda.synchronize()
    assert torch.equal(y, y_ref), "Q8_0 GEMM differs from dequant + bf16 GEMM"
    check(host(y), orc.linear(orc.round_bf16(a), host(wd)), out_dtype, f"gemm_q8_0 {M}x{N}x{K}")


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_gemm_q8_0_bias_addend_strided(orc, dev, out_dtype):
    M, N, K = 300, 384, 512
    big_a = orc.randn(SEED + 263, (M, K + 128))
    _, q8, wd = _q8_weight(orc, SEED + 264, N, K)
    bias = dev_tensor(orc.randn(SEED + 265, (N,), std=0.1), torch.float32)
    add = dev_tensor(orc.randn(SEED + 266, (M, N + 8)), out_dtype)[:, :N]
    ad = dev_tensor(big_a, torch.bfloat16)[:, 64:64 + K]
    out = torch.zeros((M, N + 16), dtype=out_dtype, device="cuda")
    dit_hip.gemm_q8_0(ad, q8, bias=bias, addend=add, out=out[:, :N])
    ref = dit_hip.gemm(ad, wd, bias=bias, addend=add, out_dtype=out_dtype, config=2)
    torch.cuda.synchronize()
    assert torch.equal(out[:, :N], ref)
    assert not out[:, N:].any(), "wrote past N"


def test_gemm_q8_0_grouped_and_large(orc, dev):
    """The five projections of a single-stream block as one grouped Q8_0
    launch (4608 rows, N = 3072 x 3 + 9216 x 2, K = 3072), by the picked
    configuration and by the eight-wave kernel, bit-identical to the bf16
    grouped GEMM on the dequantised weights."""
    M, K = 4608, 3072
    a = dev_tensor(orc.randn(SEED + 267, (M, K)), torch.bfloat16)
    items_q, items_b = [], []
    for i, N in enumerate([3072, 3072, 3072, 9216, 9216]):
        _, q8, wd = _q8_weight(orc, SEED + 270 + i, N, K)
        items_q.append((a, q8, torch.empty((M, N), dtype=torch.bfloat16, device="cuda")))
        items_b.append((a, wd, torch.empty((M, N), dtype=torch.bfloat16, device="cuda")))
    outs_q = [o.clone() for o in dit_hip.gemm_grouped(items_q)]
    outs_q7 = [o.clone() for o in dit_hip.gemm_grouped(items_q, config=7)]
    outs_q3 = dit_hip.gemm_grouped(items_q, config=3)
    outs_b = dit_hip.gemm_grouped(items_b, config=2)
    torch.cuda.synchronize()
    for oq, oq7, oq3, ob in zip(outs_q, outs_q7, outs_q3, outs_b):
        assert torch.equal(oq, ob), "picked Q8_0 configuration"
        assert torch.equal(oq7, ob), "four-wave K = 64 Q8_0 kernel"
        assert torch.equal(oq3, ob), "eight-wave Q8_0 kernel"


def test_gemm_q8_0_rejects(orc, dev):
    a = torch.zeros((64, 64), dtype=torch.bfloat16, device="cuda")
    _, q8, wd = _q8_weight(orc, SEED + 280, 64, 64)
    with pytest.raises(RuntimeError, match="mixes Q8_0 and bf16"):
        dit_hip.gemm_grouped([(a, q8, torch.empty((64, 64), dtype=torch.bfloat16, device="cuda")),
                              (a, wd, torch.empty((64, 64), dtype=torch.bfloat16, device="cuda"))])
    with pytest.raises(RuntimeError, match="does not take Q8_0"):
        dit_hip.gemm_grouped([(a, q8, torch.empty((64, 64), dtype=torch.bfloat16, device="cuda"))], config=2)
    for config in (3, 7):
        with pytest.raises(RuntimeError, match="does not take bf16"):
            dit_hip.gemm_grouped([(a, wd, torch.empty((64, 64), dtype=torch.bfloat16, device="cuda"))],
                                 config=config)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("weights", ["bf16", "q8_0"])
@pytest.mark.parametrize("M,N,K", [(1, 257, 4160), (16, 4100, 320), (7, 16400, 64),         # few rows, four or eight waves
                                   (17, 5200, 256), (250, 3204, 448), (513, 4100, 320),     # two k-groups, odd k-tiles
                                   (17, 516, 2112), (300, 253, 4160), (130, 2050, 1088)])   # K ranges, ragged
def test_gemm_few_tiles(orc, dev, M, N, K, weights, out_dtype):
    """Products of few rows or few tiles, through gemm / gemm_q8_0 (K ranges with
    a workspace) and the grouped call (none), with bias, addend and strides."""
    print(f"few tiles {weights} {M}x{N}x{K} {out_dtype}", flush=True)
    assert (dit_hip.load().dt_gemm_bf16_workspace_bytes(M, N, K) > 0) == (M > 16 and K >= 1024)
    a, b = orc.randn(SEED + 270, (M, K + 8)), orc.randn(SEED + 271, (N, K), std=0.02)
    bias, add = orc.randn(SEED + 272, (N,), std=0.1), orc.randn(SEED + 273, (M, N))
    x = dev_tensor(a, torch.bfloat16)[:, :K]
    if weights == "q8_0":
        blocks = dit_hip.quantize_q8_0(dev_tensor(b, torch.float32))
        w = dit_hip.q8_0_split(blocks.view(-1), N, K)
        bw = host(dit_hip.dequant(blocks.view(-1), dit_hip.Q8_0, N, K, torch.bfloat16))
        fn = dit_hip.gemm_q8_0
    else:
        w, bw, fn = dev_tensor(b, torch.bfloat16), orc.round_bf16(b), dit_hip.gemm
    ld = (N + 3) // 4 * 4 + 4
    out = torch.zeros((M, ld), dtype=out_dtype, device="cuda")
    fn(x, w, bias=dev_tensor(bias, torch.float32), addend=dev_tensor(add, out_dtype), out=out[:, :N])
    out2 = torch.empty((M, N), dtype=out_dtype, device="cuda")
    dit_hip.gemm_grouped([(x, w, out2)])
    torch.cuda.synchronize()
    lin = orc.linear(orc.round_bf16(a[:, :K]), bw)
    got = host(out)
    check(got[:, :N], lin + bias + as_input(add, out_dtype), out_dtype, f"few tiles {M}x{N}x{K}")
    assert not got[:, N:].any(), "wrote past N"
    check(host(out2), lin, out_dtype, f"few tiles grouped {M}x{N}x{K}")


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(1, 257, 4160), (16, 16400, 64), (513, 4100, 320), (250, 3204, 448),  # few rows; two k-groups
                                   (40, 516, 2112), (130, 2050, 2112)])                           # K ranges
def test_gemm_q8_0_sum_orders_equal_dequant(orc, dev, M, N, K, out_dtype):
    """Weights of 2^20 elements and more, whose products take sum orders of their own: a
    Q8_0 weight and its dequantised copy take the same one, alone and grouped, bit for bit."""
    print(f"gemm_q8_0 sum orders M={M} N={N} K={K} {out_dtype}", flush=True)
    assert N * K >= 1 << 20
    a = dev_tensor(orc.randn(SEED + 278, (M, K)), torch.bfloat16)
    _, q8, wd = _q8_weight(orc, SEED + 279, N, K)
    y, y_ref = dit_hip.gemm_q8_0(a, q8, out_dtype=out_dtype), dit_hip.gemm(a, wd, out_dtype=out_dtype)
    outs = [torch.empty((M, N), dtype=out_dtype, device="cuda") for _ in range(2)]
    for w, out in zip((q8, wd), outs):
        dit_hip.gemm_grouped([(a, w, out)])
    torch.cuda.synchronize()
    assert torch.equal(y, y_ref) and torch.equal(*outs)


def test_prepared_launch_keeps_its_scratch(orc, dev):
    """prepare()'s repeats of calls with scratch of their own (K ranges of a
    product, fp32 attention's parts) after that memory could be given away."""
    a, b = dev_tensor(orc.randn(SEED + 274, (130, 2112)), torch.bfloat16), dev_tensor(orc.randn(SEED + 275, (2050, 2112)), torch.bfloat16)
    assert dit_hip.load().dt_gemm_bf16_workspace_bytes(130, 2050, 2112) > 0
    assert dit_hip.load().dt_gemm_f32_workspace_bytes(130, 2050, 2112) > 0
    q = dev_tensor(orc.randn(SEED + 276, (1, 70, 2, 128)), torch.float32)
    for fn, args in ((dit_hip.gemm, (a, b)), (dit_hip.gemm_f32, (a.float(), b.float())), (dit_hip.flash_attn_f32, (q, q, q))):
        out, launch = dit_hip.prepare(fn, *args)
        first = out.clone()
        others = [torch.full((n << 20,), 255, dtype=torch.uint8, device="cuda") for n in (1, 2, 4, 8, 16)]
        out.zero_()
        launch()
        torch.cuda.synchronize()
        assert torch.equal(out, first), fn.__name__
        assert all((t == 255).all() for t in others), fn.__name__


@pytest.mark.parametrize("weights", ["bf16", "q8_0"])
@pytest.mark.parametrize("M,N,K,lda,ldb", [(128, 3072, 3072, 9_000_000, None), (128, 128, 8192, None, 17_000_000),
                                           (300, 257, 4160, 9_000_000, None), (256, 65536, 64, 4_300_000, None)])
def test_gemm_long_rows(dev, M, N, K, lda, ldb, weights):
    """Rows so far apart that a tile spans more than 2^31 bytes, alone (K ranges)
    and grouped, against the same operands packed: the sums differ by their order only."""
    print(f"gemm long rows {weights} {M}x{N}x{K} lda={lda} ldb={ldb}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(SEED + 277)
    a = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    w = torch.randn((N, K), generator=g, device="cuda") * 0.02

    def far(t, ld):
        if ld is None:
            return t
        v = torch.empty(t.shape[0] * ld, dtype=t.dtype, device="cuda").as_strided(t.shape, (ld, 1))
        return v.copy_(t)

    if weights == "q8_0":
        near = dit_hip.q8_0_split(dit_hip.quantize_q8_0(w).view(-1), N, K)
        b, one = dit_hip.Q8Weight(far(near.codes, ldb), near.scales), dit_hip.gemm_q8_0
    else:
        near, one = w.bfloat16(), dit_hip.gemm
        b = far(near, ldb and ldb // 2)
    x = far(a, lda)
    want = one(a, near, out_dtype=torch.float32)
    outs = [one(x, b, out_dtype=torch.float32), torch.empty_like(want)]
    dit_hip.gemm_grouped([(x, b, outs[1])])
    torch.cuda.synchronize()
    bound = 1e-5 * want.abs().clamp(min=1.0)  # the file's bar for fp32 output
    for got in outs:
        assert ((got - want).abs() <= bound).all(), (got - want).abs().max().item()


# ---------------------------------------------------------------- attention --
def _attn_ref(orc, q, k, v, scale=None):
    """q [B, Sq, H, D] -> oracle attention per batch on the bf16-rounded values."""
    return np.stack([orc.attention(orc.round_bf16(q[i]), orc.round_bf16(k[i]), orc.round_bf16(v[i]), scale)
                     for i in range(q.shape[0])])


ATTN_SHAPES = [(1, 300, 300, 3), (2, 128, 64, 2), (1, 77, 500, 1), (1, 64, 1, 2), (1, 1, 129, 4)]


# ------------------------------------------------------------- fp32 path --
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (130, 200, 320), (256, 256, 3072), (77, 33, 40), (300, 136, 3),
                                   (129, 260, 12288), (3, 16400, 128), (16, 100, 3072), (32, 68, 176), (17, 130, 2112),
                                   (130, 253, 4160)])
def test_gemm_f32(orc, dev, M, N, K):
    """F32 weights with F32 activations (the reference's own Linear precision)
    in exact bf16 parts, against the oracle's linear at the fp32 bar
    (|d| <= 1e-5 max(|ref|, 1)); with a bias and an addend; K of any size
    (3 and 40 take the masked loads)."""
    print(f"gemm_f32 M={M} N={N} K={K}", flush=True)
    ranges = M > 32 and K >= 3072  # taken over ranges of K; N = 253: ragged partial rows
    assert (dit_hip.load().dt_gemm_f32_workspace_bytes(M, N, K) > 0) == ranges
    a = orc.randn(SEED + 280, (M, K))
    b = orc.randn(SEED + 281, (N, K), std=0.02)
    bias = orc.randn(SEED + 282, (N,), std=0.1)
    add = orc.randn(SEED + 283, (M, N))
    y = dit_hip.gemm_f32(dev_tensor(a, torch.float32), dev_tensor(b, torch.float32),
                         bias=dev_tensor(bias, torch.float32), addend=dev_tensor(add, torch.float32))
    torch.cuda.synchronize()
    assert_fp32(host(y), orc.linear(a, b, bias) + add, what=f"gemm_f32 {M}x{N}x{K}")


def test_gemm_f32_grouped_unaligned(orc, dev):
    """A group with one member that takes element-wise loads (K = 37, rows off 16
    bytes): every member is the product it is by itself, bit for bit, the few-row
    kernel's among them."""
    probs, outs, alone, keep = [], [], [], []
    for i, (N, K, off) in enumerate([(96, 256, 0), (64, 37, 0), (130, 512, 0), (40, 128, 1)]):
        a = dev_tensor(orc.randn(SEED + 400 + i, (5, K + 4)), torch.float32)[:, off:off + K]
        b = dev_tensor(orc.randn(SEED + 410 + i, (N, K), std=0.02), torch.float32)
        outs.append(torch.empty((5, N), device="cuda"))
        alone.append(dit_hip.gemm_f32(a, b))
        keep += [a, b]
        probs.append(dit_hip.GemmProblem(a.data_ptr(), a.stride(0), b.data_ptr(), K, outs[-1].data_ptr(), N, None, 0, None,
                                         5, N, K, None, 0))
    arr = (dit_hip.GemmProblem * 4)(*probs)
    dit_hip.check(dit_hip.load().dt_gemm_f32_grouped(arr, 4, dit_hip.stream()), "dt_gemm_f32_grouped")
    torch.cuda.synchronize()
    for i, (got, want) in enumerate(zip(outs, alone)):
        assert torch.equal(got, want), f"member {i}"


def _f32_edges(case, M, N, K):
    """Operands around the range in which the fp32 GEMM takes its products in
    bf16 parts: (a, b), the changed rows or columns inside one 128 x 128 tile."""
    rng = np.random.default_rng(SEED + 284)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = (0.02 * rng.standard_normal((N, K))).astype(np.float32)
    if case == "inf":
        a[5, 3], a[140, 7], b[9, 3] = np.inf, -np.inf, 0.0
    elif case == "nan":
        a[130, K - 1], b[2, 0] = np.nan, np.nan
    elif case == "huge":  # rounds past the largest bf16, and sums near 3e38
        a[7, :], a[7, 2], b[:, 2] = 0.0, 3.4e38, 0.5
        a[150] *= np.float32(2.0 ** 60)
    elif case == "tiny":  # parts and products below the smallest normal number
        a[3] *= np.float32(2.0 ** -100)
        b[70] *= np.float32(2.0 ** -110)
        a[140] *= np.float32(2.0 ** -60)
    elif case == "zero":
        a[:, :] = 0.0
        a[129] = 1.0
    elif case == "mixed":  # one large element times a tiny one
        a[4, :], b[8, :] = 0.0, 0.0
        a[4, 1], b[:, 1] = 2.0 ** 29, 2.0 ** -90
    return a, b


@pytest.mark.parametrize("case", ["inf", "nan", "huge", "tiny", "zero", "mixed"])
@pytest.mark.parametrize("M,N,K", [(160, 100, 96), (155, 130, 37)])
def test_gemm_f32_operand_range(dev, case, M, N, K):
    """Infinities, NaN, the largest and smallest magnitudes, all-zero rows:
    against 64 bits within K fp32 roundings of the sum of magnitudes (plus one
    smallest normal number per product), non-finite results the same."""
    print(f"gemm_f32 {case} {M}x{N}x{K}", flush=True)
    a, b = _f32_edges(case, M, N, K)
    y = dit_hip.gemm_f32(dev_tensor(a, torch.float32), dev_tensor(b, torch.float32))
    torch.cuda.synchronize()
    got = host(y).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64).T
        mag = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)).T
        want = ref.astype(np.float32).astype(np.float64)
        bad = ~np.isfinite(want)
        assert np.array_equal(np.isnan(got), np.isnan(want)), "NaN elsewhere"
        assert np.array_equal(got[bad & ~np.isnan(want)], want[bad & ~np.isnan(want)]), "infinities differ"
        ok = ~bad
        bound = K * (2.0 ** -24 * mag[ok] + 2.0 ** -126)
        assert (np.abs(got[ok] - ref[ok]) <= bound).all(), np.max(np.abs(got[ok] - ref[ok]) / bound)


@pytest.mark.parametrize("K", [1, 2, 3])
def test_gemm_f32_few_terms(dev, K):
    """One, two and three products, whose roundings nothing hides: within K
    fp32 roundings of the sum of magnitudes (K = 1: the rounded product)."""
    print(f"gemm_f32 K={K}", flush=True)
    rng = np.random.default_rng(SEED + 285)
    a, b = ((1.0 + 0.02 * rng.random((300, K))).astype(np.float32) for _ in "ab")
    got = host(dit_hip.gemm_f32(dev_tensor(a, torch.float32), dev_tensor(b, torch.float32))).astype(np.float64)
    ref = a.astype(np.float64) @ b.astype(np.float64).T
    if K == 1:
        assert np.array_equal(got, ref.astype(np.float32).astype(np.float64))
    assert (np.abs(got - ref) <= K * 2.0 ** -24 * np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T).all()


@pytest.mark.parametrize("k", [0, 127, 128, 300, 1039])
def test_gemm_f32_large_operand_at(dev, k):
    """One operand out of the split's range at k: its tile leaves the split products at
    the end of a run of 128 k, or after the last; the other tiles keep them."""
    print(f"gemm_f32 large operand at k={k}", flush=True)
    rng = np.random.default_rng(SEED + 286)
    M, N, K = 200, 150, 1040
    a, b = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    plain = host(dit_hip.gemm_f32(dev_tensor(a, torch.float32), dev_tensor(b, torch.float32)))
    a[3, k] *= np.float32(2.0 ** 45)
    got = host(dit_hip.gemm_f32(dev_tensor(a, torch.float32), dev_tensor(b, torch.float32)))
    assert np.array_equal(got[128:], plain[128:])
    ref = a.astype(np.float64) @ b.astype(np.float64).T
    mag = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T
    assert (np.abs(got - ref) <= K * 2.0 ** -24 * mag).all()


def test_gemm_f32_strided_in_place(orc, dev):
    """lda = K + 4, C written into a wider buffer, and C aliasing the addend."""
    M, N, K = 200, 96, 256
    big_a = orc.randn(SEED + 284, (M, K + 4))
    b = orc.randn(SEED + 285, (N, K), std=0.02)
    c0 = orc.randn(SEED + 286, (M, N + 4))
    cd = dev_tensor(c0, torch.float32)
    dit_hip.gemm_f32(dev_tensor(big_a, torch.float32)[:, :K], dev_tensor(b, torch.float32), addend=cd[:, :N],
                     out=cd[:, :N])
    torch.cuda.synchronize()
    got = host(cd)
    assert_fp32(got[:, :N], orc.linear(big_a[:, :K], b) + c0[:, :N], what="gemm_f32 strided in place")
    assert np.array_equal(got[:, N:], c0[:, N:]), "wrote past N"


@pytest.mark.parametrize("B,Sq,Skv,H", ATTN_SHAPES + [(1, 1536, 1536, 24)])
def test_flash_attn_f32(orc, dev, B, Sq, Skv, H):
    """fp32 q, k, v (the reference's F32 attention): fp32 scores, softmax and
    products, against the oracle's attention at the fp32 bar; the last shape
    is the 1536-token single-stream block's."""
    print(f"attn_f32 B={B} Sq={Sq} Skv={Skv} H={H}", flush=True)
    q = orc.randn(SEED + 290, (B, Sq, H, 128))
    k = orc.randn(SEED + 291, (B, Skv, H, 128))
    v = orc.randn(SEED + 292, (B, Skv, H, 128))
    o = dit_hip.flash_attn_f32(dev_tensor(q, torch.float32), dev_tensor(k, torch.float32),
                               dev_tensor(v, torch.float32))
    torch.cuda.synchronize()
    ref = np.stack([orc.attention(q[i], k[i], v[i]) for i in range(B)])
    assert_fp32(host(o), ref, what=f"attn_f32 {B}x{Sq}x{Skv}x{H}")


@pytest.mark.parametrize("case", ["strided", "scale0", "peaked", "inf_q", "nan_k", "inf_v", "huge_v", "tiny_v", "zero_v"])
@pytest.mark.parametrize("B,Sq,Skv,H", [(1, 130, 33, 2), (2, 40, 260, 1), (1, 33, 31, 2)])
def test_flash_attn_f32_ranges(dev, B, Sq, Skv, H, case):
    """Ragged tiles, one or more key ranges, strided rows, and operands outside
    the range the fused kernel splits (their heads run in plain fp32): against 64
    bits within 1e-5 of the largest |v| a row can meet, NaN rows the same."""
    print(f"attn_f32 {case} B={B} Sq={Sq} Skv={Skv} H={H}", flush=True)
    g = torch.Generator().manual_seed(SEED + Skv)
    q, k, v = (torch.randn((B, S, H, 128), generator=g) for S in (Sq, Skv, Skv))
    scale = {"scale0": 0.0, "peaked": 3.0}.get(case, 128 ** -0.5)
    if case == "peaked":
        k *= 30.0  # scores of thousands: one key's weight is 1, the reference moves
    elif case == "inf_q":
        q[0, 3, 0, 5] = float("inf")
    elif case == "nan_k":
        k[0, 7, H - 1, 0] = float("nan")
    elif case == "inf_v":
        v[0, 2, 0, 9] = float("-inf")
    elif case == "huge_v":
        v[:, :, 0] *= 2.0 ** 100
    elif case == "tiny_v":
        v[:, :, H - 1] *= 2.0 ** -110
    elif case == "zero_v":
        v.zero_()
    big = torch.zeros((B, Sq, H, 132), device="cuda")
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    if case == "strided":
        big[..., :128] = qd
        qd = big[..., :128]
    o = dit_hip.flash_attn_f32(qd, kd, vd, scale=scale)
    torch.cuda.synchronize()
    q, k, v = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    s = (q @ k.transpose(-1, -2).contiguous()) * scale
    ref = (torch.softmax(s, -1) @ v).permute(0, 2, 1, 3)
    got = o.cpu().double()
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(got), nan)
    inf = torch.isinf(ref)
    assert torch.equal(got[inf], ref[inf])
    vmax = torch.where(torch.isfinite(v), v.abs(), 0.0).amax((2, 3))[:, None, :, None].expand(ref.shape)
    ok = ~nan & ~inf
    # a score's fp32 rounding, 2^-24 of 128 products' magnitudes, moves a weight by as much
    smax = (q.abs() @ k.abs().transpose(-1, -2).contiguous()).nan_to_num(0.0, 0.0).amax().item() * scale
    assert ((got - ref).abs()[ok] <= max(1e-5, 2.0 ** -23 * smax) * vmax[ok]).all()


@pytest.mark.parametrize("case", ["inf_keys", "overflow", "uniform_huge_v", "late_max", "nan_row", "ragged_inf"])
def test_flash_attn_f32_native(dev, case):
    """Heads taken on the fp32 matrix cores: scores of -inf over the first 256
    keys (infinite K; finite operands whose sum overflows), weights near 1 / Skv
    on |v| near the largest float, a maximum in the last tile, NaN rows, and
    infinities in the last (partial) key tile and query block."""
    print(f"attn_f32 native {case}", flush=True)
    g = torch.Generator().manual_seed(SEED + 293)
    Sq, Skv, H, far = 140, 301, 2, 256
    q, k, v = torch.rand((1, Sq, H, 128), generator=g) + 0.5, *(torch.randn((1, Skv, H, 128), generator=g) for _ in "kv")
    dead = torch.zeros((Sq, Skv), dtype=torch.bool)  # head 0's scores that are -inf
    if case == "inf_keys":
        k[:, :far, 0], dead[:, :far] = float("-inf"), True
    elif case == "overflow":
        q[:, 1::2, 0] = 2.0 ** 64
        k[:, :far, 0] = -2.0 ** 64
        k[:, far:, 0] = torch.arange(Skv - far).float()[None, :, None]
        dead[:, :far] = True
    elif case == "uniform_huge_v":
        q[:, :, 0], v[:, :, 0] = 0.0, 1e38 * torch.sign(v[:, :1, 0])
    elif case == "late_max":
        v[0, 0, 0, 0] = 2.0 ** -120  # out of range: head 0 is native
        k[:, -1, 0] = 4.0
    elif case == "nan_row":
        q[0, 5, 0, 3] = float("nan")
    else:
        k[:, -1, 0], dead[:, -1] = float("-inf"), True
        q[0, -1, 0, 0] = float("inf")
    o = dit_hip.flash_attn_f32(*(t.cuda() for t in (q, k, v))).cpu().double()
    torch.cuda.synchronize()
    qd, kd, vd = (t[0].double().permute(1, 0, 2) for t in (q, k, v))
    s = qd @ kd.transpose(-1, -2).contiguous() / 128 ** 0.5
    s[0][dead] = float("-inf")
    if case == "ragged_inf":
        s[0, -1] = float("nan")  # inf against keys of both signs
    ref = torch.softmax(s, -1) @ vd
    got = o[0].permute(1, 0, 2)
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(got), nan), case
    # a score's fp32 rounding, 2^-24 of 128 products' magnitudes, moves a weight by as much
    live = torch.where(torch.isfinite(s), s.abs(), 0.0).amax(-1, keepdim=True)
    if case == "overflow":
        live = live.clamp(max=64.0)  # one key's weight is 1: its score moves nothing
    bound = (1e-5 + 2.0 ** -22 * live) * vd.abs().amax((1, 2), keepdim=True)
    assert ((got - ref).abs() <= bound)[~nan].all(), case


@pytest.mark.parametrize("tiny", [2.0 ** -62, 2.0 ** -79])
def test_flash_attn_f32_one_tiny_v(dev, tiny):
    """One tiny element among ordinary V takes its head to no other arithmetic:
    every other column is bit for bit what it is with a zero there, its own
    within fp32's rounding."""
    print(f"attn_f32 one tiny v {tiny}", flush=True)
    g = torch.Generator().manual_seed(SEED + 294)
    q, k, v = (torch.randn((1, S, 2, 128), generator=g).cuda() for S in (70, 130, 130))
    v[0, :, 0, 5] = 0.0
    zero = dit_hip.flash_attn_f32(q, k, v)
    v[0, 9, 0, 5] = tiny
    got = dit_hip.flash_attn_f32(q, k, v)
    torch.cuda.synchronize()
    col = got[0, :, 0, 5].double().clone()
    p = torch.softmax((q[0, :, 0].double() @ k[0, :, 0].double().t().contiguous()) / 128 ** 0.5, -1)[:, 9] * tiny
    assert ((col - p).abs() <= 1e-5 * tiny).all()
    got[0, :, 0, 5] = 0.0
    assert torch.equal(got, zero)


@pytest.mark.parametrize("up", [79, 81, 127])
def test_flash_attn_f32_large_scale(dev, up):
    """q k around 2^-up with a scale of 1.75 2^up: on either side of the scale that
    the split products are used for, and one whose log2(e) multiple is infinite."""
    print(f"attn_f32 scale 1.75 2^{up}", flush=True)
    g = torch.Generator().manual_seed(SEED + 295)
    q, k, v = (torch.randn((1, S, 2, 128), generator=g) for S in (70, 130, 130))
    q, k = q * 2.0 ** -(up // 2), k * 2.0 ** -(up - up // 2 + 3)
    o = torch.full((1, 70, 2, 128), float("nan"), device="cuda")
    dit_hip.flash_attn_f32(q.cuda(), k.cuda(), v.cuda(), scale=1.75 * 2.0 ** up, out=o)
    torch.cuda.synchronize()
    qd, kd, vd = (t[0].double().permute(1, 0, 2) for t in (q, k, v))
    ref = torch.softmax(qd @ kd.transpose(-1, -2).contiguous() * (1.75 * 2.0 ** up), -1) @ vd
    # 128 products of a score may each lose 2^-126 times the scale below fp32's range
    bound = 1e-5 + 128 * 2.0 ** (up - 126)
    got = o.cpu().double()[0].permute(1, 0, 2)
    assert ((got - ref).abs() <= min(bound, 0.25) * vd.abs().max()).all(), (got - ref).abs().max().item()


@pytest.mark.parametrize("B,Sq,Skv,H", [(1, 3, 4100, 47), (2, 130, 7000, 13)])
def test_flash_attn_f32_workspace_groups(dev, B, Sq, Skv, H):
    """Heads whose K and V parts pass the workspace's bound are taken in several
    launches (an odd count: the last one smaller): the bound holds, and each
    (batch, head) is its attention in 64 bits."""
    print(f"attn_f32 groups B={B} Sq={Sq} Skv={Skv} H={H}", flush=True)
    parts, scores = B * H * 1536 * Skv, 8 * 4 * (Sq + 128) * Skv
    assert parts > max(scores, 256 << 20) >= dit_hip.load().dt_flash_attn_f32_workspace_bytes(B, H, Sq, Skv, 128)
    g = torch.Generator(device="cuda").manual_seed(SEED + 296)
    q, k, v = (torch.randn((B, S, H, 128), generator=g, device="cuda") for S in (Sq, Skv, Skv))
    o = dit_hip.flash_attn_f32(q, k, v)
    torch.cuda.synchronize()
    for b in range(B):
        for h in range(H):
            p = torch.softmax(q[b, :, h].double() @ k[b, :, h].double().t().contiguous() / 128 ** 0.5, -1)
            ref = p @ v[b, :, h].double()
            assert ((o[b, :, h].double() - ref).abs() <= 1e-5).all(), (b, h)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,Sq,Skv,H", ATTN_SHAPES)
def test_flash_attn(orc, dev, B, Sq, Skv, H, out_dtype):
    print(f"attn B={B} Sq={Sq} Skv={Skv} H={H} {out_dtype}", flush=True)
    q = orc.randn(SEED + 230, (B, Sq, H, 128))
    k = orc.randn(SEED + 231, (B, Skv, H, 128))
    v = orc.randn(SEED + 232, (B, Skv, H, 128))
    o = dit_hip.flash_attn(dev_tensor(q, torch.bfloat16), dev_tensor(k, torch.bfloat16),
                           dev_tensor(v, torch.bfloat16), out_dtype=out_dtype)
    torch.cuda.synchronize()
    ref = _attn_ref(orc, q, k, v)
    rel, cos = bf16_metrics(host(o), ref)
    print(f"  rel_l2={rel:.2e} cos={cos:.7f}", flush=True)
    assert_bf16(host(o), ref, f"attn {B}x{Sq}x{Skv}x{H}")


def test_flash_attn_fused_qkv_views(orc, dev):
    """q, k, v as column views of one [S, 3*H*128] projection output (token
    stride 3*H*128, head stride 128), output written into a wider buffer."""
    S, H = 257, 3
    qkv = orc.randn(SEED + 233, (S, 3 * H * 128))
    d = dev_tensor(qkv, torch.bfloat16).view(1, S, 3, H, 128)
    out = torch.zeros((1, S, H + 1, 128), dtype=torch.bfloat16, device="cuda")
    dit_hip.flash_attn(d[:, :, 0], d[:, :, 1], d[:, :, 2], out=out[:, :, :H])
    torch.cuda.synchronize()
    r = qkv.reshape(1, S, 3, H, 128)
    ref = _attn_ref(orc, r[:, :, 0], r[:, :, 1], r[:, :, 2])
    got = host(out)
    assert_bf16(got[:, :, :H], ref, "attn fused-qkv views")
    assert not got[:, :, H].any(), "wrote outside the heads"


def test_flash_attn_invariants(orc, dev):
    """Constant V rows give that constant back; scale 0 gives the mean of V."""
    S, H = 200, 2
    q = dev_tensor(orc.randn(SEED + 234, (1, S, H, 128)), torch.bfloat16)
    k = dev_tensor(orc.randn(SEED + 235, (1, S, H, 128)), torch.bfloat16)
    c = np.linspace(-2, 2, 128, dtype=np.float32)
    v_const = dev_tensor(np.broadcast_to(c, (1, S, H, 128)).copy(), torch.bfloat16)
    o = dit_hip.flash_attn(q, k, v_const, out_dtype=torch.float32)
    torch.cuda.synchronize()
    cb = as_input(c, torch.bfloat16)
    # sum_j p_j * c with sum_j p_j = 1 up to the bf16 rounding of each p_j
    assert np.allclose(host(o), np.broadcast_to(cb, (1, S, H, 128)), rtol=4e-3, atol=4e-3)
    v = orc.randn(SEED + 236, (1, S, H, 128))
    o0 = dit_hip.flash_attn(q, k, dev_tensor(v, torch.bfloat16), scale=0.0, out_dtype=torch.float32)
    torch.cuda.synchronize()
    mean = as_input(v, torch.bfloat16).mean(axis=1, keepdims=True)
    assert np.allclose(host(o0), np.broadcast_to(mean, o0.shape), rtol=1e-5, atol=1e-5)


def test_flash_attn_flux2_shape_sampled(orc, dev):
    """4608 tokens x 24 heads (a 1024^2 Flux2 step); two heads x 160 queries
    are checked against the oracle over all 4608 keys."""
    S, H = 4608, 24
    q = orc.randn(SEED + 237, (1, S, H, 128))
    k = orc.randn(SEED + 238, (1, S, H, 128))
    v = orc.randn(SEED + 239, (1, S, H, 128))
    o = host(dit_hip.flash_attn(dev_tensor(q, torch.bfloat16), dev_tensor(k, torch.bfloat16),
                                dev_tensor(v, torch.bfloat16)))
    rows = np.arange(0, S, 29)
    for h in (0, 17):
        ref = orc.attention(orc.round_bf16(q[0, rows, h:h + 1]), orc.round_bf16(k[0, :, h:h + 1]),
                            orc.round_bf16(v[0, :, h:h + 1]))
        assert_bf16(o[0, rows, h:h + 1], ref, f"attn 4608x24 head {h}")


# ---------------------------------------------- attention with the QK prologue --
# dt_flash_attn_qk_bf16 normalises and rotates q as it loads it.  Its q is
# built from the same operations in the same order as dt_qk_rmsnorm_rope's
# stored output, so the attention output is compared bit for bit with that
# kernel followed by dt_flash_attn_bf16 (and with the oracle at the bf16 bar).
from test_gpu_fused import flux_positions  # noqa: E402


def _qk_then_attn(q_segs, k, v, pos, table, axis_dim=32, base=10000.0, eps=1e-6, out_dtype=torch.bfloat16):
    B, _, H, D = q_segs[0][0].shape
    Sq = sum(q.shape[1] for q, _ in q_segs)
    qn = torch.empty((B, Sq, H, D), dtype=torch.bfloat16, device="cuda")
    t0 = 0
    for q, w in q_segs:
        n = q.shape[1]
        for b in range(B):
            dit_hip.qk_rmsnorm_rope(q[b], None, w, None, pos[t0:t0 + n], axis_dim, base, eps, table=table,
                                    q_out=qn[b, t0:t0 + n])
        t0 += n
    return dit_hip.flash_attn(qn, k, v, out_dtype=out_dtype), qn


PRO_CASES = [  # (B, txt, img, Skv, H, table n_pos or None)
    (1, 0, 300, 300, 3, 512), (2, 77, 223, 290, 2, 40), (1, 16, 48, 64, 1, None), (1, 5, 1, 129, 4, 512)]


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,n_txt,n_img,Skv,H,n_pos", PRO_CASES)
def test_flash_attn_qk_prologue_bit_exact(orc, dev, B, n_txt, n_img, Skv, H, n_pos, out_dtype):
    """One segment or txt | img with their own norm weights; q as column
    views of a wider projection; a table that covers every position, one
    that covers only some (the rest computed on the device), or none."""
    print(f"attn+qk B={B} txt={n_txt} img={n_img} Skv={Skv} H={H} n_pos={n_pos} {out_dtype}", flush=True)
    Sq = n_txt + n_img
    grid = max(1, int(np.ceil(np.sqrt(max(n_img, 1)))))
    img = [[0, i // grid, i % grid, 0] for i in range(n_img)]
    pos_np = np.array([[0, 0, 0, l] for l in range(n_txt)] + img, dtype=np.int32).reshape(Sq, 4)
    pos = torch.from_numpy(np.ascontiguousarray(pos_np)).cuda()
    table = dit_hip.rope_table(n_pos, 32, 10000.0) if n_pos else None
    proj = dev_tensor(orc.randn(SEED + 240, (B, Sq, 2 * H * 128)), torch.bfloat16).view(B, Sq, 2, H, 128)
    w_txt = dev_tensor(orc.randn(SEED + 241, (128,), mean=1.0, std=0.1), torch.float32)
    w_img = dev_tensor(orc.randn(SEED + 242, (128,), mean=1.0, std=0.1), torch.float32)
    segs = ([(proj[:, :n_txt, 1], w_txt)] if n_txt else []) + [(proj[:, n_txt:, 1], w_img)]
    k = dev_tensor(orc.randn(SEED + 243, (B, Skv, H, 128)), torch.bfloat16)
    v = dev_tensor(orc.randn(SEED + 244, (B, Skv, H, 128)), torch.bfloat16)
    got = dit_hip.flash_attn_qk(segs, k, v, pos, 32, 10000.0, table=table, out_dtype=out_dtype)
    want, qn = _qk_then_attn(segs, k, v, pos, table, out_dtype=out_dtype)
    torch.cuda.synchronize()
    assert torch.equal(got, want), f"max |d| {(got.float() - want.float()).abs().max().item():g}"
    if B == 1 and n_txt and n_img:  # and against the oracle's QK + attention
        x = host(proj)[0, :, 1]
        qo = np.concatenate([orc.qk_rmsnorm_rope(x[:n_txt], host(w_txt), pos_np[:n_txt], 32, 10000.0, 1e-6),
                             orc.qk_rmsnorm_rope(x[n_txt:], host(w_img), pos_np[n_txt:], 32, 10000.0, 1e-6)])
        ref = orc.attention(orc.round_bf16(qo), orc.round_bf16(host(k)[0]), orc.round_bf16(host(v)[0]))
        assert_bf16(host(got)[0], ref, "attn+qk vs oracle")


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Sq,Skv,H", [(128, 97, 128), (129, 97, 128), (200, 64, 100), (1, 33, 2), (32, 128, 3),
                                      (65, 161, 5)])
def test_flash_attn_block_sizes(orc, dev, Sq, Skv, H, out_dtype):
    """Both query block sizes (32 while 512 blocks hold the call on a 256-CU
    card, 128 beyond) at the ends of their tiles, q as given and before its
    QK-RMSNorm + RoPE (bit for bit the two-kernel path)."""
    print(f"attn blocks Sq={Sq} Skv={Skv} H={H} {out_dtype}", flush=True)
    n_txt = Sq // 3
    test_flash_attn_qk_prologue_bit_exact(orc, dev, 1, n_txt, Sq - n_txt, Skv, H, 40, out_dtype)
    q, k, v = (orc.randn(SEED + 249 + i, (1, S, H, 128)) for i, S in enumerate((Sq, Skv, Skv)))
    o = dit_hip.flash_attn(*(dev_tensor(t, torch.bfloat16) for t in (q, k, v)), out_dtype=out_dtype)
    torch.cuda.synchronize()
    assert_bf16(host(o), _attn_ref(orc, q, k, v), "attention")


def test_flash_attn_qk_prologue_flux2_shape(orc, dev):
    """A single-stream block's attention at 1024^2: q [4608, 24, 128] taken
    from the fused projection before its norm, 512 txt + 64x64 img positions,
    theta 1e4, the host-built table: bit-identical to the two-kernel path."""
    S, H = 4608, 24
    pos_np = flux_positions(512, 64)
    pos = torch.from_numpy(pos_np).cuda()
    table = dit_hip.rope_table(512, 32, 10000.0)
    q = dev_tensor(orc.randn(SEED + 245, (1, S, H, 128)), torch.bfloat16)
    w = dev_tensor(orc.randn(SEED + 246, (128,), mean=1.0, std=0.02), torch.float32)
    k = dev_tensor(orc.randn(SEED + 247, (1, S, H, 128)), torch.bfloat16)
    v = dev_tensor(orc.randn(SEED + 248, (1, S, H, 128)), torch.bfloat16)
    got = dit_hip.flash_attn_qk([(q, w)], k, v, pos, 32, 10000.0, table=table)
    want, _ = _qk_then_attn([(q, w)], k, v, pos, table)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_flash_attn_qk_prologue_rejects(dev):
    z = torch.zeros((1, 8, 1, 128), dtype=torch.bfloat16, device="cuda")
    w = torch.ones(128, dtype=torch.float32, device="cuda")
    pos = torch.zeros((8, 4), dtype=torch.int32, device="cuda")
    with pytest.raises(dit_hip.DtError, match="axis_dim"):
        dit_hip.flash_attn_qk([(z, w)], z, z, pos, 24, 10000.0)      # 4 x 24 != 128
    with pytest.raises(dit_hip.DtError, match="axis_dim"):
        dit_hip.flash_attn_qk([(z, w)], z, z, pos[:, :2], 36, 10000.0)  # axis_dim % 8 != 0


@pytest.mark.parametrize("lo,hi", [(32, 64), (0, 32), (0, 64), (64, 96), (96, 200)])
@pytest.mark.parametrize("inf", [True, False])
def test_flash_attn_minus_inf_tiles(dev, lo, hi, inf):
    """Keys [lo, hi) whose scores are all -inf (infinite K, or finite operands
    whose sum overflows), in blocks of 32 queries: weight 0, as with every key
    tile that a wave does not begin on; all keys -inf gives NaN."""
    print(f"attn -inf keys {lo}..{hi} inf={inf}", flush=True)
    g = torch.Generator().manual_seed(SEED + 251)
    q = torch.rand((1, 40, 2, 128), generator=g) + 0.5
    k, v = torch.randn((1, 200, 2, 128), generator=g) * 0.1, torch.randn((1, 200, 2, 128), generator=g)
    dead = (Ellipsis,) if inf else (0,)  # the dims that make a score -inf
    if not inf:
        q[:, :, 0, 0], k[:, :, 0, 0] = 0.0, 0.0
        q[:, 3, 0, 0] = 1e20
    k[(0, slice(lo, hi), 0) + dead] = float("-inf") if inf else -1e20
    qd, kd, vd = (t.bfloat16().cuda() for t in (q, k, v))
    o = dit_hip.flash_attn(qd, kd, vd).float().cpu()
    k[(0, slice(None), 0) + dead] = float("-inf") if inf else -1e20
    none = dit_hip.flash_attn(qd, k.bfloat16().cuda(), vd).float().cpu()
    torch.cuda.synchronize()
    rows = slice(None) if inf else slice(3, 4)
    assert torch.isnan(none[:, rows, 0]).all() and not torch.isnan(none[:, :, 1]).any()
    qf, kf, vf = (t.float().cpu().permute(0, 2, 1, 3) for t in (qd, kd, vd))
    s = (qf @ kf.transpose(-1, -2).contiguous()) / 128 ** 0.5
    ref = (torch.softmax(s.double(), -1) @ vf.double()).permute(0, 2, 1, 3)
    assert not torch.isnan(o).any()
    assert_bf16(o.numpy(), ref.float().numpy(), f"attention with keys {lo}..{hi} at -inf")


@pytest.mark.parametrize("Sq,Skv,H", [(320, 320, 24), (40, 33, 2), (33, 500, 3), (20, 1000, 5)])
def test_flash_attn_block_sizes_agree(dev, Sq, Skv, H):
    """Blocks of 32 queries and (the same inputs in a batch too large for them) of
    128: softmax weights rounded to bf16 at the same scale, so what differs is the
    order of fp32 sums.  That moves an exponent by about 2^-21 and so 2^-21 / 2^-9
    of the weights and results across a bf16 rounding step of 2^-8: sqrt(2^-12)
    2^-8 = 6e-5 in the 2-norm, four times which is allowed.  (Weights rounded at scales
    of their own differ by 2.7e-3.)"""
    print(f"attn block sizes agree Sq={Sq} Skv={Skv} H={H}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(SEED + 252)
    q, k, v = (torch.randn((1, S, H, 128), generator=g, device="cuda").bfloat16() for S in (Sq, Skv, Skv))
    few = dit_hip.flash_attn(q, k, v)
    B = 1024 // (H * ((Sq + 31) // 32)) + 1  # over two blocks of 32 queries per CU
    many = dit_hip.flash_attn(*(t.expand(B, -1, -1, -1).contiguous() for t in (q, k, v)))
    torch.cuda.synchronize()
    a, b = few[0].double(), many[B // 2].double()
    assert ((a - b).norm() / b.norm()).item() <= 2.4e-4
