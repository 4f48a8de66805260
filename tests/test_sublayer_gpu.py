"""GPU parity of the attention sublayer kernels (include/sdxl_hip/sublayer.h), called
through the C ABI, against the CPU oracle's restatements of the reference
(src/unet.cpp:237-263 LayerNorm, :202-222 linear, :91-119 E4M3 decode,
src/cuda/weights.cu:119-170 row quantisation) on identical fp16 inputs.

Bars:
* E4M3 decode and the row quantiser: bit-exact.
* LayerNorm, linear: the oracle's fp32 result rounded once to fp16, i.e.
  |got - ref| <= |ref| * 2^-11 (half an fp16 ulp) + a few fp32 reassociation
  ulps; written below as |ref| * 2^-10 + 1e-5 (LN) / + 1e-4 (K = 640 sums).
* The sublayers (configs[3]: LN -> fused E4M3 QKV -> attention -> fp16 out-proj +
  bias + residual; the cross half at level 2): equal to the composition of the
  individual calls (same kernels, bit-exact), and at the parity bar (2e-3 max-abs
  beyond the fp16 output's own rounding, 2e-4 mean-abs) against the oracle's
  restatement of the reference's block order (oracle.attn_sublayer /
  cross_attn_sublayer, pinned bit-exact to the reference's own transformer_block)
  on the E4M3-dequantised weights, on row subsets at full size; an fp32 torch
  restatement covers every row at the same bar.
"""
import numpy as np
import pytest

import oracle
import sdxl_hip as sh
from parity import assert_parity_f16_out

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"
THREADS = min(16, __import__("os").cpu_count() or 1)


def dev16(bits):
    return torch.from_numpy(np.ascontiguousarray(bits).view(np.int16)).to(DEV).view(torch.float16)


def host(t):
    return t.float().cpu().numpy()


def f16(x32):
    """fp32 -> fp16 bits with the oracle's rounding."""
    return oracle.f32_to_f16_bits(np.asarray(x32, np.float32))


def within_half_ulp(got, ref, abs_floor, label):
    err = np.abs(got.astype(np.float64) - ref.astype(np.float64))
    bound = np.abs(ref) * 2.0 ** -10 + abs_floor
    worst = np.max(err - bound)
    print(f"{label}: max_abs={err.max():.3e} worst_margin={worst:.3e}", flush=True)
    assert np.isfinite(got).all(), label
    assert (err <= bound).all(), (label, float(err.max()))


# ---------------------------------------------------------------- E4M3

def test_e4m3_decode_all_codes_bit_exact():
    """A one-hot activation matrix picks every weight code: c[m, n] = decode(w[n, m])."""
    table = oracle.e4m3_table()
    codes = (np.arange(256)[:, None] + np.arange(64)[None, :]) % 256
    codes = np.where(np.isnan(table[codes]), 0, codes).astype(np.uint8)  # NaN codes excluded
    w = torch.from_numpy(codes).to(DEV)
    a = torch.eye(64, dtype=torch.float16, device=DEV)
    ones = torch.ones(256, dtype=torch.float32, device=DEV)
    got = host(sh.linear(a, w, w_scale=ones))
    np.testing.assert_array_equal(got, table[codes].T)


def test_quantizer_matches_oracle_bit_exact():
    Wb = oracle.normal_f16(910, (1920, 640), 0.02)
    Wb[7, :] = 0                                  # all-zero row -> scale 1
    Wb[8, 3] = f16(np.float32([65504.0]))[0]      # large outlier dominates its row
    Wf = oracle.f16_bits_to_f32(Wb)
    q, s = sh.quantize_e4m3_rows(dev16(Wb))
    torch.cuda.synchronize()
    q_ref, s_ref = oracle.quantize_e4m3_rows(Wf)
    np.testing.assert_array_equal(s.cpu().numpy(), s_ref)
    np.testing.assert_array_equal(q.cpu().numpy(), q_ref)


# ---------------------------------------------------------------- LayerNorm

@pytest.mark.parametrize("rows,width", [(8192, 640), (77, 320), (5, 1280), (3, 2048), (1, 128), (4, 66), (77, 640),
                                        (19, 256)])
def test_layer_norm(rows, width):
    xb = oracle.normal_f16(920 + width, (rows, width))
    gb = oracle.normal_f16(921, (width,), 0.5)
    bb = oracle.normal_f16(922, (width,), 0.5)
    got = host(sh.layer_norm(dev16(xb), dev16(gb), dev16(bb)))
    ref = oracle.layer_norm(oracle.f16_bits_to_f32(xb), oracle.f16_bits_to_f32(gb), oracle.f16_bits_to_f32(bb))
    within_half_ulp(got, ref, 1e-5, f"LN {rows}x{width}")


@pytest.mark.parametrize("width", [640, 1280])
def test_layer_norm_large_mean(width):
    """Rows of mean ~100 with unit spread (the centred variance must not cancel), and a constant
    row (variance 0: y = beta): the four-rows / two-rows kernels against the oracle, fp16 and E4M3."""
    rows = 48
    xf = oracle.f16_bits_to_f32(oracle.normal_f16(1130 + width, (rows, width))) + np.float32(100.0)
    xf[5, :] = 3.25
    xb = f16(xf)
    gb = oracle.normal_f16(1131, (width,), 0.5)
    bb = oracle.normal_f16(1132, (width,), 0.5)
    ref = oracle.layer_norm(oracle.f16_bits_to_f32(xb), oracle.f16_bits_to_f32(gb), oracle.f16_bits_to_f32(bb))
    got = host(sh.layer_norm(dev16(xb), dev16(gb), dev16(bb)))
    within_half_ulp(got, ref, 2e-5, f"LN large mean {width}")
    q, s = sh.layer_norm_e4m3(dev16(xb), dev16(gb), dev16(bb))
    torch.cuda.synchronize()
    q_ref, s_ref = oracle.quantize_e4m3_rows(ref)
    s_got = s.cpu().numpy()
    np.testing.assert_allclose(s_got, s_ref, rtol=1e-5)
    y = oracle.e4m3_table()[q.cpu().numpy()] * s_got[:, None]
    err = np.abs(y.astype(np.float64) - ref)
    # as test_layer_norm_e4m3: half an E4M3 step of y / scale, 5 % for rounding ties
    bound = e4m3_half_step(ref / s_ref[:, None]) * s_ref[:, None] * 1.05 + 1e-6 * np.abs(ref) + 1e-7
    assert (err <= bound).all(), float(err.max())
    assert (q.cpu().numpy() == q_ref).mean() >= 0.9999


def test_layer_norm_strided_in_place():
    base = dev16(oracle.normal_f16(925, (50, 768)))
    x = base[:, :640]
    gb, bb = np.full(640, f16(1.0), np.uint16), np.zeros(640, np.uint16)
    ref = oracle.layer_norm(host(x), np.ones(640, np.float32), np.zeros(640, np.float32))
    tail = base[:, 640:].clone()
    sh.layer_norm(x, dev16(gb), dev16(bb), out=x)
    within_half_ulp(host(x), ref, 1e-5, "LN in place")
    assert torch.equal(base[:, 640:], tail)


# ---------------------------------------------------------------- linear

def _linear_ref(a_bits, w32, bias_bits=None, res_bits=None):
    ref = oracle.linear(oracle.f16_bits_to_f32(a_bits), w32,
                        None if bias_bits is None else oracle.f16_bits_to_f32(bias_bits))
    if res_bits is not None:
        ref = ref + oracle.f16_bits_to_f32(res_bits)
    return ref


@pytest.mark.parametrize("M,N,K", [(300, 640, 640), (129, 200, 64), (7, 1920, 640), (256, 1280, 1280),
                                   (4500, 640, 640)])  # 71 m blocks: grouped task order, partial last group
def test_linear_fp16_bias_residual(M, N, K):
    ab = oracle.normal_f16(930 + M, (M, K))
    wb = oracle.normal_f16(931 + N, (N, K), 0.02)
    bb = oracle.normal_f16(932, (N,), 0.02)
    rb = oracle.normal_f16(933, (M, N))
    got = host(sh.linear(dev16(ab), dev16(wb), bias=dev16(bb), residual=dev16(rb)))
    ref = _linear_ref(ab, oracle.f16_bits_to_f32(wb), bb, rb)
    within_half_ulp(got, ref, 1e-4, f"linear fp16 {M}x{N}x{K}")
    plain = host(sh.linear(dev16(ab), dev16(wb)))
    within_half_ulp(plain, _linear_ref(ab, oracle.f16_bits_to_f32(wb)), 1e-4, "linear fp16 plain")


@pytest.mark.parametrize("M,N", [(8192, 1920), (8100, 1920), (333, 1920), (8192, 1000)])
def test_linear_e4m3_qkv(M, N):
    """configs[3] fused QKV projection: [M, 640] x E4M3 [1920, 640] with per-row scales (M >= 8100:
    256 x 128 tiles of 8 waves; N = 1000: a ragged last column tile, with bias and residual)."""
    K = 640
    ab = oracle.normal_f16(940, (M, K))
    Wf = oracle.normal_f32(941, (N, K), 0.02)
    q, s = oracle.quantize_e4m3_rows(Wf)
    extras = N % 128 != 0
    bb = oracle.normal_f16(942, (N,), 0.02) if extras else None
    rb = oracle.normal_f16(943, (M, N)) if extras else None
    got = host(sh.linear(dev16(ab), torch.from_numpy(q).to(DEV), w_scale=torch.from_numpy(s).to(DEV),
                         bias=dev16(bb) if extras else None, residual=dev16(rb) if extras else None))
    # the first 256-row tile whole (all four wave rows), a middle block, the last rows
    rows = np.r_[0:256, M // 2:M // 2 + 32, M - 64:M] if M > 512 else np.arange(M)
    ref = _linear_ref(ab[rows], oracle.dequantize_e4m3_rows(q, s), bb, rb[rows] if extras else None)
    within_half_ulp(got[rows], ref, 1e-4, f"linear E4M3 {M}x{N}x{K}")


# Shapes of the producer-wave forms on a 256-CU device (64-row tiles, few workgroups per CU):
# fp16 weights with one round of tiles (ring of four: the per-request context K/V projections, a
# ragged 70-row call), at most 1.25 tiles per CU (ring of three: the level-2 out-projection, a
# ragged last row and column tile), and E4M3 weights (ring of two); in place over the residual.
@pytest.mark.parametrize("M,N,K,w8", [(154, 2560, 2048, False), (154, 1280, 2048, False), (70, 1000, 1280, False),
                                      (2048, 1280, 1280, False), (2040, 1276, 1280, False),
                                      (2048, 1280, 1280, True), (1990, 1220, 1280, True), (154, 2560, 2048, True)])
def test_linear_producer_waves(M, N, K, w8):
    """The projection forms whose transfers are issued by producer waves (deeper rings with fp16
    weights) against the fp32 oracle within half an fp16 ulp, with bias and residual, and in
    place (c over the residual: each element's residual read by the lane that writes it)."""
    print(f"linear producers M{M} N{N} K{K} w8={w8}", flush=True)
    ab = oracle.normal_f16(960 + M, (M, K))
    bb = oracle.normal_f16(962, (N,), 0.02)
    rb = oracle.normal_f16(963, (M, N))
    if w8:
        q, sc = oracle.quantize_e4m3_rows(oracle.normal_f32(961 + N, (N, K), 0.02))
        w, ws, w32 = torch.from_numpy(q).to(DEV), torch.from_numpy(sc).to(DEV), oracle.dequantize_e4m3_rows(q, sc)
    else:
        wb = oracle.normal_f16(961 + N, (N, K), 0.02)
        w, ws, w32 = dev16(wb), None, oracle.f16_bits_to_f32(wb)
    got = host(sh.linear(dev16(ab), w, w_scale=ws, bias=dev16(bb), residual=dev16(rb)))
    ref = _linear_ref(ab, w32, bb, rb)
    within_half_ulp(got, ref, 1e-4, f"linear producers {M}x{N}x{K} w8={w8}")
    y = dev16(rb)
    sh.linear(dev16(ab), w, w_scale=ws, bias=dev16(bb), residual=y, out=y)
    torch.cuda.synchronize()
    assert np.array_equal(host(y), got)


# Shapes of the K-split form (output projections: a residual; 64 x 160 tiles, one round on a
# 256-CU device: n % 8 == 0 and 230-256 tiles): the level-2 out-projection, ragged last row and
# column tiles, no bias; without a residual the same shapes run the 64 x 128 kernel.
@pytest.mark.parametrize("M,N,K,bias", [(2048, 1280, 1280, True), (1990, 1272, 1280, True), (2048, 1280, 640, False),
                                        (1900, 1280, 2048, True)])
def test_linear_k_split(M, N, K, bias):
    """The K-split projection (four waves per tile, each over a quarter of every K stage, partial
    tiles summed through LDS in a fixed order) against the fp32 oracle within half an fp16 ulp, and
    in place over the residual, bit-equal to the out-of-place call."""
    print(f"linear k-split M{M} N{N} K{K} bias={bias}", flush=True)
    ab = oracle.normal_f16(970 + M, (M, K))
    wb = oracle.normal_f16(971 + N, (N, K), 0.02)
    bb = oracle.normal_f16(972, (N,), 0.02) if bias else None
    rb = oracle.normal_f16(973, (M, N))
    w32 = oracle.f16_bits_to_f32(wb)
    b_dev = dev16(bb) if bias else None
    got = host(sh.linear(dev16(ab), dev16(wb), bias=b_dev, residual=dev16(rb)))
    within_half_ulp(got, _linear_ref(ab, w32, bb, rb), 1e-4, f"linear k-split {M}x{N}x{K}")
    y = dev16(rb)
    sh.linear(dev16(ab), dev16(wb), bias=b_dev, residual=y, out=y)
    torch.cuda.synchronize()
    assert np.array_equal(host(y), got)


@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (31, 40, 64), (33, 72, 128), (154, 2560, 2048), (77, 1280, 768),
                                   (200, 648, 640), (320, 2560, 576), (300, 1000, 1280)])
@pytest.mark.parametrize("extras", [False, True])
def test_linear_few_rows(M, N, K, extras):
    """The 32 x 32, 32 x 64 and 64 x 64 tiles of the K-split kernel and the rows beyond them: edges of the
    tile, K below and above its ring."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(M, K, device=DEV, generator=g).half()
    w = (torch.randn(N, K, device=DEV, generator=g) / K ** 0.5).half()
    bias = torch.randn(N, device=DEV, generator=g).half() if extras else None
    res = torch.randn(M, N, device=DEV, generator=g).half() if extras else None
    ref = a.double() @ w.double().t()
    if extras:
        ref = ref + bias.double() + res.double()
    out = res.clone() if extras else None  # in place where there is a residual
    got = sh.linear(a, w, bias=bias, residual=out if extras else None, out=out)
    # half an fp16 ulp of the result plus fp32 sums of K products of magnitude ~1/sqrt(K)
    err = (got.double() - ref).abs() - ref.abs() * 2.0 ** -11
    assert err.max().item() <= 1e-5, err.max().item()


def test_linear_k_split_strided():
    """The K-split form on strided operands: a a column slice of a wider buffer, w rows padded, the
    residual and the output column slices of wider buffers (in place and out of place)."""
    M, N, K = 2048, 1280, 1280
    ab = oracle.normal_f16(980, (M, 3 * K))
    wb = oracle.normal_f16(981, (N, K + 64), 0.02)
    bb = oracle.normal_f16(982, (N,), 0.02)
    rb = oracle.normal_f16(983, (M, 2 * N))
    a = dev16(ab)[:, K:2 * K]
    w = dev16(wb)[:, :K]
    ref = _linear_ref(np.ascontiguousarray(ab[:, K:2 * K]), oracle.f16_bits_to_f32(np.ascontiguousarray(wb[:, :K])),
                      bb, np.ascontiguousarray(rb[:, N:]))
    outbuf = torch.zeros(M, 2 * N, dtype=torch.float16, device=DEV)
    resbuf = dev16(rb)
    sh.linear(a, w, bias=dev16(bb), residual=resbuf[:, N:], out=outbuf[:, :N])
    got = host(outbuf[:, :N])
    within_half_ulp(got, ref, 1e-4, "linear k-split strided")
    assert not host(outbuf[:, N:]).any()  # nothing written past the output columns
    sh.linear(a, w, bias=dev16(bb), residual=resbuf[:, N:], out=resbuf[:, N:])
    torch.cuda.synchronize()
    assert np.array_equal(host(resbuf[:, N:]), got)
    assert np.array_equal(host(resbuf[:, :N]), oracle.f16_bits_to_f32(rb[:, :N]))


def test_linear_strided_in_place_residual():
    """a as a column slice of a wider buffer, c written over the residual (y += x W^T + b)."""
    M, K, N = 200, 640, 640
    big = dev16(oracle.normal_f16(950, (M, 3 * K)))
    a = big[:, K:2 * K]
    wb = oracle.normal_f16(951, (N, K), 0.02)
    bb = oracle.normal_f16(952, (N,), 0.02)
    yb = oracle.normal_f16(953, (M, N))
    y = dev16(yb)
    ref = _linear_ref(f16(host(a)), oracle.f16_bits_to_f32(wb), bb, yb)
    sh.linear(a, dev16(wb), bias=dev16(bb), residual=y, out=y)
    within_half_ulp(host(y), ref, 1e-4, "linear in place")


# ---------------------------------------------------------------- LayerNorm fused into the projection

@pytest.mark.parametrize("M,N,bias,strided,K", [(8192, 1920, False, False, 640), (8100, 1920, True, False, 640),
                                                (200, 640, True, True, 640), (1, 128, False, False, 640),
                                                (4096, 128, False, True, 640), (130, 3840, True, False, 640),
                                                (1000, 1920, False, False, 640), (15360, 1920, True, False, 640),
                                                (2048, 3840, False, False, 1280), (2000, 3840, True, False, 1280),
                                                (2048, 1280, True, True, 1280), (70, 1280, False, False, 1280),
                                                (1, 128, True, False, 1280), (3840, 3840, False, False, 1280),
                                                (300, 2560, True, True, 1280)])
def test_layer_norm_linear(M, N, bias, strided, K):
    """sdxl_layer_norm_linear (norm1 -> q|k|v at width 640 and 1280; at 1280 the kernel keeps K
    columns 640-1279 of the normalised rows in LDS) equals sdxl_layer_norm followed by
    sdxl_linear bit for bit (same LayerNorm rounding, same fp32 sums), and the oracle's fp32
    LayerNorm, rounded to fp16 as the reference stores it, then linear on the dequantised
    weights, within the linear bar. Non-trivial gamma/beta; ragged row blocks (8100, 200, 130,
    1); one- and several-chunk column ranges, uneven splits (1000 rows: 15 chunks over 16
    workgroups of a row block is capped at one chunk each; 130 x 3840: 30 chunks, two
    workgroups of at most 2048 columns; 15360 rows, configs[4]'s level 1: 240 row blocks, every
    workgroup on all 15 chunks; width 1280: the level-2 q|k|v [2048, 3840] and q [2048, 1280],
    configs[4]'s level 2 [3840, 3840], at most 1024 columns per workgroup: 300 x 2560 splits 20
    chunks in two); strided x and c."""
    print(f"ln_linear M{M} N{N} K{K} bias{bias} strided{strided}", flush=True)
    xb = oracle.normal_f16(1100 + M, (M, K))
    gb = oracle.normal_f16(1101, (K,), 0.5)
    bb = oracle.normal_f16(1102, (K,), 0.5)
    q, s = oracle.quantize_e4m3_rows(oracle.normal_f32(1103 + N, (N, K), 0.02))
    biasb = oracle.normal_f16(1104, (N,), 0.02) if bias else None
    if strided:
        x = dev16(np.concatenate([xb, oracle.normal_f16(1105, (M, 128))], axis=1))[:, :K]
        out_base = torch.zeros((M, N + 64), dtype=torch.float16, device=DEV)
        out = out_base[:, :N]
    else:
        x, out = dev16(xb), None
    g, b = dev16(gb), dev16(bb)
    wq, ws = torch.from_numpy(q).to(DEV), torch.from_numpy(s).to(DEV)
    bias_t = dev16(biasb) if bias else None
    got = sh.layer_norm_linear(x, g, b, wq, ws, bias=bias_t, out=out)
    comp = sh.linear(sh.layer_norm(x, g, b), wq, w_scale=ws, bias=bias_t)
    torch.cuda.synchronize()
    assert torch.equal(got, comp)
    if strided:
        assert torch.count_nonzero(out_base[:, N:]) == 0
    rows = np.r_[0:64, M // 2:M // 2 + 32, M - 70:M] if M > 256 else np.arange(M)
    n32 = oracle.layer_norm(oracle.f16_bits_to_f32(xb[rows]), oracle.f16_bits_to_f32(gb), oracle.f16_bits_to_f32(bb))
    wdq = oracle.dequantize_e4m3_rows(q, s)
    ref = _linear_ref(f16(n32), wdq, biasb)
    # the LayerNorm output may sit one fp16 rounding away from the oracle's (half an ulp
    # each, pinned by test_layer_norm); its worst-case effect on each sum is added to the bar
    ln_term = (np.abs(n32).astype(np.float64) * 2.0 ** -11) @ np.abs(wdq.astype(np.float64)).T
    err = np.abs(host(got)[rows].astype(np.float64) - ref)
    bound = np.abs(ref) * 2.0 ** -10 + 1e-4 + ln_term
    print(f"LN+linear {M}x{N}: max_abs={err.max():.3e} worst_margin={np.max(err - bound):.3e}", flush=True)
    assert (err <= bound).all(), float(err.max())


@pytest.mark.parametrize("M,N,bias,K", [(8192, 1920, False, 640), (8100, 1920, True, 640), (130, 3840, True, 640),
                                        (1, 128, False, 640), (1000, 1920, False, 640), (15360, 1920, False, 640),
                                        (2048, 3840, False, 1280), (2000, 1280, True, 1280), (70, 3840, True, 1280),
                                        (3840, 3840, False, 1280)])
def test_layer_norm_linear_e4m3_activations(M, N, bias, K):
    """sdxl_layer_norm_linear_e4m3 (E4M3 LayerNorm rows with per-row scales, fp8 MFMA, inside one
    kernel) equals sdxl_layer_norm_e4m3 followed by sdxl_linear_e4m3 bit for bit; the product
    part against the fp64 product of the decoded codes (the E4M3 LayerNorm itself is pinned to
    the oracle by test_layer_norm_e4m3); widths 640 and 1280."""
    print(f"ln_linear e4m3 M{M} N{N} K{K} bias{bias}", flush=True)
    xb = oracle.normal_f16(1120 + M, (M, K))
    gb = oracle.normal_f16(1121, (K,), 0.5)
    bb = oracle.normal_f16(1122, (K,), 0.5)
    q, s = oracle.quantize_e4m3_rows(oracle.normal_f32(1123 + N, (N, K), 0.02))
    biasb = oracle.normal_f16(1124, (N,), 0.02) if bias else None
    x, g, b = dev16(xb), dev16(gb), dev16(bb)
    wq, ws = torch.from_numpy(q).to(DEV), torch.from_numpy(s).to(DEV)
    bias_t = dev16(biasb) if bias else None
    got = sh.layer_norm_linear(x, g, b, wq, ws, bias=bias_t, fp8_activations=True)
    codes, cs = sh.layer_norm_e4m3(x, g, b)
    comp = sh.linear_e4m3(codes, cs, wq, ws, bias=bias_t)
    torch.cuda.synchronize()
    assert torch.equal(got, comp)
    rows = np.r_[0:64, M // 2:M // 2 + 32, M - 70:M] if M > 256 else np.arange(M)
    ref = oracle.dequantize_e4m3_rows(codes.cpu().numpy()[rows], cs.cpu().numpy()[rows]).astype(np.float64) @ \
        oracle.dequantize_e4m3_rows(q, s).astype(np.float64).T
    if bias:
        ref = ref + oracle.f16_bits_to_f32(biasb)[None, :]
    within_half_ulp(host(got)[rows], ref, 1e-4, f"LN E4M3 + linear {M}x{N}")


@pytest.mark.parametrize("B,S,H", [(2, 4096, 10), (2, 1024, 20)])
def test_sublayer_layer_norm_fusion_switch(B, S, H):
    """configs[3] sublayer and the level-2 self half ([2, 1024, 1280], 20 heads) with the default
    LayerNorm placement (inside the q|k|v projection at level 1; its own launch at level 2, where
    that is faster) and with the LayerNorm as its own launch (ln_fusion off), fp16 and E4M3
    activations: the same bits."""
    W = 64 * H
    x, gamma, beta, q8, s8, w_out, b_out = _sublayer_inputs(B, S, H, 1110)
    gamma = dev16(oracle.normal_f16(1111, (W,), 0.5))
    beta = dev16(oracle.normal_f16(1112, (W,), 0.5))
    for fp8 in (False, True):
        y1 = sh.attn_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H, fp8_activations=fp8)
        y2 = sh.attn_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H, fp8_activations=fp8, ln_fusion=False)
        torch.cuda.synchronize()
        assert torch.equal(y1, y2), fp8


# ---------------------------------------------------------------- sublayer

def _sublayer_inputs(B, S, H, seed):
    W = H * 64
    x = dev16(oracle.normal_f16(seed, (B, S, W)))
    gamma = torch.ones(W, dtype=torch.float16, device=DEV)
    beta = torch.zeros(W, dtype=torch.float16, device=DEV)
    Wqkv = oracle.normal_f32(seed + 1, (3 * W, W), 0.02)
    q8, s8 = oracle.quantize_e4m3_rows(Wqkv)
    w_out = dev16(oracle.normal_f16(seed + 2, (W, W), 0.02))
    b_out = dev16(oracle.normal_f16(seed + 3, (W,), 0.02))
    return x, gamma, beta, torch.from_numpy(q8).to(DEV), torch.from_numpy(s8).to(DEV), w_out, b_out


def _torch_fp32_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H):
    table = torch.from_numpy(oracle.e4m3_table()).to(DEV)
    wq = table[q8.long()] * s8[:, None]
    xf = x.float()
    B, S, W = xf.shape
    n = torch.nn.functional.layer_norm(xf, (W,), gamma.float(), beta.float(), 1e-5)
    qkv = n @ wq.T
    q, k, v = (qkv[..., i * W:(i + 1) * W].reshape(B, S, H, 64).transpose(1, 2) for i in range(3))
    outs = []
    for h in range(H):
        p = torch.softmax(q[:, h] @ k[:, h].transpose(1, 2) / 8.0, dim=-1)
        outs.append(p @ v[:, h])
    attn = torch.stack(outs, 1).transpose(1, 2).reshape(B, S, W)
    return (xf + attn @ w_out.float().T + b_out.float()).cpu().numpy()


def _row_ranges(S):
    return [(0, S)] if S <= 512 else [(0, 32), (S // 2 - 16, S // 2 + 16), (S - 32, S)]


def _oracle_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H, r0, r1):
    """The oracle's block-order self half (src/unet.cpp:500-506) on the sublayer's inputs, with
    the fused [3W, W] E4M3 weight dequantised (decode x per-channel scale) and split into the
    reference's separate q, k, v weights."""
    W = H * 64
    wqkv = oracle.dequantize_e4m3_rows(q8.cpu().numpy(), s8.cpu().numpy())
    return oracle.attn_sublayer(host(x), host(gamma), host(beta), wqkv[:W], wqkv[W:2 * W], wqkv[2 * W:],
                                host(w_out), host(b_out), H, r0, r1, threads=THREADS)


def check_vs_oracle_sublayer(y, x, gamma, beta, q8, s8, w_out, b_out, H, label, max_abs=2e-3, mean_abs=2e-4):
    got = host(y)
    S = got.shape[1]
    for r0, r1 in _row_ranges(S):
        ref = _oracle_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H, r0, r1)
        assert_parity_f16_out(got[:, r0:r1], ref[:, r0:r1], max_abs, mean_abs, label=f"{label} oracle rows {r0}:{r1}")


@pytest.mark.parametrize("B,S,H", [(2, 4096, 10), (2, 1024, 20), (1, 300, 2)])
def test_sublayer_matches_composition_and_oracle(B, S, H):
    x, gamma, beta, q8, s8, w_out, b_out = _sublayer_inputs(B, S, H, 960 + S)
    W = H * 64
    print(f"sublayer B{B} S{S} H{H}", flush=True)
    y = sh.attn_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H)
    # composition of the individual calls
    n = sh.layer_norm(x, gamma, beta)
    qkv = sh.linear(n.view(-1, W), q8, w_scale=s8)
    qkv3 = qkv.view(B, S, 3 * W)
    attn = sh.attention(qkv3[..., :W], qkv3[..., W:2 * W], qkv3[..., 2 * W:], H)
    y2 = sh.linear(attn.view(-1, W), w_out, bias=b_out, residual=x.view(-1, W)).view(B, S, W)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
    check_vs_oracle_sublayer(y, x, gamma, beta, q8, s8, w_out, b_out, H, f"sublayer B{B} S{S}")
    ref = _torch_fp32_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H)
    assert_parity_f16_out(host(y), ref, label="sublayer vs torch fp32, all rows")
    # in place (y = x): the residual read precedes the write of every element
    xi = x.clone()
    sh.attn_sublayer(xi, gamma, beta, q8, s8, w_out, b_out, H, out=xi)
    torch.cuda.synchronize()
    assert torch.equal(xi, y)


# ---------------------------------------------------------------- FP8 activations (fp8 MFMA)
# LayerNorm emitting E4M3 codes with per-row scales, and the E4M3 x E4M3 linear on the fp8
# matrix cores. No counterpart in the reference (weight-only FP8 there); the oracle is the
# fp32 LayerNorm followed by the row quantiser's rule (the one pinned bit-exact above), and
# the fp64 product of the decoded operands.

def e4m3_half_step(v):
    """Half the E4M3 spacing at |v| (normal range 2^-6 .. 448: 3 mantissa bits; subnormal 2^-9)."""
    e = np.floor(np.log2(np.maximum(np.abs(v), 2.0 ** -6)))
    return 2.0 ** (e - 3) / 2


@pytest.mark.parametrize("rows,width", [(8192, 640), (77, 320), (5, 1280), (3, 2048), (4, 66), (77, 640),
                                        (19, 256)])
def test_layer_norm_e4m3(rows, width):
    xb = oracle.normal_f16(990 + width, (rows, width))
    gb = oracle.normal_f16(991, (width,), 0.5)
    bb = oracle.normal_f16(992, (width,), 0.5)
    if rows > 3:
        xb[3, :] = f16(np.float32([2.5]))[0]  # constant row: y = beta
    q, s = sh.layer_norm_e4m3(dev16(xb), dev16(gb), dev16(bb))
    torch.cuda.synchronize()
    y = oracle.layer_norm(oracle.f16_bits_to_f32(xb), oracle.f16_bits_to_f32(gb), oracle.f16_bits_to_f32(bb))
    q_ref, s_ref = oracle.quantize_e4m3_rows(y)
    s_got = s.cpu().numpy()
    np.testing.assert_allclose(s_got, s_ref, rtol=1e-5)
    got = oracle.e4m3_table()[q.cpu().numpy()] * s_got[:, None]
    err = np.abs(got.astype(np.float64) - y)
    # Half an E4M3 step; at a rounding tie the kernel's fp32 LayerNorm value (sums in another
    # order) may round to the neighbouring code: 5% of a half step covers those few.
    bound = e4m3_half_step(y / s_ref[:, None]) * s_ref[:, None] * 1.05 + 1e-6 * np.abs(y) + 1e-7
    print(f"LN e4m3 {rows}x{width}: max_abs={err.max():.3e}, codes equal to the oracle's: "
          f"{(q.cpu().numpy() == q_ref).mean():.5f}", flush=True)
    assert (err <= bound).all()
    assert (q.cpu().numpy() == q_ref).mean() >= 0.9999


@pytest.mark.parametrize("M,N,K,extras", [(2048, 3840, 1280, False), (2000, 3800, 1280, True)])
def test_linear_e4m3_wide_tiles(M, N, K, extras):
    """E4M3 weights below 4096 rows: 128 x 256 tiles of 8 waves (2 x 4) — the level-2 QKV
    projection, and a ragged shape (last row tile of 80, last column tile of 216) with bias and
    residual."""
    ab = oracle.normal_f16(1950 + M, (M, K))
    q, s = oracle.quantize_e4m3_rows(oracle.normal_f32(1951, (N, K), 0.02))
    bb = oracle.normal_f16(1952, (N,), 0.02) if extras else None
    rb = oracle.normal_f16(1953, (M, N)) if extras else None
    got = host(sh.linear(dev16(ab), torch.from_numpy(q).to(DEV), w_scale=torch.from_numpy(s).to(DEV),
                         bias=dev16(bb) if extras else None, residual=dev16(rb) if extras else None))
    rows = np.r_[0:256, M // 2:M // 2 + 32, M - 160:M]
    ref = _linear_ref(ab[rows], oracle.dequantize_e4m3_rows(q, s), bb, rb[rows] if extras else None)
    within_half_ulp(got[rows], ref, 1e-4, f"linear E4M3 {M}x{N}x{K} (128 x 256 tiles)")


@pytest.mark.parametrize("M,N,K,extras", [(8192, 1920, 640, False), (333, 640, 640, True), (129, 200, 64, True),
                                          (256, 1280, 1280, False), (2048, 3840, 1280, False),
                                          (2000, 3800, 1280, True)])
def test_linear_e4m3_activations(M, N, K, extras):
    af = oracle.normal_f32(1000 + M, (M, K))
    aq, a_s = oracle.quantize_e4m3_rows(af)
    wq, w_s = oracle.quantize_e4m3_rows(oracle.normal_f32(1001 + N, (N, K), 0.02))
    bb = oracle.normal_f16(1002, (N,), 0.02) if extras else None
    rb = oracle.normal_f16(1003, (M, N)) if extras else None
    t = lambda x: torch.from_numpy(x).to(DEV)
    got = host(sh.linear_e4m3(t(aq), t(a_s), t(wq), t(w_s), bias=dev16(bb) if extras else None,
                              residual=dev16(rb) if extras else None))
    rows = np.r_[0:256, M // 2:M // 2 + 32, M - 64:M] if M > 512 else np.arange(M)
    ref = oracle.dequantize_e4m3_rows(aq[rows], a_s[rows]).astype(np.float64) @ \
        oracle.dequantize_e4m3_rows(wq, w_s).astype(np.float64).T
    if extras:
        ref = ref + oracle.f16_bits_to_f32(bb)[None, :] + oracle.f16_bits_to_f32(rb)[rows]
    within_half_ulp(got[rows], ref, 1e-4, f"linear E4M3 x E4M3 {M}x{N}x{K}")


@pytest.mark.parametrize("B,S,H", [(2, 4096, 10), (2, 1024, 20), (1, 300, 2)])
def test_sublayer_fp8_activations(B, S, H):
    x, gamma, beta, q8, s8, w_out, b_out = _sublayer_inputs(B, S, H, 1010 + S)
    W = H * 64
    print(f"sublayer fp8 activations B{B} S{S} H{H}", flush=True)
    y = sh.attn_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H, fp8_activations=True)
    codes, cs = sh.layer_norm_e4m3(x, gamma, beta)
    qkv = sh.linear_e4m3(codes.view(-1, W), cs, q8, s8)
    qkv3 = qkv.view(B, S, 3 * W)
    attn = sh.attention(qkv3[..., :W], qkv3[..., W:2 * W], qkv3[..., 2 * W:], H)
    y2 = sh.linear(attn.view(-1, W), w_out, bias=b_out, residual=x.view(-1, W)).view(B, S, W)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
    # The E4M3 rounding of the LayerNorm output (3 mantissa bits; no reference counterpart: its
    # FP8 path is weight-only) enters q, k, v at about 2% relative and is damped by the softmax
    # averaging and the 0.02-scale output projection: bar 4e-3 beyond the output rounding and a
    # mean of 3e-4 up to width 640 against the oracle's unquantised activations, times W / 640 above:
    # the rounding reaches the output through two W-term sums (the q|k|v projection, then the
    # out-projection), measured 5.2e-4 at width 1280.
    check_vs_oracle_sublayer(y, x, gamma, beta, q8, s8, w_out, b_out, H, f"sublayer fp8 act B{B} S{S}",
                             max_abs=4e-3, mean_abs=3e-4 * max(1.0, W / 640))


# ---------------------------------------------------------------- cross-attention sublayer
# The transformer block's second half (src/cuda/unet.cpp:120-131): LN -> to_q -> attention against
# the context's K|V (projected once per request from encoder_hidden_states [B, 77, 2048]) ->
# to_out + bias + residual.

def _cross_inputs(B, S, H, seed, ctx_len=77, ctx_dim=2048, fp8=False):
    W = H * 64
    x = dev16(oracle.normal_f16(seed, (B, S, W)))
    gamma = dev16(oracle.normal_f16(seed + 1, (W,), 0.5))
    beta = dev16(oracle.normal_f16(seed + 2, (W,), 0.1))
    ctx = dev16(oracle.normal_f16(seed + 3, (B, ctx_len, ctx_dim)))
    w_kv = dev16(oracle.normal_f16(seed + 4, (2 * W, ctx_dim), 0.02))
    if fp8:
        q8, s8 = oracle.quantize_e4m3_rows(oracle.normal_f32(seed + 5, (W, W), 0.02))
        w_q, w_q_scale = torch.from_numpy(q8).to(DEV), torch.from_numpy(s8).to(DEV)
    else:
        w_q, w_q_scale = dev16(oracle.normal_f16(seed + 5, (W, W), 0.02)), None
    w_out = dev16(oracle.normal_f16(seed + 6, (W, W), 0.02))
    b_out = dev16(oracle.normal_f16(seed + 7, (W,), 0.02))
    return x, gamma, beta, ctx, w_kv, w_q, w_q_scale, w_out, b_out


def _torch_fp32_cross(x, gamma, beta, ctx, w_kv, w_q, w_q_scale, w_out, b_out, H):
    if w_q.dtype == torch.uint8:
        wq = torch.from_numpy(oracle.e4m3_table()).to(DEV)[w_q.long()] * w_q_scale[:, None]
    else:
        wq = w_q.float()
    xf = x.float()
    B, S, W = xf.shape
    n = torch.nn.functional.layer_norm(xf, (W,), gamma.float(), beta.float(), 1e-5)
    q = (n @ wq.T).reshape(B, S, H, 64).transpose(1, 2)
    kv = ctx.float() @ w_kv.float().T
    k = kv[..., :W].reshape(B, -1, H, 64).transpose(1, 2)
    v = kv[..., W:].reshape(B, -1, H, 64).transpose(1, 2)
    p = torch.softmax(q @ k.transpose(-1, -2) / 8.0, dim=-1)
    attn = (p @ v).transpose(1, 2).reshape(B, S, W)
    return (xf + attn @ w_out.float().T + b_out.float()).cpu().numpy()


# The library's backend choice (AUTO) runs the query projection and the attention as one launch
# when seq % 64 == 0, W % 128 == 0, 65 <= ctx_len <= 80 and the grid of 64 x 128 tiles is
# resident at once (three per CU with E4M3 weights and fp16 activations, else two) and the
# attention has more than 1.5 32-row query blocks per CU (fewer run on 16-row blocks); each wave
# attends with the 32 x 64 query block it projected, and the output equals the composition of the
# individual calls bit for bit. Other shapes, and explicit backends, run the composition itself.
@pytest.mark.parametrize("B,S,H,fp8,w8,ctx_len", [
    (2, 1024, 20, False, False, 77),  # level 2, fused, fp16 weights
    (2, 1024, 20, True, True, 77),    # level 2, fused, E4M3 weights and activations
    (2, 4096, 10, False, True, 77),   # level 1, fused (640 tiles, three per CU), E4M3 weights
    (2, 4096, 10, True, True, 77),    # level 1, E4M3 activations: 640 tiles > two per CU, composition
    (1, 4096, 4, False, True, 65),    # fused, one key in the last group
    (1, 4160, 4, False, False, 80),   # fused, 16 keys in the last group
    (1, 128, 2, False, True, 65),     # few query blocks: the attention takes 16-row blocks, composition
    (1, 300, 2, False, False, 77),    # S % 64 != 0: composition
    (1, 256, 2, False, False, 64),    # 64 keys: composition
])
def test_cross_sublayer_matches_composition_and_fp32(B, S, H, fp8, w8, ctx_len):
    x, gamma, beta, ctx, w_kv, w_q, w_q_scale, w_out, b_out = _cross_inputs(B, S, H, 1100 + S, ctx_len=ctx_len,
                                                                            fp8=w8)
    W = H * 64
    print(f"cross sublayer B{B} S{S} H{H} fp8={fp8} w8={w8} ctx{ctx_len}", flush=True)
    kv = sh.project_context_kv(ctx, w_kv)
    y = sh.cross_attn_sublayer(x, gamma, beta, w_q, w_q_scale, kv, w_out, b_out, H, fp8_activations=fp8)
    y_flash = sh.cross_attn_sublayer(x, gamma, beta, w_q, w_q_scale, kv, w_out, b_out, H, fp8_activations=fp8,
                                     backend=sh.FLASH_SM80)  # explicit backend: the composition
    # composition of the individual calls
    if fp8:
        codes, cs = sh.layer_norm_e4m3(x, gamma, beta)
        q = sh.linear_e4m3(codes.view(-1, W), cs, w_q, w_q_scale)
    else:
        q = sh.linear(sh.layer_norm(x, gamma, beta).view(-1, W), w_q, w_scale=w_q_scale)
    attn = sh.attention(q.view(B, S, W), kv[..., :W], kv[..., W:], H)
    y2 = sh.linear(attn.view(-1, W), w_out, bias=b_out, residual=x.view(-1, W)).view(B, S, W)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
    assert torch.equal(y_flash, y2)
    # oracle: the reference's block order (src/unet.cpp:508-512) with the context projected in
    # fp32; fp8 activations (E4M3 LayerNorm output, no reference counterpart) get 4e-3 max-abs and
    # a mean-abs bar of 5e-4 up to width 640, growing as sqrt(W / 640) above: the activations' 3-bit
    # mantissa rounding accumulates over the W terms of each projected value
    mean_fp8 = 5e-4 * max(1.0, W / 640) ** 0.5
    wq = oracle.dequantize_e4m3_rows(w_q.cpu().numpy(), w_q_scale.cpu().numpy()) if w8 else host(w_q)
    wkv = host(w_kv)
    got = host(y)
    for r0, r1 in _row_ranges(S):
        ref = oracle.cross_attn_sublayer(host(x), host(gamma), host(beta), wq, host(ctx), wkv[:W], wkv[W:],
                                         host(w_out), host(b_out), H, r0, r1, threads=THREADS)
        assert_parity_f16_out(got[:, r0:r1], ref[:, r0:r1], 4e-3 if fp8 else 2e-3, mean_fp8 if fp8 else 2e-4,
                              label=f"cross sublayer B{B} S{S} oracle rows {r0}:{r1}")
    ref = _torch_fp32_cross(x, gamma, beta, ctx, w_kv, w_q, w_q_scale, w_out, b_out, H)
    assert_parity_f16_out(got, ref, 4e-3 if fp8 else 2e-3, mean_fp8 if fp8 else 2e-4,
                          label="cross sublayer vs torch fp32, all rows")
    xi = x.clone()  # in place
    sh.cross_attn_sublayer(xi, gamma, beta, w_q, w_q_scale, kv, w_out, b_out, H, out=xi, fp8_activations=fp8)
    torch.cuda.synchronize()
    assert torch.equal(xi, y)


# ---------------------------------------------------------------- random shapes
# Seeded random calls of the projection (fp16 or E4M3 weights; bias, residual), the LayerNorm and
# the LayerNorm inside the E4M3 projection (fp16 or E4M3 activations), each checked elementwise
# against torch fp32 on the same device values (E4M3 codes decoded by torch's float8_e4m3fn):
# one fp16 ulp at |ref| plus the accumulation's rounding (2^-16 of sum |a||w|; for the LayerNorm
# projection the normalised rows' fp16 rounding, 2^-10 of sum |ln||w|, or their E4M3 rounding,
# 2^-4), and the fused forms bit-equal to their two-launch compositions.

@pytest.mark.parametrize("seed", range(3))
def test_random_projection_and_layer_norm_shapes(seed):
    import random
    rng = random.Random(2000 + seed)
    for n in range(40):
        kind = rng.choice(["lin16", "lin16ks", "lin8", "ln", "lnlin", "lnlin8"])
        M = rng.choice([rng.randint(1, 300), rng.randint(1, 5000)])
        g = torch.Generator(device="cuda").manual_seed(seed * 1000 + n)
        if kind in ("lin16", "lin16ks", "lin8"):
            K, N = 64 * rng.randint(1, 24), 4 * rng.randint(1, 768)
            if kind == "lin16ks":  # shapes of the K-split form on 256 CUs: 232-256 tiles of 64 x 160, a residual
                M, N = rng.randint(1793, 2048), 8 * rng.randint(141, 160)
            a = torch.randn(M, K, device="cuda", generator=g).half()
            w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).half()
            bias = torch.randn(N, device="cuda", generator=g).half() if rng.random() < 0.5 else None
            res = (torch.randn(M, N, device="cuda", generator=g).half()
                   if kind == "lin16ks" or rng.random() < 0.5 else None)
            label = f"{kind} M{M} N{N} K{K} bias={bias is not None} residual={res is not None}"
            print(label, flush=True)
            if kind == "lin8":
                wq, ws = sh.quantize_e4m3_rows(w)
                wf = wq.view(torch.float8_e4m3fn).float() * ws[:, None]
                got = sh.linear(a, wq, w_scale=ws, bias=bias, residual=res)
            else:
                wf = w.float()
                got = sh.linear(a, w, bias=bias, residual=res)
            ref = a.float() @ wf.T
            if bias is not None:
                ref = ref + bias.float()
            if res is not None:
                ref = ref + res.float()
            bound = 2.0 ** -10 * ref.abs() + 2.0 ** -16 * (a.float().abs() @ wf.abs().T) + 1e-5
        elif kind == "ln":
            W = 2 * rng.randint(1, 1024)
            x = (torch.randn(M, W, device="cuda", generator=g) * rng.choice([1, 5]) + rng.choice([0, 3])).half()
            gm = torch.randn(W, device="cuda", generator=g).half()
            bt = torch.randn(W, device="cuda", generator=g).half()
            label = f"ln M{M} W{W}"
            print(label, flush=True)
            got = sh.layer_norm(x, gm, bt)
            ref = torch.nn.functional.layer_norm(x.float(), (W,), gm.float(), bt.float(), 1e-5)
            bound = 2.0 ** -10 * ref.abs() + 2e-3 * gm.float().abs() + 1e-4
        else:
            K, N = rng.choice([640, 1280]), 128 * rng.randint(1, 16)
            x = torch.randn(M, K, device="cuda", generator=g).half()
            gm = (1 + 0.1 * torch.randn(K, device="cuda", generator=g)).half()
            bt = (0.1 * torch.randn(K, device="cuda", generator=g)).half()
            wq, ws = sh.quantize_e4m3_rows((torch.randn(N, K, device="cuda", generator=g) * 0.05).half())
            bias = torch.randn(N, device="cuda", generator=g).half() if rng.random() < 0.5 else None
            fp8 = kind == "lnlin8"
            label = f"{kind} M{M} N{N} K{K} bias={bias is not None}"
            print(label, flush=True)
            got = sh.layer_norm_linear(x, gm, bt, wq, ws, bias=bias, fp8_activations=fp8)
            if fp8:
                codes, cs = sh.layer_norm_e4m3(x, gm, bt)
                comp = sh.linear_e4m3(codes, cs, wq, ws, bias=bias)
            else:
                comp = sh.linear(sh.layer_norm(x, gm, bt), wq, w_scale=ws, bias=bias)
            torch.cuda.synchronize()
            assert torch.equal(got, comp), label
            ln = torch.nn.functional.layer_norm(x.float(), (K,), gm.float(), bt.float(), 1e-5)
            wf = wq.view(torch.float8_e4m3fn).float() * ws[:, None]
            ref = ln @ wf.T + (bias.float() if bias is not None else 0.0)
            bound = 2.0 ** -10 * ref.abs() + (2.0 ** -4 if fp8 else 2.0 ** -10) * (ln.abs() @ wf.abs().T) + 1e-4
        torch.cuda.synchronize()
        assert bool(torch.isfinite(got.float()).all()), label
        excess = float(((got.float() - ref).abs() - bound).max())
        assert excess <= 0.0, (label, excess)


@pytest.mark.parametrize("seed", range(2))
def test_random_sublayers_equal_their_compositions(seed):
    """Seeded random self- and cross-attention sublayers (fp16 or E4M3 weights, fp16 or E4M3
    activations, LayerNorm fusion on or off, 1-128 context tokens, ragged sequence lengths): the one
    call equals the composition of the individual calls bit for bit, whichever fused forms the
    library picks."""
    import random
    rng = random.Random(3000 + seed)
    done = 0
    while done < 25:
        cross = rng.random() < 0.5
        B, H = rng.randint(1, 2), rng.choice([1, 2, 4, 5, 10, 20])
        W = 64 * H
        S = rng.choice([rng.randint(1, 300), rng.randint(1, 4096), 64 * rng.randint(1, 64)])
        if B * S * W > 12e6:
            continue
        w8 = rng.random() < 0.7
        fp8 = w8 and rng.random() < 0.4
        g = torch.Generator(device="cuda").manual_seed(seed * 1000 + done)
        x = torch.randn(B, S, W, device="cuda", generator=g).half()
        gm = (1 + 0.1 * torch.randn(W, device="cuda", generator=g)).half()
        bt = (0.1 * torch.randn(W, device="cuda", generator=g)).half()
        w_out = (torch.randn(W, W, device="cuda", generator=g) * 0.02).half()
        b_out = (torch.randn(W, device="cuda", generator=g) * 0.02).half()
        n_in = W if cross else 3 * W
        w_in = (torch.randn(n_in, W, device="cuda", generator=g) * 0.02).half()
        wq, ws = sh.quantize_e4m3_rows(w_in) if w8 else (w_in, None)
        if cross:
            L, C = rng.randint(1, 128), rng.choice([768, 1280, 2048])
            ctx = torch.randn(B, L, C, device="cuda", generator=g).half()
            kv = sh.project_context_kv(ctx, (torch.randn(2 * W, C, device="cuda", generator=g) * 0.02).half())
            label = f"cross B{B} S{S} H{H} L{L} w8={w8} fp8={fp8}"
            print(label, flush=True)
            y = sh.cross_attn_sublayer(x, gm, bt, wq, ws, kv, w_out, b_out, H, fp8_activations=fp8)
        else:
            lnf = rng.random() < 0.5
            label = f"self B{B} S{S} H{H} w8={w8} fp8={fp8} ln_fusion={lnf}"
            print(label, flush=True)
            y = sh.attn_sublayer(x, gm, bt, wq, ws, w_out, b_out, H, fp8_activations=fp8, ln_fusion=lnf)
        if fp8:
            codes, cs = sh.layer_norm_e4m3(x, gm, bt)
            proj = sh.linear_e4m3(codes.view(-1, W), cs, wq, ws)
        else:
            proj = sh.linear(sh.layer_norm(x, gm, bt).view(-1, W), wq, w_scale=ws)
        if cross:
            attn = sh.attention(proj.view(B, S, W), kv[..., :W], kv[..., W:], H)
        else:
            qkv = proj.view(B, S, 3 * W)
            attn = sh.attention(qkv[..., :W], qkv[..., W:2 * W], qkv[..., 2 * W:], H)
        y2 = sh.linear(attn.view(-1, W), w_out, bias=b_out, residual=x.view(-1, W)).view(B, S, W)
        torch.cuda.synchronize()
        assert torch.equal(y, y2), label
        done += 1


def test_level2_sublayers_hip_graph_replays():
    """The level-2 self and cross sublayer calls (LayerNorm, projections incl. the K-split
    out-projection, attention) captured in one HIP graph: no allocation or memset inside the
    calls; four replays with unrelated eager work between them each equal the eager results."""
    B, S, H = 2, 1024, 20
    x, gamma, beta, q8, s8, w_out, b_out = _sublayer_inputs(B, S, H, 1500)
    cx, cg, cb, ctx, w_kv, w_q, w_q_scale, cw_out, cb_out = _cross_inputs(B, S, H, 1600)
    kv = sh.project_context_kv(ctx, w_kv)
    y_self, y_cross = torch.empty_like(x), torch.empty_like(cx)
    ws_self = torch.empty(1 << 26, dtype=torch.uint8, device=DEV)
    ws_cross = torch.empty(1 << 26, dtype=torch.uint8, device=DEV)

    def calls():
        sh.attn_sublayer(x, gamma, beta, q8, s8, w_out, b_out, H, out=y_self, workspace=ws_self)
        sh.cross_attn_sublayer(cx, cg, cb, w_q, w_q_scale, kv, cw_out, cb_out, H, out=y_cross, workspace=ws_cross)

    calls()
    torch.cuda.synchronize()
    eager_self, eager_cross = y_self.clone(), y_cross.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        calls()  # warm-up on the capture stream
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        calls()
    for i in range(4):
        y_self.fill_(float("nan"))
        y_cross.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y_self, eager_self), i
        assert torch.equal(y_cross, eager_cross), i
        _ = (x.float() * 2).sum().item()  # unrelated eager work between replays
