"""The tiled kernel of the online family (head_dim <= 160, every dtype) against 64-bit attention and
the per-row kernel: edges of its key sub-tiles, query blocks and padded head dimensions, its three
workgroup forms, masks, causal limits, unaligned rows, and values its 16-bit planes cannot carry."""
import pytest

import sdxl_hip as sh

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# Half a unit of the output's last place, relative (none for FP32 beyond the absolute bound).
OUT_ROUNDING = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}
# Scores: sums of D <= 160 products of N(0,1) values, |score| < 8 after scaling, each within
# sqrt(160) * 2^-24 * 8 < 1e-5 of the exact one; probabilities move by that relative error and the
# output by its share of max |v| < 5, less the averaging over keys.
ABS = 2e-5


def tensors(seed, B, H, Sq, Sk, D, dtype):
    g = torch.Generator(device=DEV).manual_seed(seed)
    make = lambda s: torch.randn(B, s, H * D, device=DEV, generator=g).to(DTYPES[dtype])
    return make(Sq), make(Sk), make(Sk)


def reference(q, k, v, H, causal=False, key_mask=None):
    B, Sq, W = q.shape
    Sk, D = k.shape[1], W // H
    out = torch.zeros(B, Sq, W, dtype=torch.float64, device=DEV)
    for b in range(B):
        for h in range(H):
            c = slice(h * D, (h + 1) * D)
            s = q[b, :, c].double() @ k[b, :, c].double().t() / D ** 0.5
            if key_mask is not None:
                s.masked_fill_(key_mask[b][None] == 0, float("-inf"))
            if causal:
                s.masked_fill_(torch.ones(Sq, Sk, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
            out[b, :, c] = torch.nan_to_num(torch.softmax(s, -1)) @ v[b, :, c].double()
    return out


def check(got, ref, dtype):
    err = (got.double() - ref).abs() - OUT_ROUNDING[dtype] * ref.abs()
    assert err.max().item() <= ABS, err.max().item()


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("B,H,Sq,Sk,D", [
    (1, 1, 1, 1, 8), (2, 3, 31, 33, 16), (1, 2, 65, 64, 32), (1, 2, 129, 65, 40),
    (1, 3, 64, 127, 64), (2, 2, 63, 128, 72), (1, 2, 130, 129, 96), (1, 2, 33, 200, 128),
    (1, 2, 70, 31, 136), (2, 1, 97, 300, 160),
    (1, 3, 50, 77, 7), (1, 2, 66, 90, 33), (2, 2, 40, 70, 50), (1, 2, 35, 100, 159),  # rows not 16-byte aligned
    (2, 40, 1000, 70, 40), (1, 20, 900, 260, 64), (1, 33, 1000, 150, 56)])  # one and two key groups on full grids
def test_tiled_shapes(B, H, Sq, Sk, D, dtype):
    if dtype != "f32" and D == 64:
        D = 56  # 16-bit head_dim 64 runs elsewhere
    q, k, v = tensors(B + Sq + D, B, H, Sq, Sk, D, dtype)
    for causal in (False, True):
        check(sh.attention(q, k, v, H, causal=causal), reference(q, k, v, H, causal), dtype)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("causal", [False, True])
def test_tiled_key_mask(dtype, causal):
    B, H, Sq, Sk, D = 3, 2, 150, 170, 80
    q, k, v = tensors(5, B, H, Sq, Sk, D, dtype)
    g = torch.Generator(device=DEV).manual_seed(6)
    mask = (torch.rand(B, Sk, device=DEV, generator=g) < 0.6).int()
    mask[0, :100] = 0  # whole sub-tiles hidden, and with causal whole rows
    mask[1] = 0        # nothing visible: zeros
    got = sh.attention(q, k, v, H, causal=causal, key_mask=mask)
    check(got, reference(q, k, v, H, causal, mask), dtype)
    assert (got[1] == 0).all()


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_tiled_unaligned_and_strided_rows(dtype):
    """head_dim 64 and 48 as slices of wider rows, aligned and off by one element."""
    for D, offset in ((64 if dtype == "f32" else 48, 8), (48, 1), (64, 3)):
        B, H, S = 2, 3, 75
        wide = torch.randn(B, S, 3 * H * D + 17, device=DEV, generator=torch.Generator(device=DEV).manual_seed(D)).to(DTYPES[dtype])
        q, k, v = (wide[..., offset + i * H * D: offset + (i + 1) * H * D] for i in range(3))
        check(sh.attention(q, k, v, H), reference(q, k, v, H), dtype)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.3e38, 3.402e38])
def test_tiled_values_planes_cannot_carry(dtype, where, value):
    """Infinities, NaN and FP32 values above the largest bf16 give what the per-row kernel gives."""
    B, H, Sq, Sk, D = 1, 2, 70, 100, 72
    q, k, v = tensors(9, B, H, Sq, Sk, D, dtype)
    {"q": q, "k": k, "v": v}[where][0, 57, D + 3] = value
    got = sh.attention(q, k, v, H).float()
    ref = sh.attention(q, k, v, H, backend=sh.WARP_ONLINE).float()
    torch.testing.assert_close(got, ref, rtol=2.0 ** -7 if dtype == "bf16" else 2e-3, atol=1e-3, equal_nan=True)


@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.402e38])
@pytest.mark.parametrize("dim", [3, 300])  # either half of the output's dims
def test_d512_values_planes_cannot_carry(where, value, dim):
    S = 70
    q, k, v = tensors(17, 1, 1, S, 100, 512, "f32")
    {"q": q, "k": k, "v": v}[where][0, 57, dim] = value
    got = sh.attention(q, k, v, 1)
    ref = sh.attention(q, k, v, 1, backend=sh.WARP_ONLINE)
    if where == "q" and value != value:
        assert got[0, 57].isnan().all()  # the per-row kernel takes such a row's keys for hidden
        got[0, 57] = ref[0, 57]
    torch.testing.assert_close(got, ref, rtol=2e-3, atol=1e-3, equal_nan=True)


@pytest.mark.parametrize("B,H,Sq,Sk", [
    (1, 1, 33, 1), (1, 2, 64, 31), (2, 1, 100, 32), (1, 1, 130, 33), (1, 1, 65, 64), (1, 1, 1, 65), (1, 2, 40, 97),
    (1, 9, 950, 70),   # 270 blocks of 32 queries on 256 CUs: 64 queries per workgroup
    (1, 6, 1000, 70)])  # 192: 32 queries, all output dims
def test_d512_blocks(B, H, Sq, Sk):
    q, k, v = tensors(Sq + Sk, B, H, Sq, Sk, 512, "f32")
    check(sh.attention(q, k, v, H), reference(q, k, v, H), "f32")


def test_tiled_large_logits():
    """Logits of a few hundred, rising along the keys: the running maximum moves in every sub-tile."""
    B, H, S, D = 1, 2, 300, 64
    q, k, v = tensors(11, B, H, S, S, D, "f32")
    q = q * 16
    k = k * torch.linspace(1, 6, S, device=DEV)[None, :, None]
    # a score error of 2^-24 * 160 * |score| (< 600) moves a probability by up to 6e-3 at worst;
    # sums of rounding errors are far smaller: sqrt(64) * 2^-24 * 600 * max |v|
    err = (sh.attention(q, k, v, H).double() - reference(q, k, v, H)).abs().max().item()
    assert err <= 8 * 2.0 ** -24 * 600 * 5, err


@pytest.mark.parametrize("D", [160, 161])
def test_tiled_limit_of_the_head_dimension(D):
    q, k, v = tensors(13, 1, 2, 40, 50, D, "f32")
    check(sh.attention(q, k, v, 2), reference(q, k, v, 2), "f32")


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [
    (1, 2, 70, 70, 40, True), (1, 1, 131, 131, 160, True), (2, 3, 90, 200, 33, True), (2, 2, 100, 100, 7, False),
    (2, 40, 1000, 70, 40, False), (1, 33, 1000, 150, 56, True)])  # one and two key groups on full grids
def test_tiled_special_values_reach_their_rows_alone(B, H, Sq, Sk, D, causal, where, value, dtype):
    """Rows that a causal limit keeps away from an infinity or a NaN stay finite; every other row as on
    the per-row kernel, on each workgroup form, also with rows left over from the groups that start over."""
    q, k, v = tensors(Sq + D, B, H, Sq, Sk, D, dtype)
    at = 37
    {"q": q, "k": k, "v": v}[where][0, at, D + 3 if H > 1 else 3] = value
    got = sh.attention(q, k, v, H, causal=causal).float()
    ref = sh.attention(q, k, v, H, causal=causal, backend=sh.WARP_ONLINE).float()
    torch.testing.assert_close(got, ref, rtol=2.0 ** -7 if dtype == "bf16" else 2e-3, atol=1e-3, equal_nan=True)
    if causal and where != "q":
        assert got[0, :at].isfinite().all()


@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 9, 950, 70), (1, 6, 1000, 70), (1, 1, 70, 300), (1, 9, 950, 32)])
@pytest.mark.parametrize("where", ["q", "k", "v", "all"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.402e38])
def test_d512_special_values_on_every_form(B, H, Sq, Sk, where, value):
    """As test_d512_values_planes_cannot_carry, on 64 queries per workgroup, on 32 with all output dims,
    and on two workgroups per query block; and with every query of a block of rows special."""
    q, k, v = tensors(Sq + Sk, B, H, Sq, Sk, 512, "f32")
    h = H - 1
    if where == "all":
        q[0, :64, 512 * h + 5] = value
        rows = range(0, 64)
    else:
        {"q": q, "k": k, "v": v}[where][0, 27, 512 * h + 300] = value
        rows = [27] if where == "q" else []
    got = sh.attention(q, k, v, H)
    ref = sh.attention(q, k, v, H, backend=sh.WARP_ONLINE)
    if value != value:
        for r in rows:  # the per-row kernel takes such a row's keys for hidden
            assert got[0, r, 512 * h:].isnan().all()
            got[0, r, 512 * h:] = ref[0, r, 512 * h:]
    torch.testing.assert_close(got, ref, rtol=2e-3, atol=1e-3, equal_nan=True)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("D", [80, 33])
def test_tiled_small_probabilities_keep_their_bits(D, dtype):
    """Two visible keys, one of weight ~1 with V = 0, one of weight exp(-a), a = 11 .. 24, with the largest
    fp16 value: the output shows the small weight's own accuracy. fp16 planes hold it within 2^-40 of the
    largest weight."""
    B, H, S = 1, 2, 96
    q, k, v = (torch.zeros(B, S, H * D, device=DEV, dtype=DTYPES[dtype]) for _ in range(3))
    q[..., ::D] = torch.linspace(11, 24, S, device=DEV).to(DTYPES[dtype])[None, :, None]
    k[..., ::D] = -60
    k[:, 0, ::D] = 0
    k[:, 5, ::D] = -1  # in the first key's sub-tile, so under its maximum
    v[:, 5] = 65504 if dtype == "f16" else 65280
    got = sh.attention(q, k, v, H, scale=1.0).double()
    w = torch.exp(-q[..., ::D].double()).repeat_interleave(D, dim=-1)
    ref = w / (1 + w) * v[0, 5, 0].double()
    # a fp32 argument of exp2 up to 35 moves the weight by 35 ln 2 * 2^-24 < 2^-18
    bound = ref * (OUT_ROUNDING[dtype] + 2.0 ** -18) + (2.0 ** -25 + 2.0 ** -24 if dtype == "f16" else 0)
    worst = ((got - ref).abs() / bound).max().item()
    assert worst <= 1, worst


@pytest.mark.parametrize("D,H,S", [(64, 2, 100), (72, 40, 300), (33, 2, 70), (512, 1, 100), (512, 9, 950)])
@pytest.mark.parametrize("small", ["v", "q", "k", "weights", "one q", "part of v"])
def test_small_fp32_values_keep_their_bits(D, H, S, small):
    """FP32 values below 2^-110, whose third bf16 plane would fall under bf16's range, count in full: V
    alone, Q or K against values that bring the scores back to the ordinary, weights below 2^-110 whose V
    does, one Q value of a row, and a column of V."""
    keys = 90
    q, k, v = tensors(S + D, 1, H, S, keys, D, "f32")
    tiny, huge = 2.0 ** -118, 2.0 ** 118
    if small == "v":
        v = v * tiny
    elif small == "q":
        q, k = q * tiny, k * huge
    elif small == "k":
        q, k = q * huge, k * tiny
    elif small == "one q":
        q[0, 3, 1], k[0, :, 1] = 2.0 ** -123 / 3, k[0, :, 1] * 2.0 ** 123
        q[0, :3, 1] = q[0, 4:, 1] = 0
    elif small == "part of v":
        v[..., 2] *= tiny
    else:  # one key far above the rest, whose V is zero
        q, k = torch.zeros_like(q), torch.zeros_like(k)
        q[..., ::D] = torch.linspace(84, 86, S, device=DEV)[None, :, None] * D ** 0.5
        k[..., ::D] = -1
        k[:, 7, ::D] = 0
        v = v * 2.0 ** 100
        v[:, 7] = v[:, 32:] = 0
    got, ref = sh.attention(q, k, v, H).double(), reference(q, k, v, H)
    err = (got - ref).abs()
    if small == "part of v":  # column by column: a tiny column must be right beside ordinary ones
        cols = torch.zeros_like(err, dtype=torch.bool)
        cols[..., 2] = True
        worst = max((err[cols].norm() / ref[cols].norm()).item(), (err[~cols].norm() / ref[~cols].norm()).item())
    else:
        rows = slice(3, 4) if small == "one q" else slice(None)
        worst = (err[:, rows].norm() / ref[:, rows].norm()).item()
    # fp32 sums: a few 1e-7; a fp32 argument of exp2 near 120 moves a weight by up to 2^-17
    assert worst <= (2.0 ** -17 if small == "weights" else 2e-6), worst


@pytest.mark.parametrize("B,D,backend", [(2 ** 19 + 8, 8, sh.AUTO),           # tiled or per-row: 2^24 + 256 pairs
                                         (2 ** 21 + 4, 8, sh.WARP_ONLINE),    # per-row: 2^26 + 128
                                         (2 ** 19 + 8, 64, sh.AUTO)])         # 16-bit head_dim 64
def test_more_pairs_than_one_grid_holds(B, D, backend):
    """More single-row (batch, head) pairs than one launch of the kernel takes. One visible key: the output
    is V, where a key mask leaves it."""
    H = 32
    q = torch.ones(B, 1, H * D, device=DEV, dtype=torch.float16)
    v = torch.randn(B, 1, H * D, device=DEV, dtype=torch.float16)
    got = torch.full_like(v, float("nan"))
    sh.attention(q, q, v, H, backend=backend, out=got)
    assert torch.equal(got, v)
    mask = torch.ones(B, 1, dtype=torch.int32, device=DEV)
    mask[-1] = mask[1] = 0
    v[-1] = v[1] = 0
    assert torch.equal(sh.attention(q, q, v, H, key_mask=mask, backend=backend), v)


@pytest.mark.parametrize("dtype,B,H,Sq,Sk,D", [
    ("f32", 256, 8, 1, 84, 40), ("f32", 128, 16, 4, 16, 160), ("f32", 1, 8, 3, 4, 80), ("f32", 32, 64, 1, 1, 7),
    ("f16", 256, 8, 1, 34, 80), ("bf16", 256, 8, 4, 4, 40)])
def test_few_queries_and_keys_on_the_per_row_kernel(dtype, B, H, Sq, Sk, D):
    """Calls on whose tiles most queries would be missing take the per-row kernel: its results, bit for bit,
    with a key mask and a causal limit too."""
    q, k, v = tensors(Sk, B, H, Sq, Sk, D, dtype)
    mask = (torch.rand(B, Sk, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3)) < 0.7).int()
    for causal in (False, True):
        for key_mask in (None, mask):
            assert torch.equal(sh.attention(q, k, v, H, causal=causal, key_mask=key_mask),
                               sh.attention(q, k, v, H, causal=causal, key_mask=key_mask, backend=sh.WARP_ONLINE))


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("D", [80, 128, 160, 90, 127])  # aligned rows, and rows that are not at padded 96 and 128
def test_tiled_two_key_groups(D, dtype):
    """512 blocks of 32 queries: two key groups at every padded head dimension above 64, in 16 bits too."""
    q, k, v = tensors(D, 2, 8, 1000, 150, D, dtype)
    for causal in (False, True):
        check(sh.attention(q, k, v, 8, causal=causal), reference(q, k, v, 8, causal), dtype)


@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 9, 950, 32), (1, 9, 950, 33), (1, 9, 950, 64), (1, 6, 1000, 31)])
def test_d512_few_key_blocks(B, H, Sq, Sk):
    """64 queries per workgroup with one key block, one and a bit, and two; 32 queries with less than one."""
    q, k, v = tensors(Sq + Sk, B, H, Sq, Sk, 512, "f32")
    check(sh.attention(q, k, v, H), reference(q, k, v, H), "f32")


@pytest.mark.parametrize("H,Sq,Sk,D", [(1, 70, 45, 512), (9, 950, 45, 512), (6, 1000, 70, 512), (1, 40, 31, 512),
                                       (2, 100, 77, 64), (8, 2000, 150, 80), (2, 70, 45, 33)])
def test_rows_past_the_keys_are_not_read_into_the_result(H, Sq, Sk, D):
    """K and V are the leading rows of longer buffers whose next rows are NaN."""
    q, k, v = tensors(Sq + Sk, 1, H, Sq, Sk + 64, D, "f32")
    k[:, Sk:] = v[:, Sk:] = float("nan")
    k, v = k[:, :Sk], v[:, :Sk]
    check(sh.attention(q, k, v, H), reference(q, k, v, H), "f32")
