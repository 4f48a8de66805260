"""Ragged and masked 16-bit head_dim-64 calls on every workgroup kind, against 64-bit attention: key
counts around the edges of the last stage, query counts that leave half a unit empty, key masks with
hidden ends, and the anchor update in the groups that ragged calls branch around."""
import pytest

import sdxl_hip as sh

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
# Rounding of the probabilities and of the output (unit roundoff 2^-11, 2^-8): |error| <= 2 u sum_j
# p_j |v_j| <= 2 u max |v| at worst, far less where the probabilities spread; max |v| < 5.5.
UNIT = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def tensors(seed, B, H, Sq, Sk, dtype, q_scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    make = lambda s, c=1.0: (torch.randn(B, s, H * 64, device=DEV, generator=g) * c).to(DTYPES[dtype])
    return make(Sq, q_scale), make(Sk), make(Sk)


def check(q, k, v, H, dtype, causal=False, key_mask=None, rows=None):
    got = sh.attention(q, k, v, H, causal=causal, key_mask=key_mask)
    B, Sq, _ = q.shape
    Sk = k.shape[1]
    worst = 0.0
    for b in range(B):
        for h in range(H):
            c = slice(h * 64, (h + 1) * 64)
            s = q[b, :, c].double() @ k[b, :, c].double().t() / 8
            if key_mask is not None:
                s.masked_fill_(key_mask[b][None] == 0, float("-inf"))
            if causal:
                s.masked_fill_(torch.ones(Sq, Sk, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
            p = torch.nan_to_num(torch.softmax(s, -1))
            ref = p @ v[b, :, c].double()
            bound = 2 * UNIT[dtype] * (p @ v[b, :, c].double().abs()) + 1e-6
            worst = max(worst, ((got[b, :, c].double() - ref).abs() / bound).max().item())
    assert worst <= 1.0, worst
    return got


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("B,H,Sq,Sk", [
    # key-split workgroups on the 64-KiB kernel, alone and beside whole ones
    (1, 2, 450, 449), (1, 2, 512, 511), (1, 3, 321, 480), (1, 2, 640, 545), (1, 2, 200, 576), (2, 20, 988, 988),
    # ... on the 32-KiB kernel (three workgroups per CU)
    (1, 75, 700, 450), (1, 75, 700, 481), (1, 75, 700, 512),
    # mixed workgroups within one head (blocks a multiple of 10 per head) and across two
    (2, 16, 2560, 129), (4, 8, 2559, 191), (2, 10, 4090, 160), (4, 20, 930, 223), (4, 20, 930, 1000),
    # whole workgroups
    (2, 20, 300, 300), (1, 2, 130, 129)])
def test_ragged(B, H, Sq, Sk, dtype):
    check(*tensors(Sq + Sk, B, H, Sq, Sk, dtype), H, dtype)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Sq,Sk", [
    (2, 3, 150, 170), (3, 2, 333, 500), (2, 2, 700, 300), (1, 5, 257, 1025),
    (2, 256, 200, 190)])  # whole workgroups: more units than key-split ones are used for
def test_masked(B, H, Sq, Sk, causal, dtype):
    q, k, v = tensors(Sq + Sk, B, H, Sq, Sk, dtype)
    g = torch.Generator(device=DEV).manual_seed(1)
    if causal:
        check(q, k, v, H, dtype, causal=True)
    kept = torch.zeros(B, Sk, dtype=torch.int32, device=DEV)
    kept[0, 40: Sk - 70] = 1                                  # hidden at both ends
    if B > 1:
        kept[1] = (torch.rand(Sk, device=DEV, generator=g) < 0.5).int()
    got = check(q, k, v, H, dtype, causal=causal, key_mask=kept)
    if B > 2:
        assert (got[2] == 0).all()                            # nothing visible
    one = torch.zeros(B, Sk, dtype=torch.int32, device=DEV)
    one[:, Sk // 2] = -7                                      # any nonzero word shows its key
    check(q, k, v, H, dtype, causal=causal, key_mask=one)


@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 2, 450, 449), (1, 75, 700, 450), (4, 20, 930, 223), (2, 20, 300, 300)])
def test_ragged_anchor_update(B, H, Sq, Sk):
    """A key far above the rest in a middle group, in the last complete one and in the ragged one."""
    for at in (Sk // 2, Sk // 32 * 32 - 5, Sk - 1):
        q, k, v = tensors(at, B, H, Sq, Sk, "f16", q_scale=4.0)
        k[:, at] = 3 * q.mean(dim=1)
        k[:, at] += k[:, at].sign() * 4
        check(q, k, v, H, "f16")
        check(q, k, v, H, "f16", causal=True)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,S", [(1, 2, 320), (2, 256, 256)])  # key-split and whole workgroups
@pytest.mark.parametrize("top", [40, 70])
def test_masked_largest_weight_is_exact(B, H, S, top, causal, dtype):
    """Masked calls keep the running maximum exact, also in groups without a hidden key: keys 0-31
    score 0, one later key a little above, the others far below, so every weight is a power of two or
    zero and the output rounds once, at the end (half a unit, and 2^-17 for the fp32 arithmetic)."""
    q, k, v = (torch.zeros(B, S, H * 64, device=DEV) for _ in range(3))
    rows = torch.linspace(0.9, 1.1, S, device=DEV)
    q[..., ::64] = 8 * rows[None, :, None]
    k[:, 32:, ::64] = -60
    k[:, top, ::64] = 3.4
    v[:, :128] = 1 + torch.rand(B, 1, H * 64, device=DEV, generator=torch.Generator(device=DEV).manual_seed(S))
    v[:, :32] *= 0.25
    q, k, v = (x.to(DTYPES[dtype]) for x in (q, k, v))
    mask = torch.ones(B, S, dtype=torch.int32, device=DEV)
    mask[:, -1] = 0
    got = sh.attention(q, k, v, H, causal=causal, key_mask=None if causal else mask)[:, 96:]
    score = q[:, 96:, ::64].double() * k[:, top, None, ::64].double() / 8       # [B, rows, H]
    weight = torch.exp(score).repeat_interleave(64, dim=-1)
    ref = (weight * v[:, top, None].double() + 32 * v[:, 0, None].double()) / (weight + 32)
    half_unit = torch.exp2(torch.floor(torch.log2(ref))) * UNIT[dtype]
    excess = ((got.double() - ref).abs() - half_unit) / ref
    assert excess.max().item() <= 2.0 ** -17, excess.max().item()


# as in test_ragged: key-split workgroups on either kernel, mixed ones within one head and across two, whole ones
KINDS = [(1, 2, 450, 449), (1, 75, 700, 450), (2, 16, 2560, 129), (4, 20, 930, 223), (2, 20, 300, 300)]


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("B,H,Sq,Sk", KINDS)
@pytest.mark.parametrize("masked", [False, True])
def test_ragged_strided_rows(B, H, Sq, Sk, masked, dtype):
    """K and V as column slices of one wide buffer (equal strides), and K from a wider buffer than V, with
    which a mixed workgroup stays within one head."""
    W = H * 64
    g = torch.Generator(device=DEV).manual_seed(Sk)
    wide = torch.randn(B, Sk, 3 * W + 64, device=DEV, generator=g).to(DTYPES[dtype])
    q = torch.randn(B, Sq, W, device=DEV, generator=g).to(DTYPES[dtype])
    v = torch.randn(B, Sk, W + 8, device=DEV, generator=g).to(DTYPES[dtype])
    mask = torch.ones(B, Sk, dtype=torch.int32, device=DEV)
    mask[:, Sk // 3: Sk // 2] = 0
    for key, value in ((wide[..., W:2 * W], wide[..., 2 * W:3 * W]), (wide[..., 8:W + 8], v[..., :W])):
        check(q, key, value, H, dtype, key_mask=mask if masked else None)


@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 2, 450, 449), (1, 75, 700, 450), (1, 32, 2560, 129), (1, 80, 930, 223),
                                       (1, 40, 300, 300)])
def test_ragged_rows_past_the_keys_are_not_read_into_the_result(B, H, Sq, Sk):
    """K and V are the leading rows of longer buffers whose next rows are NaN."""
    q, k, v = tensors(Sk, B, H, Sq, Sk + 128, "f16")
    k[:, Sk:] = v[:, Sk:] = float("nan")
    check(q, k[:, :Sk], v[:, :Sk], H, "f16")
    check(q, k[:, :Sk], v[:, :Sk], H, "f16", causal=True)
