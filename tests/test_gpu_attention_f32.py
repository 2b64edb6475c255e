"""One-pass float32 attention: parity with the CPU oracle and with the materialised path, masks in
every layout, bitwise batch invariance.

Tolerance (tests/_parity.py, as for the materialised float32 path): rtol 1e-5 of |O| + 2 (P |V|) per
element.  The kernel's own error is some 2^-24 times the root of the longest sum (head size and
key count below 2^10 here), well inside it.
"""

import math

import pytest
import torch

from batch_invariant_ops import scaled_dot_product_attention_batch_invariant as sdpa
from batch_invariant_ops import _native as nat

from _parity import check_sdpa
from _tol import assert_bitwise


def randn(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def test_sizes_taken_and_argument_errors():
    lib = nat.load(require_gpu=False)
    ok = lib.biops_sdpa_f32_supported
    assert ok(2, 4, 7, 9, 4, 128) and ok(1, 1, 1, 0, 128, 4)
    assert not ok(1, 1, 1, 1, 132, 4) and not ok(1, 1, 1, 1, 6, 4) and not ok(1, 1, 1, 1, 4, 130)
    for batch in (1, 1 << 24, 1 << 32):  # any number of samples: the path depends on one sample's sizes
        assert ok(batch, 16, 1, 5, 64, 64) and lib.biops_sdpa_f32_workspace_size(batch, 16, 1, 500, 64, 64) >= 0
    p = 256

    def call(d=64, q=p, sk=64, hkv=2, mask=None, mcode=0, causal=0):
        return lib.biops_sdpa_f32(1, 4, hkv, 3, 5, d, 64, q, 0, 0, 64, p, 0, 0, sk, p, 0, 0, 64, mask, mcode, 0, 0, 5, 1,
                                  causal, 1.0, p, None, 0, None)

    assert call(d=66) == 5 and call(hkv=3) == 1 and call(q=None) == 1
    assert call(q=p + 4) == 2 and call(sk=66) == 2
    assert call(mask=p, mcode=nat.BF16) == 3 and call(mask=p, mcode=nat.BOOL, causal=1) == 1


SHAPES = (
    # B, Hq, Hkv, Lq, Lk, D, Dv: query rows around the 128-row tile and its 32-row wavefronts, keys around
    # the 32-key block, head sizes on both sides of every class of the dispatch
    (2, 4, 2, 129, 257, 64, 64),
    (1, 2, 1, 128, 33, 72, 72),
    (2, 3, 3, 31, 32, 68, 96),
    (1, 2, 2, 33, 31, 80, 40),
    (1, 2, 2, 1, 1, 4, 4),
    (1, 4, 1, 200, 95, 96, 8),
    (1, 2, 2, 161, 300, 128, 128),
    (2, 2, 1, 97, 64, 100, 64),
    (1, 1, 1, 5, 65, 8, 100),
)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ("full", "causal", "boolean", "additive"))
@pytest.mark.parametrize("shape", SHAPES)
def test_f32_sdpa_matches_oracle_and_materialized(shape, kind, monkeypatch):
    B, Hq, Hkv, Lq, Lk, D, Dv = shape
    seed = 9500 + 10 * SHAPES.index(shape)
    q, k, v = randn(B, Hq, Lq, D, seed=seed), randn(B, Hkv, Lk, D, seed=seed + 1), randn(B, Hkv, Lk, Dv, seed=seed + 2)
    kw = dict(enable_gqa=Hq != Hkv, is_causal=kind == "causal")
    mask = None
    if kind in ("boolean", "additive"):
        keep = torch.rand(B, 1, Lq, Lk, generator=torch.Generator().manual_seed(seed + 3)) > 0.3
        keep[:, :, Lq // 2] = False  # a fully masked row gives 0
        keep[:, :, :, : Lk // 2] &= torch.arange(Lq).view(-1, 1) % 2 == 0  # the maximum appears late
        mask = keep
        if kind == "additive":
            mask = torch.rand(B, 1, Lq, Lk, generator=torch.Generator().manual_seed(seed + 4)) * -10
            mask[~keep] = -math.inf
    dev = dict(kw, attn_mask=None if mask is None else mask.cuda())
    out = sdpa(q.cuda(), k.cuda(), v.cuda(), **dev)
    check_sdpa(out, q, k, v, attn_mask=mask, what=f"float32 vs oracle {shape}", **kw)
    if mask is not None:
        assert torch.count_nonzero(out[:, :, Lq // 2]) == 0
        wide = torch.zeros(B, 1, Lq, 2 * Lk + 3, dtype=mask.dtype)  # same mask, key stride 2, odd row stride
        wide[..., 1:1 + 2 * Lk:2] = mask
        strided = sdpa(q.cuda(), k.cuda(), v.cuda(), **dict(kw, attn_mask=wide.cuda()[..., 1:1 + 2 * Lk:2]))
        assert_bitwise(strided, out, "strided mask")
    monkeypatch.setenv("BIOPS_ATTENTION_MATERIALIZE", "1")
    mat = sdpa(q.cuda(), k.cuda(), v.cuda(), **dev)
    assert torch.allclose(out, mat, rtol=1e-5, atol=2e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ("full", "causal", "boolean"))
@pytest.mark.parametrize("D", (64, 72, 128))
def test_f32_sdpa_is_batch_invariant(D, kind):
    """Samples alone (a workgroup per 128 keys), a batch that fills the chip (the workgroups merge their
    keys themselves), and views of wider buffers (head and row strides of their own)."""
    B, Lk = 48, 290
    assert nat.load().biops_sdpa_f32_workspace_size(1, 6, 150, Lk, D, D) > 0
    assert nat.load().biops_sdpa_f32_workspace_size(B, 6, 150, Lk, D, D) == 0
    q = randn(B, 150, 6, D, seed=9700).cuda().transpose(1, 2)
    kc, vc = (randn(B, 310, 2, D + 4, seed=9701 + i).cuda() for i in range(2))
    k, v = (x[:, 9:9 + Lk, :, :D].transpose(1, 2) for x in (kc, vc))
    mask = None
    if kind == "boolean":
        mask = torch.rand(B, 1, 150, Lk, generator=torch.Generator().manual_seed(9710)) > 0.3
        mask[:, :, ::3, :128] = False  # a whole group of keys masked out
        mask[:, :, 7] = False
        mask = mask.cuda()

    def run(sl, contiguous=False):
        args = [x[sl].contiguous() if contiguous else x[sl] for x in (q, k, v)]
        return sdpa(*args, attn_mask=None if mask is None else mask[sl], is_causal=kind == "causal", enable_gqa=True)

    full = run(slice(0, B))
    for j in (0, 21, 47):
        one = slice(j, j + 1)
        assert_bitwise(run(one), full[one], f"sample {j}")
        assert_bitwise(run(one, contiguous=True), full[one], f"sample {j} contiguous")


@pytest.mark.gpu
def test_f32_sdpa_large_scores_and_unread_rows():
    """Scores of several hundred (the running maximum grows block by block), NaN past the keys."""
    q = randn(1, 2, 70, 64, seed=9800)
    k = randn(1, 2, 130, 64, seed=9801) * torch.linspace(1, 30, 130).view(1, 1, -1, 1)
    v = randn(1, 2, 130, 64, seed=9802)
    kc, vc = (torch.full((1, 2, 200, 64), math.nan, device="cuda") for _ in "kv")
    kc[:, :, :130], vc[:, :, :130] = k.cuda(), v.cuda()
    out = sdpa(q.cuda(), kc[:, :, :130], vc[:, :, :130])
    # the scores' own rounding (relative 2^-24 of up to 2^10) moves a probability by up to 2^-13
    ref = torch.softmax((q.double() @ k.double().transpose(-1, -2)) / 8.0, -1) @ v.double()
    assert torch.allclose(out.cpu().double(), ref, rtol=2.0**-11, atol=2.0**-11)


@pytest.mark.gpu
@pytest.mark.parametrize("B", (1, 160))
def test_f32_sdpa_masks_of_the_lowest_value(B):
    """Padding written as the type's lowest value instead of -inf: keys in front, keys at the back, a whole
    row (which averages V), with one workgroup per 128 keys and with one per query tile."""
    L = 300
    q, k, v = (randn(B, 4, L, 64, seed=9810 + i) for i in range(3))
    mask = torch.zeros(B, 1, L, L)
    low = torch.finfo(torch.float32).min
    mask[:, :, 0:90, :140] = low
    mask[:, :, 90:200, 100:] = low
    mask[:, :, 200:210] = low
    out = sdpa(q.cuda(), k.cuda(), v.cuda(), attn_mask=mask.cuda())
    one = slice(B - 1, B)
    check_sdpa(out[one], q[one], k[one], v[one], attn_mask=mask[one], what="lowest value")


@pytest.mark.gpu
@pytest.mark.parametrize("B", (1, 160))
def test_f32_sdpa_passes_nan_on(B, monkeypatch):
    """128 keys of NaN (whose running maximum stays -inf) before or after others give NaN in every row of
    their head; a row of which no score compares gives 0, as the softmax kernels have it."""
    q, k, v = (randn(B, 4, 300, 64, seed=9820 + i).cuda() for i in range(3))
    q[:, 0, 5] = math.nan
    k[:, 1, :128] = math.nan
    k[:, 2, 128:256] = math.nan
    out = sdpa(q, k, v)
    assert out[:, 1:3].isnan().all() and torch.count_nonzero(out[:, 0, 5]) == 0
    assert out[:, 0].isfinite().all() and out[:, 3].isfinite().all()
    monkeypatch.setenv("BIOPS_ATTENTION_MATERIALIZE", "1")
    assert torch.equal(sdpa(q, k, v).isnan(), out.isnan())


@pytest.mark.gpu
def test_f32_sdpa_probabilities_to_the_last_bits():
    """Two keys with scores 0 and -x: the output is exp(-x) / (1 + exp(-x)).  expf is within 1 ulp, the sum,
    the reciprocal and the product round once more each: under 4 ulps, 2^-21 of the value (taking the
    exponential of a rounded multiple of x was off by up to x 2^-24 more)."""
    x = torch.linspace(0.0, 86.0, 1024)
    q, k, v = (torch.zeros(1, 1, n, 4) for n in (1024, 2, 2))
    q[0, 0, :, 0] = x
    k[0, 0, 1, 0] = -1.0
    v[0, 0, 1] = 1.0
    out = sdpa(q.cuda(), k.cuda(), v.cuda(), scale=1.0)
    ref = torch.sigmoid(-x.double())[:, None].expand(-1, 4)
    assert torch.allclose(out[0, 0].cpu().double(), ref, rtol=2.0**-21, atol=0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ("base", "pitch", "keys", "wide", "shared"))
def test_f32_sdpa_views_give_the_bits_of_their_copies(layout):
    """Rows that are not 16-byte aligned (an offset base, an odd pitch, keys behind an odd offset) and
    rows further apart than the kernel's 32-bit offsets take the same path as an aligned copy."""
    B, H, L, D = 3, 2, 200, 64

    def view(seed):
        if layout == "base":
            return randn(B * H * L * D + 1, seed=seed).cuda()[1:].view(B, H, L, D)
        if layout == "pitch":
            return randn(B, L, H, D + 1, seed=seed).cuda()[..., :D].transpose(1, 2)
        if layout == "shared":  # one odd-pitch sample and head for all
            return randn(1, 1, L, D + 1, seed=seed).cuda()[..., :D].expand(B, H, L, D)
        if layout == "keys":
            return randn(B, H, L * D + 3, seed=seed).cuda()[..., 3:].view(B, H, L, D)
        t = torch.empty(((L - 1) << 25) + D, device="cuda").as_strided((1, 1, L, D), (0, 0, 1 << 25, 1))
        t.copy_(randn(1, 1, L, D, seed=seed))
        return t.expand(B, H, L, D)

    if layout == "wide":
        L = 9  # 1 GiB of rows
    q, k, v = (view(9830 + i) for i in range(3))
    copies = [x.clone(memory_format=torch.contiguous_format) for x in (q, k, v)]
    out = sdpa(q, k, v)
    assert_bitwise(out, sdpa(*copies), "copy")
    assert_bitwise(sdpa(q[1:2], k[1:2], v[1:2]), out[1:2], "one sample")


@pytest.mark.gpu
def test_f32_sdpa_of_more_tiles_than_a_launch_has():
    """2^24 and some query tiles: 256 threads each are more than one launch takes."""
    B, H = (1 << 20) + 3, 16
    q = torch.randn(B, H, 1, 4, generator=torch.Generator("cuda").manual_seed(9840), device="cuda")
    k, v = (randn(1, H, 5, 4, seed=9841 + i).cuda() for i in range(2))
    out = sdpa(q, k.expand(B, H, 5, 4), v.expand(B, H, 5, 4))
    for rows in (slice(0, 2), slice(B - 5, B)):
        n = rows.stop - rows.start
        assert_bitwise(sdpa(q[rows], k.expand(n, H, 5, 4), v.expand(n, H, 5, 4)), out[rows], str(rows))


@pytest.mark.gpu
@pytest.mark.parametrize("B", (1, 160))
def test_f32_sdpa_values_behind_a_mask(B, monkeypatch):
    """A masked key has the weight 0, and 0 times NaN or infinity is NaN in every row that attends to anything:
    in the 128 keys of a chunk without a visible key as elsewhere."""
    q, k, v = (randn(B, 4, 400, 64, seed=9850 + i).cuda() for i in range(3))
    mask = torch.ones(B, 1, 1, 400, dtype=torch.bool, device="cuda")
    mask[..., :150] = False
    mask[..., 260:] = False
    v[:, 0, 3, 5] = math.nan
    v[:, 1, 130, 6] = math.inf
    v[:, 2, 390, 7] = math.nan
    out = sdpa(q, k, v, attn_mask=mask)
    for head, column in ((0, 5), (1, 6), (2, 7)):
        assert out[:, head, :, column].isnan().all()
    assert int(out.isnan().sum()) == 3 * B * 400
    monkeypatch.setenv("BIOPS_ATTENTION_MATERIALIZE", "1")
    assert torch.equal(sdpa(q, k, v, attn_mask=mask).isnan(), out.isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ("full", "causal", "boolean", "additive"))
@pytest.mark.parametrize("D,Dv", ((4, 64), (64, 8), (72, 72), (80, 40), (96, 96), (100, 128), (128, 36)))
@pytest.mark.parametrize("lq,lk", ((1, 1), (31, 33), (33, 128), (65, 129), (40, 260)))
def test_f32_sdpa_of_few_rows_has_the_bits_of_a_large_launch(lq, lk, D, Dv, kind):
    """One sample (a workgroup per 32 query rows and 128 keys) and a batch that fills the chip."""
    B, H = 160, 8
    seed = 9860 + lk
    q, k, v = randn(B, H, lq, D, seed=seed).cuda(), randn(B, 2, lk, D, seed=seed + 1).cuda(), randn(B, 2, lk, Dv, seed=seed + 2).cuda()
    k *= torch.linspace(0.5, 4, lk, device="cuda").view(-1, 1)  # the maximum grows from block to block
    v[7, 0, 0, 0] = math.inf
    mask = None
    if kind in ("boolean", "additive"):
        g = torch.Generator().manual_seed(seed + 3)
        mask = torch.rand(B, 1, lq, lk, generator=g) > 0.3
        mask[:, :, ::3, :32] = False  # a block, and for some rows more, without a visible key
        mask[:, :, 1::5, :128] = False
        if kind == "additive":
            mask = torch.where(mask, torch.rand(B, 1, lq, lk, generator=g) * -5, torch.tensor(-math.inf))
        mask = mask.cuda()

    def run(rows):
        return sdpa(q[rows], k[rows], v[rows], attn_mask=None if mask is None else mask[rows],
                    is_causal=kind == "causal", enable_gqa=True)

    full = run(slice(None))
    for j in (0, 7, B - 1):
        one = slice(j, j + 1)
        assert torch.equal(run(one).isnan(), full[one].isnan())
        assert_bitwise(run(one).nan_to_num(1.0), full[one].nan_to_num(1.0), f"sample {j}")


@pytest.mark.gpu
def test_f32_rows_keep_what_a_view_repeats():
    """The aligned copy of an operand that is repeated over samples, heads or rows has it once."""
    from batch_invariant_ops.batch_invariant_ops import _f32_rows

    t = torch.arange(7 * 5, dtype=torch.float32, device="cuda").view(1, 1, 7, 5)[..., :4]
    for view in (t.expand(3, 2, 7, 4), t[:, :, 2:3].expand(3, 2, 6, 4), t[:, :, :1], t[:, :, :0].expand(3, 2, 0, 4)):
        rows, strides = _f32_rows(view)
        assert torch.equal(rows, view) and rows.data_ptr() % 16 == 0 and all(st % 4 == 0 for st in strides)
        assert rows.untyped_storage().nbytes() <= 7 * 5 * 4
