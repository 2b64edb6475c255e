"""Attention of few query rows against many keys (keys split over workgroups): parity with the CPU
oracle and with the materialised path, bitwise batch invariance, and the rule that picks it.

Parity as for the fused kernel (tests/_parity.py): the roundings are the same, only the fp32
orders of the row sum and of the P V sum differ.
"""

import math

import pytest
import torch

from batch_invariant_ops import scaled_dot_product_attention_batch_invariant as sdpa
from batch_invariant_ops import _native as nat

from _parity import check_sdpa, check_sdpa_against
from _tol import assert_bitwise

DTYPES16 = (torch.bfloat16, torch.float16)


def randn(*shape, seed, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def size(B, Hq, Hkv, Lq, Lk, D=128, Dv=128, dtype=nat.BF16, causal=0):
    return nat.load(require_gpu=False).biops_sdpa_split_workspace_size(dtype, B, Hq, Hkv, Lq, Lk, D, Dv, causal)


def test_which_calls_are_split():
    """By the sizes of one sample only: the batch size never changes the answer."""
    for batch in (1, 3, 64):
        assert size(batch, 16, 4, 1, 513) > 0 and size(batch, 16, 4, 16, 4096) > 0
        assert size(batch, 16, 4, 1, 512) < 0 and size(batch, 16, 4, 17, 4096) < 0
        assert size(batch, 16, 4, 1, 4096, causal=nat.CAUSAL_TOP_LEFT) < 0
        assert size(batch, 16, 4, 1, 4096, dtype=nat.F32) < 0
        assert size(batch, 16, 4, 1, 4096, D=264) < 0 and size(batch, 16, 4, 1, 4096, Dv=12) < 0
    assert size(1, 16, 3, 1, 4096) < 0 and size(0, 16, 4, 1, 4096) < 0
    assert nat.load(require_gpu=False).biops_sdpa_split_max_query() == 16


def test_large_workspaces_are_left_to_the_fused_kernel():
    """Which path runs changes no bit, so the batch may enter here: 2 GiB at most."""
    assert 0 < size(64, 64, 8, 1, 32768) <= 2 << 30
    assert size(64, 64, 8, 16, 32768) < 0 and size(1, 8, 8, 1, 1 << 23) < 0
    assert size(1 << 20, 64, 64, 16, 4096) < 0  # also past the launch limits


@pytest.mark.gpu
def test_without_memory_for_the_workspace(monkeypatch):
    q = randn(2, 8, 3, 64, seed=9430, dtype=torch.bfloat16).cuda()
    k, v = (randn(2, 2, 700, 64, seed=9431 + i, dtype=torch.bfloat16).cuda() for i in range(2))
    out = sdpa(q, k, v, enable_gqa=True)
    empty = torch.empty

    def refuse(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no workspace")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", refuse)
    assert_bitwise(sdpa(q, k, v, enable_gqa=True), out, "fused kernel instead")


def test_argument_errors_come_before_any_launch():
    lib = nat.load(require_gpu=False)
    p = 256
    need = size(1, 4, 4, 1, 600)

    def call(dtype=nat.BF16, lk=600, q=p, sk=128, mask=None, mcode=0, ld=600, ws=p, nbytes=need):
        return lib.biops_sdpa_split(dtype, 1, 4, 4, 1, lk, 128, 128, q, 0, 0, 128, p, 0, 0, sk, p, 0, 0, 128,
                                    mask, mcode, 0, 0, ld, 1, 1.0, p, ws, nbytes, None)

    assert call(dtype=nat.F32) == 1 and call(lk=100) == 1 and call(q=None) == 1
    assert call(q=p + 2) == 2 and call(sk=130) == 2 and call(ws=p + 16) == 2
    assert call(nbytes=need - 1) == 5
    assert call(mask=p, mcode=nat.F32) == 3 and call(mask=p + 1, mcode=nat.BOOL) == 2


SHAPES = (
    # B, Hq, Hkv, Lq, Lk, D, Dv: packed rows 1, 4, 31, 32, 33, 64, 66 and 128; key counts around the 64-key
    # wavefront, the 256-key workgroup and the value split (256 keys up to 2048, then 512)
    (2, 1, 1, 1, 513, 128, 128),
    (2, 16, 4, 1, 576, 128, 128),
    (1, 1, 1, 16, 767, 64, 64),
    (1, 31, 1, 1, 768, 64, 40),
    (1, 4, 1, 8, 769, 72, 128),
    (2, 6, 2, 11, 1000, 256, 256),
    (1, 8, 2, 16, 2048, 128, 64),
    (1, 12, 2, 11, 2049, 8, 200),
    (1, 8, 1, 16, 2561, 128, 128),
)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES16)
@pytest.mark.parametrize("mask_kind", ("none", "boolean", "additive"))
@pytest.mark.parametrize("shape", SHAPES)
def test_split_sdpa_matches_oracle_and_materialized(dtype, mask_kind, shape, monkeypatch):
    B, Hq, Hkv, Lq, Lk, D, Dv = shape
    if mask_kind != "none":
        Lk = -(-Lk // 4) * 4  # masks of other key counts take the materialised path
    seed = 9000 + 10 * SHAPES.index(shape)
    q = randn(B, Hq, Lq, D, seed=seed, dtype=dtype)
    k = randn(B, Hkv, Lk, D, seed=seed + 1, dtype=dtype)
    v = randn(B, Hkv, Lk, Dv, seed=seed + 2, dtype=dtype)
    mask = None
    if mask_kind != "none":
        keep = torch.rand(B, 1, Lq, Lk, generator=torch.Generator().manual_seed(seed + 3)) > 0.2
        keep[:, :, Lq // 2] = False  # a fully masked row gives 0
        keep[0, :, :, : Lk // 2] = False  # whole workgroups without a visible key
        mask = keep
        if mask_kind == "additive":
            mask = (torch.rand(B, 1, Lq, Lk, generator=torch.Generator().manual_seed(seed + 4)) * -10).to(dtype)
            mask[~keep] = -math.inf
    assert size(B, Hq, Hkv, Lq, Lk, D, Dv) > 0
    kw = dict(enable_gqa=Hq != Hkv)
    dev = dict(kw, attn_mask=None if mask is None else mask.cuda())
    out = sdpa(q.cuda(), k.cuda(), v.cuda(), **dev)
    check_sdpa(out, q, k, v, attn_mask=mask, what=f"split vs oracle {shape}", **kw)
    if mask is not None:
        assert torch.count_nonzero(out[:, :, Lq // 2]) == 0
    monkeypatch.setenv("BIOPS_ATTENTION_MATERIALIZE", "1")
    mat = sdpa(q.cuda(), k.cuda(), v.cuda(), **dev)
    check_sdpa_against(out, mat, q, k, v, attn_mask=mask, min_exact=0.9, what="split vs materialised", **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES16)
@pytest.mark.parametrize("mask_kind", ("none", "boolean", "additive", "lowest"))
@pytest.mark.parametrize("shape", SHAPES + ((1, 2, 1, 3, 9000, 64, 128), (40, 14, 2, 5, 1029, 128, 136)))
def test_query_rows_in_chunks_give_the_bits_of_one_call(dtype, mask_kind, shape):
    """A row's bits are the same in a call of up to 16 query rows (split) and in a longer one (fused)."""
    B, Hq, Hkv, Lq, Lk, D, Dv = shape
    if mask_kind != "none":
        Lk = -(-Lk // 4) * 4
    seed = 9450 + Lk
    q = randn(B, Hq, Lq + 30, D, seed=seed, dtype=dtype).cuda()
    k = (randn(B, Hkv, Lk, D, seed=seed + 1, dtype=dtype) * torch.linspace(0.2, 3, Lk).view(-1, 1).to(dtype)).cuda()
    v = randn(B, Hkv, Lk, Dv, seed=seed + 2, dtype=dtype).cuda()
    mask = None
    if mask_kind != "none":
        g = torch.Generator().manual_seed(seed + 3)
        mask = torch.rand(B, 1, Lq + 30, Lk, generator=g) > 0.2
        mask[:, :, Lq // 2] = False
        mask[0, :, :, : Lk // 2] = False
        if mask_kind != "boolean":
            keep = mask
            mask = (torch.rand(B, 1, Lq + 30, Lk, generator=g) * -10).to(dtype)
            mask[~keep] = -math.inf if mask_kind == "additive" else torch.finfo(dtype).min
        mask = mask.cuda()
    assert size(B, Hq, Hkv, Lq, Lk, D, Dv) > 0 and size(B, Hq, Hkv, Lq + 30, Lk, D, Dv) < 0
    for scale in (None, 0.3):
        whole = sdpa(q, k, v, attn_mask=mask, scale=scale, enable_gqa=Hq != Hkv)
        for first in (0, 13):
            rows = slice(first, first + Lq)
            part = sdpa(q[:, :, rows], k, v, attn_mask=None if mask is None else mask[:, :, rows], scale=scale,
                        enable_gqa=Hq != Hkv)
            assert_bitwise(part, whole[:, :, rows], f"rows from {first}")


# Row and column blocks of the value kernel by launch size (256 compute units): (batch, query heads, kv
# heads, query rows, keys, head size, value size), blocks of rows x columns.
LAUNCHES = (
    ((100, 8, 2, 2, 530, 64, 64), "16 x 64"),
    ((150, 8, 2, 1, 530, 64, 72), "16 x 128"),
    ((40, 8, 2, 1, 2500, 64, 64), "4 x 32"),
    ((60, 8, 2, 1, 2500, 64, 128), "4 x 64"),
    ((100, 8, 2, 1, 2500, 64, 128), "4 x 128"),
    ((15, 16, 2, 1, 2100, 64, 128), "8 x 16"),
    ((30, 16, 2, 1, 2100, 64, 128), "8 x 32"),
    ((60, 16, 2, 1, 2100, 64, 128), "8 x 64"),
    ((80, 16, 2, 1, 2100, 64, 128), "8 x 128"),
    ((64, 14, 2, 4, 600, 64, 136), "32 x 64"),
    ((64, 14, 2, 6, 600, 64, 136), "64 x 128"),
)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,blocks", LAUNCHES)
def test_value_blocks_give_the_bits_of_one_call(shape, blocks):
    B, Hq, Hkv, Lq, Lk, D, Dv = shape
    g = torch.Generator("cuda").manual_seed(9470)
    q, k, v = (torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
               for s in ((B, Hq, 20, D), (B, Hkv, Lk, D), (B, Hkv, Lk, Dv)))
    whole = sdpa(q, k, v, enable_gqa=True)
    assert_bitwise(sdpa(q[:, :, :Lq], k, v, enable_gqa=True), whole[:, :, :Lq], blocks)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES16)
def test_infinities_and_nan_in_chunks_of_query_rows(dtype):
    """NaN and infinite queries, keys and values reach the same outputs at any number of query rows."""
    q = randn(4, 4, 40, 64, seed=9480, dtype=dtype).cuda()
    k, v = (randn(4, 2, 1100, 64, seed=9481 + i, dtype=dtype).cuda() for i in range(2))
    q[0, 1, 3] = math.nan
    k[1, 0, 70:200] = math.nan
    k[2, 1, 500, 0] = math.inf
    v[3, 0, 5] = math.nan
    v[3, 1, 1099] = math.inf
    mask = torch.ones(4, 1, 1, 1100, dtype=torch.bool, device="cuda")
    mask[3, ..., 1000:] = False
    for m in (None, mask):
        whole = sdpa(q, k, v, attn_mask=m, enable_gqa=True)
        part = sdpa(q[:, :, :7], k, v, attn_mask=m, enable_gqa=True)
        assert torch.equal(part.isnan(), whole[:, :, :7].isnan())
        assert_bitwise(part.nan_to_num(1.0), whole[:, :, :7].nan_to_num(1.0), "finite outputs")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES16)
@pytest.mark.parametrize("heads", ((16, 4, 1), (64, 8, 16), (8, 8, 5)))
def test_split_sdpa_is_batch_invariant(dtype, heads):
    """Samples alone and in a batch large enough for several row tiles per workgroup; the batch is
    a view of a longer cache (row and batch strides of their own)."""
    Hq, Hkv, Lq = heads
    B, Lk = 9, 1111
    q = randn(B, Lq, Hq, 128, seed=9200, dtype=dtype).cuda().transpose(1, 2)
    kc = randn(B, Lk + 50, Hkv, 128, seed=9201, dtype=dtype).cuda()
    vc = randn(B, Lk + 50, Hkv, 128, seed=9202, dtype=dtype).cuda()
    k, v = kc[:, 7:7 + Lk].transpose(1, 2), vc[:, 7:7 + Lk].transpose(1, 2)
    full = sdpa(q, k, v, enable_gqa=Hq != Hkv)
    for j in (0, 4, 8):
        one = slice(j, j + 1)
        assert_bitwise(sdpa(q[one], k[one], v[one], enable_gqa=Hq != Hkv), full[one], f"sample {j} alone")
        assert_bitwise(sdpa(q[one].contiguous(), k[one].contiguous(), v[one].contiguous(), enable_gqa=Hq != Hkv),
                       full[one], f"sample {j} contiguous")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES16)
def test_split_sdpa_masks_of_the_lowest_value(dtype):
    """Padding written as the type's lowest value instead of -inf: whole wavefronts and workgroups of
    keys in front, at the back, and all keys (which averages V)."""
    q = randn(3, 8, 4, 64, seed=9250, dtype=dtype)
    k, v = (randn(3, 2, 1100, 64, seed=9251 + i, dtype=dtype) for i in range(2))
    mask = torch.zeros(3, 1, 4, 1100, dtype=dtype)
    low = torch.finfo(dtype).min
    mask[0, :, :, :700] = low
    mask[1, :, :, 300:] = low
    mask[2, :, 1] = low
    out = sdpa(q.cuda(), k.cuda(), v.cuda(), attn_mask=mask.cuda(), enable_gqa=True)
    check_sdpa(out, q, k, v, attn_mask=mask, what="lowest value", enable_gqa=True)


@pytest.mark.gpu
def test_split_sdpa_ignores_what_lies_past_the_keys():
    """Key and value rows past the end (NaN here) reach no output."""
    kc, vc = (torch.full((1, 2, 700, 64), math.nan, dtype=torch.bfloat16, device="cuda") for _ in "kv")
    q = randn(1, 4, 2, 64, seed=9300, dtype=torch.bfloat16).cuda()
    k, v = (randn(1, 2, 613, 64, seed=9301 + i, dtype=torch.bfloat16).cuda() for i in range(2))
    kc[:, :, :613], vc[:, :, :613] = k, v
    assert_bitwise(sdpa(q, kc[:, :, :613], vc[:, :, :613], enable_gqa=True), sdpa(q, k, v, enable_gqa=True), "")


@pytest.mark.gpu
def test_split_sdpa_in_a_graph():
    q = randn(2, 8, 1, 128, seed=9400, dtype=torch.bfloat16).cuda()
    k, v = (randn(2, 2, 2100, 128, seed=9401 + i, dtype=torch.bfloat16).cuda() for i in range(2))
    sdpa(q, k, v, enable_gqa=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sdpa(q, k, v, enable_gqa=True)
    for seed in (9410, 9420, 9430):
        q.copy_(randn(2, 8, 1, 128, seed=seed, dtype=torch.bfloat16))
        k.copy_(randn(2, 2, 2100, 128, seed=seed + 1, dtype=torch.bfloat16))
        eager = sdpa(q, k, v, enable_gqa=True)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert_bitwise(out, eager, f"replay {seed}")
