"""Kernel 1 parity: HIP prefill attention vs the fp32 oracle (through the C ABI)."""
import ctypes

import pytest
import torch

import oracle
from daisy_amd import _lib, ops
from helpers import assert_close_bf16, check_prefill_of_many_heads, say

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, D, seed, normalise=False):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, T, H, D, generator=g) for _ in range(3))
    if normalise:
        q, k, v = (oracle.rms_norm(t) for t in (q, k, v))
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


def _oracle(q, k, v, window, cos=None, sin=None, doc_start=None, scale=0.12, rows=None):
    if cos is not None:
        q, k = oracle.apply_rope(q, cos, sin), oracle.apply_rope(k, cos, sin)
    q_, k_, v_ = (t.transpose(1, 2) for t in (q, k, v))
    if rows is None and q.shape[1] <= 2048:
        o = oracle.windowed_attention(q_, k_, v_, window, scale, doc_start)
    else:
        o = oracle.windowed_attention_blockwise(q_, k_, v_, window, scale, doc_start, rows=rows)
    return o.transpose(1, 2), k


CASES = [
    # B, T, H, D, window, rope, docs
    (1, 256, 4, 64, 128, True, False),      # plumbing config shape
    (2, 512, 2, 128, 200, True, False),
    (1, 300, 3, 128, 64, True, True),       # ragged T, documents
    (1, 129, 1, 128, None, False, False),   # full causal, one row past a block
    (2, 64, 2, 64, 1, False, False),        # window 1: every query sees only itself
    (1, 1, 1, 128, 16, True, False),        # single token
    (1, 1000, 2, 128, 1000, True, True),    # window == T
    (1, 96, 2, 8, 16, True, True),          # scalar kernel (small head dim)
    (1, 40, 1, 2, None, True, False),       # scalar kernel, head dim 2 (no truncation in the tables)
    # longer sequences: many tiles per query block, rotated tile order with a wrap
    (1, 1111, 2, 128, 300, True, True),     # ragged T, documents, window shorter than a block
    (2, 1024, 1, 64, 1000, True, False),    # head dim 64, window just under T
    (1, 1300, 2, 128, None, False, False),  # full causal
    (1, 2048, 1, 128, 64, False, True),     # window of one tile: most tiles of a block are skipped
]


@pytest.mark.parametrize("B,T,H,D,window,rope,docs", CASES)
def test_prefill_matches_oracle(B, T, H, D, window, rope, docs):
    say(f"prefill case B{B} T{T} H{H} D{D} W{window} rope={rope} docs={docs}")
    q, k, v = _inputs(B, T, H, D, seed=T + D)
    cos = sin = doc_start = None
    if rope:
        cos, sin = oracle.rope_tables(D, T + 5)
    if docs:
        ids = torch.randint(0, 7, (T,), generator=torch.Generator().manual_seed(1))
        doc_start = oracle.doc_start_from_ids(ids, 3)
    ref, k_ref = _oracle(q, k, v, window, None if cos is None else cos[:T], None if sin is None else sin[:T], doc_start)
    dev = "cuda:0"
    o, k_rot = ops.prefill_attention(
        q.to(dev), k.to(dev), v.to(dev), window=window,
        cos=None if cos is None else cos.to(dev), sin=None if sin is None else sin.to(dev),
        doc_start=None if doc_start is None else doc_start.to(dev))
    torch.cuda.synchronize()
    assert_close_bf16(o, ref, "o")
    if rope:
        bad = (k_rot.cpu() != k_ref)
        assert not bad.any(), (f"rotated keys must be bit-identical to the oracle's bf16 RoPE: {int(bad.sum())} of "
                               f"{bad.numel()} differ, max diff {(k_rot.cpu().float() - k_ref.float()).abs().max().item():.3e}")
    else:
        assert k_rot is None
    if D in (64, 128):
        check_prefill_of_many_heads(*(t.to(dev) for t in (q, k, v)), ref, "oracle case", k_rot=k_ref if rope else None, window=window,
                                    cos=None if cos is None else cos.to(dev), sin=None if sin is None else sin.to(dev),
                                    doc_start=None if doc_start is None else doc_start.to(dev))


def test_prefill_strided_views_of_merged_qkv():
    """q, k, v as chunks of one [B, T, 3H, D] projection output, as the module passes them."""
    B, T, H, D = 2, 384, 4, 128
    g = torch.Generator().manual_seed(7)
    qkv = torch.randn(B, T, 3 * H, D, generator=g).bfloat16()
    q, k, v = qkv.chunk(3, dim=-2)
    cos, sin = oracle.rope_tables(D, T)
    ref, _ = _oracle(q, k, v, 100, cos, sin)
    dq = qkv.to("cuda:0")
    q2, k2, v2 = dq.chunk(3, dim=-2)
    o, _ = ops.prefill_attention(q2, k2, v2, window=100, cos=cos.cuda(), sin=sin.cuda())
    assert_close_bf16(o, ref, "o")


@pytest.mark.parametrize("H,D,T", [(4, 128, 333), (3, 128, 200), (2, 64, 130)])
def test_prefill_outputs_with_caller_strides(H, D, T):
    """o and the rotated keys written into views with other strides ([B, H, T, D] storage, the ring's
    layout; rows of a wider buffer) equal the contiguous results bit for bit, and nothing outside the
    views is touched.  Odd H takes the one-head-per-thread pre-pass, even H the two-head one."""
    B, W = 2, 70
    q, k, v = (t.cuda() for t in _inputs(B, T, H, D, seed=21))
    cos, sin = (t.cuda() for t in oracle.rope_tables(D, T))
    o_ref, k_ref = ops.prefill_attention(q, k, v, window=W, cos=cos, sin=sin)
    # [B, H, T, D] storage seen as [B, T, H, D]
    o_bhtd = torch.full((B, H, T, D), 7.0, dtype=torch.bfloat16, device="cuda:0")
    k_bhtd = torch.full((B, H, T, D), 7.0, dtype=torch.bfloat16, device="cuda:0")
    ops.prefill_attention(q, k, v, window=W, cos=cos, sin=sin, out=o_bhtd.transpose(1, 2), k_out=k_bhtd.transpose(1, 2))
    assert torch.equal(o_bhtd.transpose(1, 2), o_ref) and torch.equal(k_bhtd.transpose(1, 2), k_ref)
    # rows of a wider buffer: [B, T, H, D + 16] with the last 16 channels of every row left alone
    o_wide = torch.full((B, T, H, D + 16), 7.0, dtype=torch.bfloat16, device="cuda:0")
    k_wide = torch.full((B, T, H, D + 16), 7.0, dtype=torch.bfloat16, device="cuda:0")
    ops.prefill_attention(q, k, v, window=W, cos=cos, sin=sin, out=o_wide[..., :D], k_out=k_wide[..., :D])
    assert torch.equal(o_wide[..., :D], o_ref) and torch.equal(k_wide[..., :D], k_ref)
    assert bool((o_wide[..., D:] == 7.0).all()) and bool((k_wide[..., D:] == 7.0).all())
    say(f"strided outputs H={H} D={D} T={T}: equal to the contiguous results")


def test_prefill_long_sequence_sampled_rows():
    """T = 16384 with a 2048 window: spot-check rows against the blockwise oracle."""
    B, T, H, D, W = 1, 16384, 2, 128, 2048
    q, k, v = _inputs(B, T, H, D, seed=3)
    rows = torch.cat([torch.arange(0, 64), torch.arange(2040, 2060), torch.arange(8000, 8032), torch.arange(T - 64, T)])
    ref, _ = _oracle(q, k, v, W, rows=rows)
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=W)
    assert_close_bf16(o[:, rows.cuda()], ref, "o[rows]")


@pytest.mark.parametrize("T,window,docs", [(63, None, False), (64, None, False), (65, None, True), (193, 383, False), (1000, 384, False), (1000, 385, True),
                                           (1025, 575, False), (777, 640, True)])
def test_prefill_tiles_of_64_keys(T, window, docs):
    """Head dim 64 takes 64 keys per tile from a window of 384 on: rows that end before, at and behind a tile's and a product's end,
    windows whose first key lies in either half of a tile, documents that start anywhere in one."""
    q, k, v = _inputs(1, T, 3, 64, seed=T)
    doc_start = None
    if docs:
        doc_start = oracle.doc_start_from_ids(torch.randint(0, 60, (T,), generator=torch.Generator().manual_seed(2)), 3)
    ref, _ = _oracle(q, k, v, window, doc_start=doc_start)
    check_prefill_of_many_heads(q.cuda(), k.cuda(), v.cuda(), ref, f"T{T} W{window}", window=window,
                                doc_start=None if doc_start is None else doc_start.cuda())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,T,H,window", [(1, 257, 1, None), (1, 288, 3, None), (1, 289, 2, None), (2, 161, 2, 97), (1, 200, 3, 98), (1, 1023, 8, 128),
                                          (1, 1025, 8, 128), (1, 1030, 12, None), (1, 1537, 9, None), (3, 31, 2, None)])
def test_few_query_blocks_on_both_sides_of_eight_wavefronts(B, T, H, window, D):
    """Wavefronts with no tile, one, and several; the last tile short; as many workgroups as either rule allows, and more."""
    q, k, v = _inputs(B, T, H, D, seed=T)
    rows = None if T <= 1100 else torch.cat([torch.arange(40), torch.arange(T - 70, T)])
    ref, _ = _oracle(q, k, v, window, rows=rows)
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=window)
    assert_close_bf16(o if rows is None else o[:, rows.cuda()], ref, f"T{T} H{H} W{window}")


def test_prefill_is_deterministic_and_window_invariant():
    """A window >= T equals full causal attention bit for bit; repeated calls agree."""
    B, T, H, D = 1, 320, 2, 128
    q, k, v = (t.cuda() for t in _inputs(B, T, H, D, seed=11))
    a, _ = ops.prefill_attention(q, k, v, window=None)
    b, _ = ops.prefill_attention(q, k, v, window=T)
    c, _ = ops.prefill_attention(q, k, v, window=T + 1000)
    assert torch.equal(a, b) and torch.equal(a, c)
    q, k, v = (t.repeat(1, 1, 200, 1) for t in (q, k, v))      # more query blocks than the kernel for few of them takes
    a, b, c = (ops.prefill_attention(q, k, v, window=w)[0] for w in (None, T, T + 1000))
    assert torch.equal(a, b) and torch.equal(a, c)


def test_prefill_rejects_bad_arguments():
    q = torch.zeros(1, 8, 1, 64, dtype=torch.bfloat16, device="cuda:0")
    with pytest.raises(RuntimeError, match="head_dim"):
        ops.prefill_attention(torch.zeros(1, 8, 1, 7 * 2 + 1, dtype=torch.bfloat16, device="cuda:0"),
                              torch.zeros(1, 8, 1, 15, dtype=torch.bfloat16, device="cuda:0"),
                              torch.zeros(1, 8, 1, 15, dtype=torch.bfloat16, device="cuda:0"), window=4)
    with pytest.raises(TypeError):
        ops.prefill_attention(q.float(), q.float(), q.float(), window=4)
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.prefill_attention(q.cpu(), q.cpu(), q.cpu(), window=4)


# Documents change the order in which the blocks of 128 queries are worked on: every block once, whatever the lengths.  Rows of more
# blocks than the order covers, (batch, head) pairs that do and do not divide among the XCDs, documents of one token, one document.
@pytest.mark.parametrize("B,T,H,D,W,starts", [(1, 8300, 8, 64, 1024, (0, 1, 700, 4000, 4128, 8299)), (1, 8300, 3, 128, None, (0, 2500, 2501, 6000)),
                                              (2, 3333, 16, 64, 256, (0,)), (1, 65537, 2, 64, 128, (0, 31000)), (1, 65536, 2, 64, 128, (0, 31000)),
                                              (1, 5000, 5, 128, 300, tuple(range(0, 5000, 61)))])
def test_documents_equal_their_own_calls(B, T, H, D, W, starts):
    g = torch.Generator(device="cuda").manual_seed(T + H)
    q, k, v = (torch.randn(B, T, H, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    bounds = list(starts) + [T]
    doc = torch.cat([torch.full((b - a,), a, dtype=torch.int32, device="cuda") for a, b in zip(bounds, bounds[1:])])
    o, _ = ops.prefill_attention(q, k, v, window=W, doc_start=doc)
    for a, b in zip(bounds, bounds[1:]):
        ref, _ = ops.prefill_attention(q[:, a:b], k[:, a:b], v[:, a:b], window=W)
        # two bf16 roundings of the same sums over other tiles of keys, with bf16 probabilities
        assert ((o[:, a:b].float() - ref.float()).norm() / ref.float().norm()).item() < 1e-2


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H", [1, 2, 3, 4, 6, 12])
@pytest.mark.parametrize("B,T", [(1, 1), (2, 37), (1, 300)])
def test_rotated_keys_are_the_oracles_bits(D, H, B, T):
    """One, two and four heads a thread; counts of rows that leave surplus lanes in the last workgroup; keys at strides of their own."""
    q, k, v = _inputs(B, T, H, D, seed=H + T)
    cos, sin = oracle.rope_tables(D, T)
    kd = torch.zeros(B, T, H, D + 8, dtype=torch.bfloat16, device="cuda")[..., :D].copy_(k)
    _, kr = ops.prefill_attention(q.cuda(), kd, v.cuda(), window=None, cos=cos.cuda(), sin=sin.cuda())
    assert torch.equal(kr.cpu(), oracle.apply_rope(k, cos, sin))


@pytest.mark.parametrize("D,H,T,surplus", [(128, 12, 45, 0), (128, 12, 42, 1), (128, 12, 44, 2), (128, 12, 43, 3), (128, 3, 89, 1), (128, 3, 86, 3),
                                           (64, 12, 170, 0), (64, 12, 177, 1), (64, 12, 174, 2), (64, 12, 171, 3), (64, 6, 171, 3), (64, 1, 513, 3)])
@pytest.mark.parametrize("pad", [0, 8])
def test_keys_rotated_in_place(D, H, T, surplus, pad):
    """``k_out`` is ``k``: every row is rotated once, by the lanes that own it.  A lane takes 16 bytes of one, two or four heads; lengths that
    leave none to three whole wavefronts of the last workgroup without rows."""
    heads = 4 if D == 64 and H % 4 == 0 else 2 if H % 2 == 0 else 1
    assert -(T * H // heads * D // 8) % 256 // 64 == surplus
    q, k, v = _inputs(1, T, H, D, seed=T + H)
    cos, sin = oracle.rope_tables(D, T)
    kd = torch.zeros(1, T, H, D + pad, dtype=torch.bfloat16, device="cuda")[..., :D].copy_(k)
    o_ref, k_ref = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=None, cos=cos.cuda(), sin=sin.cuda())
    o, kr = ops.prefill_attention(q.cuda(), kd, v.cuda(), window=None, cos=cos.cuda(), sin=sin.cuda(), k_out=kd)
    assert kr.data_ptr() == kd.data_ptr()
    assert torch.equal(kr.cpu(), oracle.apply_rope(k, cos, sin)) and torch.equal(kr, k_ref) and torch.equal(o, o_ref)


@pytest.mark.parametrize("T,H,D,window,docs", [
    (4001, 5, 128, 200, 0), (4100, 3, 128, 1500, 0), (6500, 5, 64, 130, 0), (4224, 6, 128, 129, 0),   # runs of blocks, their remainder among them
    (2048, 15, 128, 300, 0), (2049, 15, 128, 300, 0), (2048, 16, 128, 600, 0), (5120, 8, 128, 2560, 0), (5121, 8, 128, 2560, 0),
    (7168, 8, 64, 200, 0), (7169, 8, 64, 200, 0), (3100, 13, 128, 200, 0), (5000, 13, 64, 700, 0), (2700, 12, 128, 1300, 0),
    (5120, 8, 128, None, 3), (8192, 8, 128, 4096, 3), (8193, 8, 128, 4096, 3), (5120, 8, 128, 1100, 3), (5121, 8, 128, 1100, 3),
    (5600, 16, 64, None, 3), (5633, 16, 64, None, 3),
    (7700, 13, 128, 200, 3), (7400, 14, 128, 200, 3), (12000, 12, 64, 1000, 3), (1000, 110, 128, 120, 3),      # eighths of a pair, with and without a remainder, none
])
def test_prefill_on_both_sides_of_the_block_size_rule(T, H, D, window, docs):
    """Sizes around the numbers of blocks at which the kernel with 32 queries per workgroup hands over to the one with 128, and pairs
    that are no multiple of eight; the first rows, some of every block and the last ones against the oracle."""
    q, k, v = _inputs(1, T, H, D, seed=T + H, normalise=True)
    doc_start = None
    if docs:
        ids = torch.ones(T, dtype=torch.long)
        ids[[T // 5, T // 2 + 3]] = 0
        doc_start = oracle.doc_start_from_ids(ids, 0)
    rows = torch.cat([torch.arange(0, T, 97), torch.arange(T - 3, T)]).unique()
    lo = torch.zeros(T, dtype=torch.long) if window is None else (torch.arange(T) - window + 1).clamp(min=0)
    if doc_start is not None:
        lo = torch.maximum(lo, doc_start.long())
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=window, doc_start=None if doc_start is None else doc_start.cuda())
    visible = (torch.arange(T)[None] <= rows[:, None]) & (torch.arange(T)[None] >= lo[rows][:, None])
    for h in range(0, H, max(H // 3, 1)):
        s = (q[0, rows, h].float() @ k[0, :, h].float().T * 0.12).masked_fill(~visible, float("-inf"))
        assert_close_bf16(o[0, rows.cuda(), h], s.softmax(-1) @ v[0, :, h].float(), f"o, head {h}")


@pytest.mark.parametrize("T,H,D,window,docs,split", [
    # no window
    (4096, 12, 128, None, 0, True), (4097, 12, 128, None, 0, False), (1000, 36, 128, None, 0, True), (1000, 37, 128, None, 0, False),
    (6144, 16, 64, None, 0, True), (6145, 16, 64, None, 0, False),
    # a window; with runs of blocks, their remainder among them; keys past an XCD's L2
    (4001, 5, 128, 800, 0, True), (4100, 3, 128, 1000, 0, True), (4300, 3, 128, 200, 0, True), (6500, 5, 64, 130, 0, True),
    (3328, 8, 128, 200, 0, True), (3329, 8, 128, 200, 0, False), (3072, 6, 128, 200, 0, True), (3073, 6, 128, 200, 0, False),
    (2048, 16, 128, 800, 0, True), (2049, 16, 128, 800, 0, False), (5120, 8, 128, 2560, 0, True), (5121, 8, 128, 2561, 0, False),
    (4096, 6, 128, 2000, 0, True), (4097, 6, 128, 2000, 0, False),
    (7168, 8, 64, 200, 0, True), (7169, 8, 64, 200, 0, False), (8192, 5, 64, 4000, 0, True), (8193, 5, 64, 4000, 0, False),
    (3100, 13, 128, 200, 0, False), (5000, 13, 64, 700, 0, False), (2700, 12, 128, 1300, 0, False), (2700, 12, 128, 1350, 0, True),
    # documents
    (4608, 8, 128, None, 3, True), (4609, 8, 128, None, 3, False), (4608, 8, 128, 1100, 3, True), (4609, 8, 128, 1100, 3, False),
    (3328, 8, 128, 800, 3, True), (3329, 8, 128, 800, 3, False), (3072, 6, 128, 200, 3, True), (3073, 6, 128, 200, 3, False),
    (4096, 6, 128, 2000, 3, True), (4097, 6, 128, 2000, 3, False), (4096, 7, 128, None, 3, True), (4097, 7, 128, None, 3, False),
    (3200, 20, 64, None, 3, True), (3201, 20, 64, None, 3, False), (7168, 8, 64, 700, 3, True), (7169, 8, 64, 700, 3, False),
    (8192, 5, 64, 700, 3, True), (8193, 5, 64, 700, 3, False), (11264, 5, 64, None, 3, True), (11265, 5, 64, None, 3, False),
    # eighths of a pair, with and without a remainder, none
    (7700, 13, 128, 200, 3, False), (7400, 14, 128, 200, 3, False), (12000, 12, 64, 1000, 3, False), (1000, 110, 128, 120, 3, False),
])
def test_prefill_block_size_rule_and_every_head(T, H, D, window, docs, split):
    """Sizes around the numbers of blocks at which the kernel with 32 queries per workgroup hands over to the one with 128 (the rule itself is
    asked which), and pairs that are no multiple of eight; the first rows, some of every block and the last ones against the oracle."""
    wanted = _lib.load()._ZN5daisy20prefill_split_wantedEiiiib
    wanted.restype = ctypes.c_bool
    assert wanted(H, T, D, window or 0, bool(docs)) == split
    q, k, v = _inputs(1, T, H, D, seed=T + H, normalise=True)
    doc_start = None
    if docs:
        ids = torch.ones(T, dtype=torch.long)
        ids[[T // 5, T // 2 + 3]] = 0
        doc_start = oracle.doc_start_from_ids(ids, 0)
    rows = torch.cat([torch.arange(0, T, 97), torch.arange(T - 3, T)]).unique()
    lo = torch.zeros(T, dtype=torch.long) if window is None else (torch.arange(T) - window + 1).clamp(min=0)
    if doc_start is not None:
        lo = torch.maximum(lo, doc_start.long())
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=window, doc_start=None if doc_start is None else doc_start.cuda())
    visible = (torch.arange(T)[None] <= rows[:, None]) & (torch.arange(T)[None] >= lo[rows][:, None])
    for h in range(H) if H <= 20 else (*range(8), *range(H - 8, H)):      # (every remainder by eight: the order of blocks depends on it)
        s = (q[0, rows, h].float() @ k[0, :, h].float().T * 0.12).masked_fill(~visible, float("-inf"))
        assert_close_bf16(o[0, rows.cuda(), h], s.softmax(-1) @ v[0, :, h].float(), f"o, head {h}")
