"""Online-softmax stress for kernels 1 and 2: logits whose running row maximum moves a lot.

The ordinary parity cases use scale 0.12 on unit-variance inputs: scores a few log2 units wide, so the
rescale of the running sums almost never fires after a row's first tile.  Here scale = 1 and the keys are
built so that the score of a (query, key) pair grows (or falls) steadily with the key's position: the row
maximum rises tile after tile by a chosen amount -- 5, 12 or 40 log2 units: a prefill kernel moves its reference
when a lane's share of a tile's sum exceeds 2^12, some tiles late, about each, or in each (old contributions
scaled by ~2^-40); decode follows the maximum -- or sits in the first / last key a query
sees.  Checked against the fp32 oracle at the usual bf16 tolerances.
"""
import pytest
import torch

import oracle
from daisy_amd import ops
from helpers import assert_close_bf16, check_prefill_of_many_heads, say

pytestmark = pytest.mark.gpu

LOG2E = 1.4426950408889634


def _structured(B, T, H, D, rise_per_32_keys, seed, noise=0.3):
    """q, k, v [B, T, H, D] bf16 with  <q_i, k_j> ~= c * j  (+ noise of a few units), where c makes the score,
    in log2 units, move by `rise_per_32_keys` over 32 consecutive keys (negative: the score falls with j)."""
    g = torch.Generator().manual_seed(seed)
    u = torch.nn.functional.normalize(torch.randn(B, 1, H, D, generator=g), dim=-1)
    a = 4.0
    j = torch.arange(T, dtype=torch.float32).view(1, T, 1, 1)
    slope = rise_per_32_keys / 32.0 / LOG2E / a            # natural-log units per key, divided by |q . u|
    q = a * u + noise * torch.randn(B, T, H, D, generator=g)
    k = slope * j * u + noise * torch.randn(B, T, H, D, generator=g)
    v = torch.randn(B, T, H, D, generator=g)
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


def _random_large(B, T, H, D, seed):
    """q, k ~ 3 N(0,1) (scores hundreds of log2 units apart), v ~ N(0,1) (outputs of a size at which the rounding of
    the bf16 result itself stays well inside the tolerance)."""
    g = torch.Generator().manual_seed(seed)
    q, k = ((3.0 * torch.randn(B, T, H, D, generator=g)).bfloat16() for _ in range(2))
    return q, k, torch.randn(B, T, H, D, generator=g).bfloat16()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("window", [None, 200, 1])
@pytest.mark.parametrize("rise", [5.0, 12.0, 40.0, -12.0, -40.0, "random"])
def test_prefill_large_logits(D, window, rise):
    """T = 700: 5.5 query blocks, 22 key tiles; with window 200 the tile order is rotated (every block starts in
    the middle of its range and wraps), so a rising score puts the row maximum in a tile that is visited in the
    middle of the walk and a falling one in the tile visited right after the wrap.  Two heads run on the kernel for few query
    blocks, whose wavefronts take every fourth tile; the repeated heads on the one that walks all of them."""
    if window == 1 and rise not in (5.0, "random"):
        pytest.skip("one key per row: the structure does not matter")
    B, T, H = 1, 700, 2
    say(f"prefill large logits D{D} window {window} rise {rise}")
    q, k, v = _random_large(B, T, H, D, seed=D) if rise == "random" else _structured(B, T, H, D, rise, seed=D + 1)
    ref = oracle.windowed_attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), window, 1.0).transpose(1, 2)
    s = torch.einsum("bihd,bjhd->bhij", q.float(), k.float()) * LOG2E
    say(f"  score range in log2 units: {s.min().item():.0f} .. {s.max().item():.0f}")
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=window, scale=1.0)
    assert_close_bf16(o, ref, "o")
    check_prefill_of_many_heads(q.cuda(), k.cuda(), v.cuda(), ref, f"rise {rise}", window=window, scale=1.0)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("above", [11.0, 11.9, 12.1, 15.0, 140.0])
@pytest.mark.parametrize("at", [130, 400, 639])
def test_prefill_one_key_above_the_reference(D, above, at):
    """All scores 0 but those of one key, `above` log2 units higher for every third query (for the others lower): on either side of
    2^12, the share of a tile's sum that makes the reference move, and past what fp32 holds without it.  The key lies behind the tiles
    that set the references; a lane holds it alone in a tile, so that it is the sum."""
    T, H = 700, 2
    g = torch.Generator().manual_seed(D + at)
    q, k = torch.zeros(1, T, H, D), torch.zeros(1, T, H, D)
    q[..., 3] = torch.where(torch.arange(T) % 3 == 0, 4.0, -4.0).view(1, T, 1)
    k[:, at, :, 3] = above / LOG2E / 4.0
    q, k, v = q.bfloat16(), k.bfloat16(), torch.randn(1, T, H, D, generator=g).bfloat16()
    ref = oracle.windowed_attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), None, 1.0).transpose(1, 2)
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=None, scale=1.0)
    assert_close_bf16(o, ref, "o")
    check_prefill_of_many_heads(q.cuda(), k.cuda(), v.cuda(), ref, f"{above} above", window=None, scale=1.0)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("window", [None, 200])
@pytest.mark.parametrize("levels", [(0.0, 200.0, -200.0, 140.0, -140.0), (-300.0, 300.0, 0.0, -13.0, 11.0)])
def test_prefill_documents_that_start_inside_a_wavefront(D, window, levels):
    """Queries on both sides of a document's start in one wavefront: those behind it have no reference while the tiles of the document
    ahead pass, and get one at their first key, however far their scores (of one level per document, in log2 units) lie from 0."""
    T, H, starts = 700, 2, (0, 45, 333, 334, 499)
    g = torch.Generator().manual_seed(D)
    q, k = (0.3 * torch.randn(1, T, H, D, generator=g) for _ in range(2))
    q[..., 3] = 4.0
    doc_start = torch.zeros(T, dtype=torch.int32)
    for at, level in zip(starts, levels):
        k[:, at:, :, 3] = level / LOG2E / 4.0
        doc_start[at:] = at
    q, k, v = q.bfloat16(), k.bfloat16(), torch.randn(1, T, H, D, generator=g).bfloat16()
    ref = oracle.windowed_attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), window, 1.0, doc_start).transpose(1, 2)
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=window, scale=1.0, doc_start=doc_start.cuda())
    assert_close_bf16(o, ref, "o")
    check_prefill_of_many_heads(q.cuda(), k.cuda(), v.cuda(), ref, "documents", window=window, scale=1.0, doc_start=doc_start.cuda())


@pytest.mark.parametrize("D", [64, 128])
def test_prefill_large_logits_with_rotation_and_documents(D):
    """The same with RoPE in the call and document bounds (masked tiles take the same softmax path)."""
    B, T, H, W = 2, 515, 2, 300
    q, k, v = _random_large(B, T, H, D, seed=7 * D)
    cos, sin = oracle.rope_tables(D, T)
    doc_start = torch.zeros(T, dtype=torch.int32)
    doc_start[130:] = 130
    doc_start[401:] = 401
    qr, kr = oracle.apply_rope(q, cos, sin), oracle.apply_rope(k, cos, sin)
    ref = oracle.windowed_attention(qr.transpose(1, 2), kr.transpose(1, 2), v.transpose(1, 2), W, 1.0, doc_start).transpose(1, 2)
    o, _ = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), window=W, scale=1.0, cos=cos.cuda(), sin=sin.cuda(),
                                 doc_start=doc_start.cuda())
    assert_close_bf16(o, ref, "o")
    check_prefill_of_many_heads(q.cuda(), k.cuda(), v.cuda(), ref, "documents", window=W, scale=1.0, cos=cos.cuda(), sin=sin.cuda(),
                                doc_start=doc_start.cuda())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nsplit", [0, 1, 5])
@pytest.mark.parametrize("rise", [5.0, 12.0, 40.0, -40.0, "random"])
def test_decode_large_logits(D, nsplit, rise):
    """One query over a ring of 1000 rows whose scores rise / fall with the slot index (the kernel streams the ring
    in physical order, every lane group and every split keeps its own running maximum, and the merges across lane
    groups, wavefronts and splits see partial maxima that are far apart)."""
    B, H, W = 2, 3, 1000
    say(f"decode large logits D{D} nsplit {nsplit} rise {rise}")
    if rise == "random":
        _, kc, vc = _random_large(B, W, H, D, seed=D + 3)
        q = (3.0 * torch.randn(B, H, D, generator=torch.Generator().manual_seed(5))).bfloat16()
    else:
        q_all, kc, vc = _structured(B, W, H, D, rise, seed=D + 4)
        q = q_all[:, 0]
    kc, vc = kc.transpose(1, 2).contiguous(), vc.transpose(1, 2).contiguous()     # [B, H, W, D]
    g = torch.Generator().manual_seed(11)
    kn, vn = ((torch.randn(B, H, D, generator=g)).bfloat16() for _ in range(2))
    slot = 617
    k_exp, v_exp = kc.clone(), vc.clone()
    k_exp[:, :, slot], v_exp[:, :, slot] = kn, vn
    ref = oracle.sdpa(q[:, :, None], k_exp, v_exp, None, 1.0)[:, :, 0]
    o = ops.decode_attention(q.cuda(), kn.cuda(), vn.cuda(), kc.cuda(), vc.cuda(), n_rows=W, new_idx=slot,
                             write_back=True, scale=1.0, nsplit=nsplit)
    assert_close_bf16(o, ref, "o")
