"""Chunked KDA at the edges of its tiling: chunks of 32 positions, key widths of 64 and 128 channels, groups
of 32 value columns, and keys that overlap so strongly that the triangle's inverse carries the result."""
import pytest
import torch
import torch.nn.functional as F

import oracle
from daisy_amd import _lib, chunk_kda
from helpers import assert_close_bf16

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, Dk, Dv, seed, overlap=0.0):
    g = torch.Generator().manual_seed(seed)
    q, k = (F.normalize(torch.randn(B, T, H, Dk, generator=g), dim=-1) for _ in range(2))
    k = F.normalize((1 - overlap) * k + overlap * k[:, :1], dim=-1)
    v = torch.randn(B, T, H, Dv, generator=g)
    gl = F.logsigmoid(torch.randn(B, T, H, Dk, generator=g) + 3 * overlap)
    beta = torch.sigmoid(torch.randn(B, T, H, generator=g) + 3 * overlap)
    return q.bfloat16(), k.bfloat16(), v.bfloat16(), gl, beta


def _run(q, k, v, gl, beta, **kw):
    o, S = chunk_kda(q.cuda(), k.cuda(), v.cuda(), gl.cuda(), beta.cuda(), output_final_state=True, use_qk_l2norm_in_kernel=True, **kw)
    return o.cpu(), S.cpu()


@pytest.mark.parametrize("Dk,Dv", [(64, 32), (72, 40), (128, 128)])
@pytest.mark.parametrize("T", [1, 16, 31, 32, 33, 63, 65, 96, 97, 161])
def test_kda_chunk_edges(T, Dk, Dv):
    q, k, v, gl, beta = _inputs(2, T, 2, Dk, Dv, seed=T + Dk)
    o_ref, S_ref = oracle.kda_recurrent(q, k, v, gl, beta)
    o, S = _run(q, k, v, gl, beta)
    assert_close_bf16(o, o_ref, "o")
    assert ((S - S_ref).norm() / S_ref.norm()).item() <= 1e-3


@pytest.mark.parametrize("decay", [3.0, 6.0, 9.0, 13.0, 22.0, 60.0])
def test_kda_decays_around_the_limits(decay):
    """Per-row decays whose sums over 16, 8 and 4 rows fall on either side of exp(-80)."""
    q, k, v, _, beta = _inputs(1, 96, 2, 128, 32, seed=4)
    g = torch.Generator().manual_seed(9)
    gl = -decay * (0.5 + torch.rand(1, 96, 2, 128, generator=g)) * torch.rand(1, 1, 2, 128, generator=g).round()
    o_ref, S_ref = oracle.kda_recurrent(q, k, v, gl, beta)
    o, S = _run(q, k, v, gl, beta)
    assert_close_bf16(o, o_ref, "o")
    assert ((S - S_ref).norm() / S_ref.norm()).item() <= 1e-3


@pytest.mark.parametrize("overlap", [0.5, 0.9])
def test_kda_overlapping_keys(overlap):
    q, k, v, gl, beta = _inputs(1, 160, 2, 128, 64, seed=3, overlap=overlap)
    o_ref, S_ref = oracle.kda_recurrent(q, k, v, gl, beta)
    o, S = _run(q, k, v, gl, beta)
    assert_close_bf16(o, o_ref, "o")
    assert ((S - S_ref).norm() / S_ref.norm()).item() <= 1e-3


# 64 sequences: the most that a wavefront looks up by itself; 65 and more: from a table.  `behind`: rows after the last sequence.
@pytest.mark.parametrize("lengths,behind", [((1, 31, 0, 32, 33, 64, 5), 0), ((97,), 3), ((32, 32), 65), ((3, 0, 33) * 21 + (1,), 7),
                                            ((3, 0, 33) * 21 + (1, 40), 7), ((2,) * 130, 0)])
def test_kda_packed_chunk_slots(lengths, behind):
    q, k, v, gl, beta = _inputs(1, sum(lengths) + behind, 3, 64, 64, seed=sum(lengths))
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    torch.full((sum(lengths) + behind, 3, 64), float("nan"), dtype=torch.bfloat16, device="cuda")     # (what fresh memory may hold)
    o, S = _run(q, k, v, gl, beta, cu_seqlens=cu.cuda())
    assert not o[:, sum(lengths):].any()
    for i, n in enumerate(lengths):
        a = int(cu[i])
        if n == 0:
            continue
        o_ref, S_ref = oracle.kda_recurrent(*(t[:, a:a + n] for t in (q, k, v, gl, beta)))
        assert_close_bf16(o[:, a:a + n], o_ref, f"sequence {i}: o")
        assert ((S[i:i + 1] - S_ref).norm() / S_ref.norm()).item() <= 1e-3


# Blocks of the workspace (37 KiB per chunk and head, 21 for up to 64 key channels) beyond 128 MB are stored past the caches.  Heads are
# independent: the same bits as from calls on the other side of the line.
@pytest.mark.parametrize("T,H,Dk", [(3712, 32, 128), (8200, 48, 128), (6560, 48, 64)])
def test_kda_workspace_sizes_agree(T, H, Dk):
    assert (T + 31) // 32 * H * (37 if Dk > 64 else 21) * 1024 > (400 << 20 if T > 8000 else 128 << 20)
    assert (H + 7) // 8 * 8 * 4 >= 192 or T < 4000      # (four groups of value columns per head)
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(1, T, H, d, generator=g, device="cuda").bfloat16() for d in (Dk, Dk, 128))
    gl = F.logsigmoid(torch.randn(1, T, H, Dk, generator=g, device="cuda"))
    beta = torch.sigmoid(torch.randn(1, T, H, generator=g, device="cuda"))
    kw = dict(output_final_state=True, use_qk_l2norm_in_kernel=True)
    o, S = chunk_kda(q, k, v, gl, beta, **kw)
    for h in range(0, H, 8):
        part = [t[:, :, h:h + 8].contiguous() for t in (q, k, v, gl, beta)]
        o8, S8 = chunk_kda(*part, **kw)
        assert torch.equal(o[:, :, h:h + 8], o8) and torch.equal(S[:, h:h + 8], S8)


# More chains than compute units: packed sequences start longest first (a lane per sequence, few enough of them for their rows), unless they
# are in that order.  Each one's rows and states are those of a call of its own, from a state of its own.
@pytest.mark.parametrize("lengths", [(40, 33, 512, 0, 512, 130), (600, 300, 300, 20, 1), (1, 31, 700, 64, 65, 64, 1000, 0)])
@pytest.mark.parametrize("D", [64, 128])
def test_kda_packed_longest_first(lengths, D):
    H, n, T = 16, len(lengths), sum(lengths)
    q, k, v, gl, beta = _inputs(1, T + 5, H, D, 128, seed=T)
    s0 = torch.randn(n, H, D, 128, generator=torch.Generator().manual_seed(n))
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    assert n * H * 4 > 256 and T // 32 + n >= n * n
    o, S = _run(q, k, v, gl, beta, cu_seqlens=cu.cuda(), initial_state=s0.cuda())
    assert not o[:, T:].any()
    for i, m in enumerate(lengths):
        if m == 0:
            assert torch.equal(S[i], s0[i])
            continue
        o1, S1 = _run(*(t[:, cu[i]:cu[i] + m].contiguous() for t in (q, k, v, gl, beta)), initial_state=s0[i:i + 1].cuda())
        assert torch.equal(o[:, cu[i]:cu[i] + m], o1) and torch.equal(S[i:i + 1], S1)


# More groups of 32 value columns than compute units: groups of 64, whole ones, with a dead half, and with columns that end inside a
# half.  Sequences are independent: the same bits as from a call of one of them, in groups of 32.
@pytest.mark.parametrize("B,T,H,Dk,Dv", [(40, 33, 8, 64, 40), (9, 97, 16, 128, 96), (33, 1, 8, 72, 64), (17, 160, 8, 128, 72), (12, 129, 12, 64, 128)])
def test_kda_wide_column_groups(B, T, H, Dk, Dv):
    assert B * H * ((Dv + 31) // 32) > 256 >= (H + 7) // 8 * 8 * ((Dv + 31) // 32)
    q, k, v, gl, beta = _inputs(B, T, H, Dk, Dv, seed=B + T)
    s0 = torch.randn(B, H, Dk, Dv, generator=torch.Generator().manual_seed(B))
    o, S = _run(q, k, v, gl, beta, initial_state=s0.cuda())
    for b in (0, B // 2, B - 1):
        part = [t[b:b + 1].contiguous() for t in (q, k, v, gl, beta)]
        o1, S1 = _run(*part, initial_state=s0[b:b + 1].cuda())
        assert torch.equal(o[b:b + 1], o1) and torch.equal(S[b:b + 1], S1)
    o_ref, S_ref = oracle.kda_recurrent(*part, initial_state=s0[B - 1:])
    assert_close_bf16(o[B - 1:], o_ref, "o")
    assert ((S[B - 1:] - S_ref).norm() / S_ref.norm()).item() <= 1e-3


# Groups of 64 where they take fewer rounds of 256 workgroups than groups of 32, and as many rounds because of a dead half.
@pytest.mark.parametrize("B,T,H,Dk,Dv,wide", [(40, 33, 8, 64, 40, True), (11, 97, 16, 128, 96, True), (22, 160, 8, 128, 72, True), (17, 160, 8, 128, 72, False),
                                              (9, 97, 16, 128, 96, False), (6, 65, 16, 64, 160, False)])
def test_kda_column_groups_by_rounds(B, T, H, Dk, Dv, wide):
    assert ((B * H * ((Dv + 63) // 64) + 255) // 256 < (B * H * ((Dv + 31) // 32) + 255) // 256) == wide
    test_kda_wide_column_groups(B, T, H, Dk, Dv)


# ... of which there are more than compute units too: packed sequences start longest first.
@pytest.mark.parametrize("D,Dv", [(64, 128), (128, 96)])
def test_kda_packed_wide_column_groups_longest_first(D, Dv):
    lengths, H = (40, 33, 512, 0, 512, 130, 700, 64, 513), 16
    n, T = len(lengths), sum(lengths)
    assert n * H * ((Dv + 63) // 64) > 256 and T // 32 + n >= n * n
    q, k, v, gl, beta = _inputs(1, T + 5, H, D, Dv, seed=T)
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    torch.full((T + 5, H, Dv), float("nan"), dtype=torch.bfloat16, device="cuda")
    o, S = _run(q, k, v, gl, beta, cu_seqlens=cu.cuda())
    assert not o[:, T:].any()
    for i, m in enumerate(lengths):
        if m:
            o1, S1 = _run(*(t[:, cu[i]:cu[i] + m].contiguous() for t in (q, k, v, gl, beta)))
            assert torch.equal(o[:, cu[i]:cu[i] + m], o1) and torch.equal(S[i:i + 1], S1)


# Packed sequences of more groups of 32 than compute units, of both shapes that the kernel chooses from on the device, 64 columns (chains of like
# lengths) and 32 (a long one); ranked by length and not; ends at whole groups of 64 or not, narrow heads (32 always).
@pytest.mark.parametrize("H,D,Dv", [(16, 128, 128), (16, 128, 96), (16, 64, 128), (32, 104, 64)])
@pytest.mark.parametrize("lengths", [(40, 33, 512, 0, 512, 130, 700, 64, 513), (300, 290, 310, 250, 333, 301, 280, 299), (33, 64, 2000, 5, 31, 0, 90, 7, 160),
                                     (1, 32, 33) * 5, (900, *(20,) * 40)])
def test_kda_packed_wide_column_groups(lengths, H, D, Dv):
    n, T = len(lengths), sum(lengths)
    assert n * H * ((Dv + 31) // 32) > 256
    q, k, v, gl, beta = _inputs(1, T + 5, H, D, Dv, seed=T)
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    torch.full((T + 5, H, Dv), float("nan"), dtype=torch.bfloat16, device="cuda")
    o, S = _run(q, k, v, gl, beta, cu_seqlens=cu.cuda())
    assert not o[:, T:].any()
    for i, m in enumerate(lengths):
        if m:
            o1, S1 = _run(*(t[:, cu[i]:cu[i] + m].contiguous() for t in (q, k, v, gl, beta)))
            assert torch.equal(o[:, cu[i]:cu[i] + m], o1) and torch.equal(S[i:i + 1], S1)
        else:
            assert not S[i].any()


# ... of one to one and a half rounds, where the 256th and 257th longest chain decide too: alike, all but one alike, one long.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lengths", [(300, 310, 290, 305, 333, 300, 281, 299, 320), (300,) * 4 + (7,) + (410,) * 4, (90, 0, 150, 2000, 33, 64, 100, 31, 160)])
def test_kda_packed_wide_column_groups_of_two_rounds(lengths, D):
    assert 256 < len(lengths) * 16 * 2 <= 384 and sum((m + 31) // 32 for m in lengths) >= len(lengths) ** 2
    test_kda_packed_wide_column_groups(lengths, 16, D, 64)


# The blocks themselves, all of their bytes, from call to call: a 16-byte store's data registers written again by the next instruction
# changed the low terms of rows 28 .. 31 of M in 2 % of the blocks, which only those of the last chunk show in a result, and by an ulp.
@pytest.mark.parametrize("T,H,D", [(3712, 8, 128), (3712, 12, 64)])
def test_kda_blocks_are_the_same_in_every_call(T, H, D):
    lib = _lib.load()
    q, k, v, gl, beta = (t.cuda() for t in _inputs(1, T, H, D, D, seed=T))
    n = lib.daisy_kda_workspace_bytes(1, T, H, D, D, 64)
    blocks = [torch.zeros(n, dtype=torch.uint8, device="cuda") for _ in range(4)]
    o, S = torch.empty(1, T, H, D, dtype=torch.bfloat16, device="cuda"), torch.empty(1, H, D, D, device="cuda")
    assert q.dtype == torch.bfloat16 and gl.dtype == beta.dtype == torch.float32 and all(t.is_contiguous() for t in (q, k, v, gl, beta))
    for ws in blocks:
        assert lib.daisy_kda_chunk_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), gl.data_ptr(), 0, beta.data_ptr(), None, o.data_ptr(), S.data_ptr(),
                                       1, T, H, D, D, 64, D ** -0.5, 1, 1e-6, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream) == 0
    assert blocks[0].any() and all(torch.equal(ws, blocks[0]) for ws in blocks[1:])


# One key channel carries everything and decays by a step whose factor two bf16 terms hold worst (2^-18 off, the same way in every
# link), beta = -2: errors of A add up over the links of the triangle's inverse.  Eight other channels make the block steep.  What every
# block leaves: three splits in two terms and a dropped product of the lower ones, 2^-18 each, and fp32's roundings over 16 links.
# Blocks whose steep rows lie eight apart have A's operands in two terms too: three times 2^-18 in each link.
FP32_LINKS, TWO_TERM_LINKS = 4 * 2 ** -18 + 16 * 2 ** -22, 4 * 2 ** -18 + 16 * 3 * 2 ** -18


@pytest.mark.parametrize("Dk", [64, 128])
@pytest.mark.parametrize("steep,bound", [
    (lambda g: g.fill_(-25.), FP32_LINKS),              # every group of four rows beyond exp(-80)
    (lambda g: g[:, 0].fill_(-100.), FP32_LINKS),       # the first row alone
    (lambda g: g[:, 6].fill_(-100.), FP32_LINKS),
    (lambda g: g[:, 15].fill_(-100.), FP32_LINKS),      # the last one, on no side of any difference of the block
    (lambda g: g.fill_(-12.), TWO_TERM_LINKS),          # eight rows beyond it, four not
], ids=["all", "first", "one", "last", "eight"])
def test_kda_steep_blocks_against_fp64(Dk, steep, bound):
    q, k, v, _, _ = _inputs(1, 16, 2, Dk, 32, seed=Dk)
    k.zero_()[..., 0] = 1
    gl = torch.zeros(1, 16, 2, Dk)
    gl[..., 0] = -0.2197265625
    steep(gl[..., -8:])
    beta = torch.full((1, 16, 2), -2.)
    _, S_ref = oracle.kda_recurrent(q, k, v, gl, beta, use_qk_l2norm=False, dtype=torch.float64)
    _, S = chunk_kda(q.cuda(), k.cuda(), v.cuda(), gl.cuda(), beta.cuda(), output_final_state=True)
    err = ((S.cpu().double() - S_ref).norm() / S_ref.norm()).item()
    print(f"state error {err:.2e} of {bound:.2e}")
    assert err <= bound


# A log-decay of minus infinity forgets its channel.  Rows at either side of the blocks of 16 and the chunks of 32.
@pytest.mark.parametrize("Dk", [64, 128])
@pytest.mark.parametrize("rows", [(31,), (0,), (15, 16), (32, 63), (5, 6, 40), (62, 63)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_kda_infinite_decays(Dk, rows, dtype):
    for T in (32, 64):
        at = [r for r in rows if r < T]
        if not at:
            continue
        q, k, v, gl, beta = _inputs(1, T, 2, Dk, 32, seed=T + rows[0])
        gl = gl.to(dtype)
        gl[:, at, 0, ::3] = -torch.inf       # a third of the channels of one head, all of the other
        gl[:, at, 1] = -torch.inf
        o_ref, S_ref = oracle.kda_recurrent(q, k, v, gl, beta)
        o, S = _run(q, k, v, gl, beta)
        assert_close_bf16(o, o_ref, f"T = {T}: o")
        assert ((S - S_ref).norm() / S_ref.norm()).item() <= 1e-3
    gl[:, T // 2, 0, 0] = torch.nan          # not taken for a decay
    assert _run(q, k, v, gl, beta)[1][:, 0].isnan().any()
