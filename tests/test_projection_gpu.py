"""The tiled projection kernel (``csrc/proj.hip``) at the edges of its tiles, with and without the QKV epilogue, and
the attention kernel for few query blocks around its tile edges and on both sides of the rule that picks it."""
import pytest
import torch

import oracle
from daisy_amd import CausalSelfAttention, WindowMask, _lib, ops
from tests.helpers import assert_close_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tile,K", [(0, 128), (1, 384), (2, 128), (3, 256), (4, 64), (5, 192), (6, 64), (7, 192)])
@pytest.mark.parametrize("M,N", [(1, 8), (31, 64), (33, 72), (127, 136), (129, 256), (257, 520)])
def test_tiles_against_fp64(tile, K, M, N):
    g = torch.Generator().manual_seed(M * 1000 + N)
    x, w, b = (torch.randn(*s, generator=g).bfloat16() for s in ((M, K), (N, K), (N,)))
    ref = x.double() @ w.double().t()
    xd = torch.zeros(M, K + 8, dtype=torch.bfloat16, device=DEV)[:, :K].copy_(x)      # rows at a stride of their own
    for bias in (None, b):
        y = _lib.native().linear(xd, w.to(DEV), None if bias is None else bias.to(DEV), 4, tile)
        if y is None:
            assert tile == 0 and M <= 4 or bias is not None     # the rule left the product to another kernel
            continue
        r = ref if bias is None else ref + bias.double()
        err = (y.cpu().double() - r).abs()
        assert (err <= r.abs() * 2 ** -8 + K ** 0.5 * 1e-5 + 1e-3).all(), err.max().item()


@pytest.mark.parametrize("tile,K", [(10, 128), (10, 640), (9, 256), (9, 512)])
@pytest.mark.parametrize("M,N", [(1, 8), (15, 32), (17, 40), (33, 200), (130, 72)])
def test_smallest_tiles_against_fp64(tile, K, M, N):
    """Remainders of tiles of 16 and 32 rows and 32 columns; fewer K steps than stages, and more."""
    test_tiles_against_fp64(tile, K, M, N)


@pytest.mark.parametrize("tile,bk,stages", [(1, 128, 3), (2, 128, 4), (3, 128, 3), (4, 64, 3), (5, 64, 4), (6, 64, 2), (9, 128, 4), (10, 128, 4)])
@pytest.mark.parametrize("more", [-2, -1, 0, 1, 2, 5])
def test_tiles_around_as_many_steps_as_stages_against_fp64(tile, bk, stages, more):
    """From fewer steps of K than there are stages, where every step is one of the last, to a few more, where stages are reused."""
    K = bk * max(stages + more, 1)
    test_tiles_against_fp64(tile, K, 70, 136)


@pytest.mark.parametrize("M", [2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("N,K", [(1024, 192), (2048, 64), (2056, 128), (5464, 128), (8200, 64), (16392, 72), (1024, 72)])
def test_few_rows_on_both_sides_of_the_rule_against_fp64(M, N, K):
    """Few rows on either side of the limit where the weight-streaming kernel hands over to the tiled one, and sizes that one refuses."""
    g = torch.Generator().manual_seed(M * N)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    with torch.no_grad():
        y = _lib.native().linear(x.to(DEV), w.to(DEV), None, 4, 0)
    assert (y is None) == (M > 4 and K % 64 != 0)
    if y is not None:
        r = x.double() @ w.double().t()
        err = (y.cpu().double() - r).abs()
        assert (err <= r.abs() * 2 ** -8 + K ** 0.5 * 1e-5 + 1e-3).all(), err.max().item()


@pytest.mark.parametrize("M", [5, 16, 17, 100, 128, 129, 200])
def test_products_on_both_sides_of_the_smallest_tiles_rule(M):
    """The rule by sizes gives the bits of the tiles it picks among (same order of the sums in all of them)."""
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, 512, generator=g, device=DEV).bfloat16()
    w = torch.randn(520, 512, generator=g, device=DEV).bfloat16()
    with torch.no_grad():
        y = _lib.native().linear(x, w, None, 4, 0)
        for tile in (1, 9, 10):
            assert torch.equal(y, _lib.native().linear(x, w, None, 4, tile))


@pytest.mark.parametrize("M,N,own", [(999, 6144, False), (1000, 6144, True), (6009, 1024, False), (6017, 1024, True), (8192, 1024, True), (8193, 1024, False)])
def test_large_products_on_both_sides_of_the_rule(M, N, own):
    """From 384 to 512 tiles of 128 x 128 and 1000 rows on; the few rows compared are the first, the last and some of every row of tiles."""
    K = 576
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    with torch.no_grad():
        y = _lib.native().linear(x.to(DEV), w.to(DEV), None, 4, 0)
    assert (y is not None) == own
    if own:
        rows = torch.cat([torch.arange(0, M, 61), torch.tensor([M - 1])])
        r = x[rows].double() @ w.double().t()
        err = (y[rows.to(DEV)].cpu().double() - r).abs()
        assert (err <= r.abs() * 2 ** -8 + K ** 0.5 * 1e-5 + 1e-3).all(), err.max().item()


@pytest.mark.parametrize("M,N,K,own", [(6017, 1024, 1024, True), (4608, 1536, 1088, False), (4609, 1536, 1088, True), (4609, 1536, 1536, True),
                                       (4609, 1536, 1600, False), (4096, 2048, 2048, False), (24576, 256, 1024, True), (49152, 128, 1024, False)])
def test_large_products_of_long_rows_and_one_column_of_tiles(M, N, K, own):
    """From 384 (rows of more than 1024: 440) to 512 tiles of 128 x 128, two columns of them and 1000 rows on; the few rows compared are the
    first, the last and some of every row of tiles."""
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    with torch.no_grad():
        y = _lib.native().linear(x.to(DEV), w.to(DEV), None, 4, 0)
    assert (y is not None) == own
    if own:
        rows = torch.cat([torch.arange(0, M, 61), torch.tensor([M - 1])])
        r = x[rows].double() @ w.double().t()
        err = (y[rows.to(DEV)].cpu().double() - r).abs()
        assert (err <= r.abs() * 2 ** -8 + K ** 0.5 * 1e-5 + 1e-3).all(), err.max().item()


@pytest.mark.parametrize("H,D", [(2, 128), (6, 64), (3, 64)])
@pytest.mark.parametrize("B,T", [(1, 5), (2, 64), (1, 129), (3, 200), (1, 1100)])
@pytest.mark.parametrize("ve", [False, True])
def test_layer_prefill_matches_the_oracle(H, D, B, T, ve):
    dim = H * D
    torch.manual_seed(T)
    attn = CausalSelfAttention(dim, H, D, receives_ve=ve, layer_idx=0, max_seq_len=T)
    with torch.no_grad():
        attn.qkvo_w.copy_((torch.randn(4, dim, dim) * 0.05).bfloat16())
    x, vals = torch.randn(B, T, dim).bfloat16(), torch.randn(B, T, dim).bfloat16()
    y_ref, k_ref, v_ref = oracle.attn_prefill(x, attn.qkvo_w.detach(), H, D, attn.rotary.cos, attn.rotary.sin, 70,
                                              ve=vals if ve else None, g_ve=0.3228 if ve else None)
    attn = attn.to(DEV).eval()
    with torch.no_grad():
        y, k, v = attn.prefill(x.to(DEV), vals.to(DEV) if ve else None, attn_mask=WindowMask(70), debug=True)
        assert attn.last_q is not None and attn.last_q.shape == (B, T, H, D)
        y2 = attn(x.to(DEV), vals.to(DEV) if ve else None, attn_mask=WindowMask(70))
    assert torch.equal(y, y2)                     # the output may or may not take the queries' place
    assert_close_bf16(k, k_ref, "k", max_abs=4e-2)
    assert_close_bf16(v, v_ref, "v", max_abs=4e-2)
    assert_close_bf16(y, y_ref, "y")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H", [(1, 1), (2, 4), (8, 33)])      # few blocks; few blocks in XCD groups; many blocks
@pytest.mark.parametrize("T,window,docs", [(1, None, False), (32, None, False), (33, 5, False), (127, 64, True), (161, None, True),
                                           (300, 33, False)])
def test_attention_on_both_sides_of_the_block_rule(D, B, H, T, window, docs):
    g = torch.Generator(device=DEV).manual_seed(T)
    q, k, v = (torch.randn(B, T, H, D, generator=g, device=DEV).bfloat16() for _ in range(3))
    doc = None
    if docs:
        doc = torch.zeros(T, dtype=torch.int32, device=DEV)
        doc[T // 3:] = T // 3
        doc[T - 2:] = T - 2
    o, _ = ops.prefill_attention(q, k, v, window=window, doc_start=doc)
    pos = torch.arange(T, device=DEV)
    lo = torch.zeros_like(pos) if window is None else (pos - window + 1).clamp_min(0)
    if doc is not None:
        lo = torch.maximum(lo, doc.long())
    seen = (pos[None, :] <= pos[:, None]) & (pos[None, :] >= lo[:, None])
    s = torch.matmul(q.float().transpose(1, 2), k.float().transpose(1, 2).transpose(2, 3).contiguous()) * 0.12
    p = s.masked_fill(~seen, float("-inf")).softmax(-1)
    ref = torch.matmul(p, v.float().transpose(1, 2).contiguous()).transpose(1, 2)
    assert_close_bf16(o, ref, f"o T={T}")


@pytest.mark.parametrize("D,B,H", [(64, 8, 33), (128, 7, 37)])       # many blocks, in XCD groups and not
@pytest.mark.parametrize("T,window", [(300, 64), (257, 40), (384, 383)])
def test_a_lone_document_changes_nothing_and_one_that_opens_with_the_last_row_only_that(D, B, H, T, window):
    g = torch.Generator(device=DEV).manual_seed(T)
    q, k, v = (torch.randn(B, T, H, D, generator=g, device=DEV).bfloat16() for _ in range(3))
    plain, _ = ops.prefill_attention(q, k, v, window=window)
    doc = torch.zeros(T, dtype=torch.int32, device=DEV)
    assert torch.equal(ops.prefill_attention(q, k, v, window=window, doc_start=doc)[0], plain)
    doc[-1] = T - 1
    o, _ = ops.prefill_attention(q, k, v, window=window, doc_start=doc)
    own = (T - 1) // 32 * 32               # the rows of the last row's wavefront share its rescaling, and with it their rounding:
    assert torch.equal(o[:, :own], plain[:, :own])
    want = torch.cat([plain[:, own:-1], v[:, -1:]], 1).float()       # bf16 weights (2^-9) on either side, two roundings of the outputs
    assert ((o[:, own:].float() - want).abs() <= 2.0 ** -7 * v.float().abs().max()).all()


def test_calls_that_something_intercepts_reach_the_library_op():
    """Tangents, subclasses, vmap and autocast of a decode batch's projection (64 rows: above the few-rows kernel)."""
    from daisy_amd.attention import step_linear
    g = torch.Generator().manual_seed(7)
    x, w, dx = (torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((64, 256), (512, 256), (64, 256)))
    with torch.no_grad():
        assert _lib.native().linear(x, w, None, 4, 0) is not None
        import torch.autograd.forward_ad as fwad
        with fwad.dual_level():
            y = fwad.unpack_dual(step_linear(fwad.make_dual(x, dx), w))
            assert torch.equal(y.tangent, torch.nn.functional.linear(dx, w))
        assert torch.equal(torch.vmap(lambda a: step_linear(a, w))(x[None]), torch.nn.functional.linear(x[None], w))

        class Sub(torch.Tensor):
            pass

        assert type(step_linear(x.as_subclass(Sub), w)) is Sub
        with torch.autocast("cuda", torch.float16):
            assert step_linear(x, w).dtype == torch.float16


@pytest.mark.parametrize("limit", [1, 4, 8])
@pytest.mark.parametrize("N,K", [(1024, 512), (4608, 512), (8200, 448)])
def test_the_limit_of_rows_chooses_the_kernel(N, K, limit):
    """Up to that many rows go to the weight-streaming kernel (a row's bits do not depend on how many there are), more to the tiled
    one, whatever the columns."""
    g = torch.Generator().manual_seed(N)
    x, w = torch.randn(9, K // 2, generator=g), torch.randn(N, K // 2, generator=g)
    # (sums that nearly cancel, so that their order shows in bf16)
    x, w = torch.cat([x, x], 1).bfloat16().to(DEV), torch.cat([w, 0.01 * torch.randn(N, K // 2, generator=g) - w], 1).bfloat16().to(DEV)
    with torch.no_grad():
        rows, tiled = ops.linear_rows(x[:8], w), _lib.native().linear(x, w, None, 4, 4)
        assert not torch.equal(rows, tiled[:8])            # (so that bits tell the kernels apart)
        for M in (1, 3, 4, 5, 8, 9):
            y = _lib.native().linear(x[:M], w, None, limit, 0)
            assert torch.equal(y, rows[:M] if M <= limit else tiled[:M]), M


def test_tiled_product_of_one_row_broadcast():
    x, w = torch.randn(1, 128, device=DEV).bfloat16(), torch.randn(1024, 128, device=DEV).bfloat16()
    with torch.no_grad():
        y = _lib.native().linear(x.expand(6, 128), w, None, 4, 0)
        assert torch.equal(y, _lib.native().linear(x.repeat(6, 1), w, None, 4, 0))
