"""What the modules hand to the one-call path (``daisy_amd/_native.so``) and which calls it serves."""
import ctypes
from ctypes import c_int, c_int64, c_void_p

import pytest
import torch

from daisy_amd import CausalSelfAttention, KimiLinearSelfAttention, KVCache, WindowMask, _lib, norm


class _Recorder:
    """Stands in for the extension: keeps the arguments and answers like it."""

    def __init__(self, answer):
        self.answer, self.args = answer, None

    def __getattr__(self, name):
        def call(*args):
            self.name, self.args = name, args
            return self.answer
        return call


def _attn(dim=128, H=2, D=64, ve=True, **kw):
    torch.manual_seed(0)
    return CausalSelfAttention(dim, H, D, receives_ve=ve, layer_idx=0, max_seq_len=64, **kw).eval()


@pytest.mark.parametrize("x_dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ve_dtype", [None, torch.float32, torch.bfloat16])
def test_activations_reach_the_one_call_path_in_the_weights_dtype(x_dtype, ve_dtype, monkeypatch):
    attn = _attn(ve=ve_dtype is not None)
    x = torch.randn(1, 5, 128).to(x_dtype)
    ve = None if ve_dtype is None else torch.randn(1, 5, 128).to(ve_dtype)
    kv = torch.zeros(1, 5, 2, 64)
    ext = _Recorder((x, None, kv, kv))
    monkeypatch.setattr(_lib, "native", lambda: ext)
    attn.prefill(x, ve, attn_mask=WindowMask(4))
    assert ext.name == "layer_prefill" and ext.args[0].dtype == torch.bfloat16 and torch.equal(ext.args[0], x.bfloat16())
    got_ve = ext.args[8]
    assert got_ve is None if ve is None else got_ve.dtype == torch.bfloat16 and torch.equal(got_ve, ve.bfloat16())
    cache = KVCache(L=1, B=1, H=2, W=8, D=64, device="cpu", dtype=torch.bfloat16)
    ext.answer = (x, None, None)
    one = None if ve is None else ve[:, :1]
    attn.step(x[:, :1], cache.ring(0), cache.ring(0), 0, one, 8)
    assert ext.name == "layer_step" and ext.args[0].dtype == torch.bfloat16
    assert ext.args[7] is None if ve is None else ext.args[7].dtype == torch.bfloat16


@pytest.mark.parametrize("debug", [False, True, 0, 1, "yes"])
def test_debug_taps_are_asked_for_by_truth(debug, monkeypatch):
    """The extension looks for True itself: any other true value used to leave ``last_q`` empty."""
    attn, kv = _attn(ve=False), torch.zeros(1, 5, 2, 64)
    ext = _Recorder((kv, kv, kv, kv))
    monkeypatch.setattr(_lib, "native", lambda: ext)
    attn.prefill(torch.randn(1, 5, 128), None, attn_mask=WindowMask(4), debug=debug)
    assert ext.args[15] is bool(debug)


@pytest.mark.gpu
@pytest.mark.parametrize("ve", [False, True])
def test_fp32_activations_equal_the_bf16_ones_they_round_to(ve, monkeypatch):
    attn = _attn(ve=ve).to("cuda:0")
    with torch.no_grad():
        attn.qkvo_w.normal_(std=0.05)
    g = torch.Generator(device="cuda:0").manual_seed(1)
    x, vals = (torch.randn(2, 33, 128, generator=g, device="cuda:0") for _ in range(2))
    served = []

    class Spy:
        def __getattr__(self, name):
            return lambda *a: served.append(getattr(ext, name)(*a)) or served[-1]

    ext = _lib.native()
    monkeypatch.setattr(_lib, "native", Spy)
    outs = []
    with torch.no_grad():
        for xs, vs in ((x, vals), (x.bfloat16(), vals.bfloat16())):
            cache = KVCache(L=1, B=2, H=2, W=16, D=64, device="cuda:0", dtype=torch.bfloat16)
            y, k, v = attn.prefill(xs, vs if ve else None, attn_mask=WindowMask(7))
            s, _, _ = attn.step(xs[:, :1].contiguous(), cache.ring(0), cache.ring(0), 0, vs[:, :1].contiguous() if ve else None, 16)
            outs.append((y, k, v, s, cache.k, cache.v))
    assert len(served) == 4 and all(r is not None for r in served)
    for a, b in zip(*outs):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
@torch.no_grad()
def test_shapes_that_the_kernels_functions_refuse_are_refused_in_one_call_too():
    attn = _attn(ve=False).to("cuda:0")
    x = torch.randn(1, 9, 128, device="cuda:0").bfloat16()
    bounds = torch.zeros(9, dtype=torch.int32, device="cuda:0")
    attn.prefill(x, None, attn_mask=WindowMask(4, bounds))
    for bad in (bounds[None], bounds[:, None], bounds[:8], bounds.long()):
        with pytest.raises(ValueError, match="doc_start"):
            attn.prefill(x, None, attn_mask=WindowMask(4, bad))
    layer = KimiLinearSelfAttention(128, 2, max_seq_len=16, head_dim=64).to("cuda:0").eval()
    for call in (lambda: layer.prefill(x, None), lambda: layer.step(x[:, :1], None, None, 9, None, None)):
        layer.reset_history()
        layer.prefill(x, None)
        layer._conv_state = tuple(w.transpose(1, 2).contiguous() for w in layer._conv_state)
        with pytest.raises(ValueError, match="cache must be"):
            call()


class _Segment(ctypes.Structure):
    _fields_ = [("x", c_void_p), ("x_sm", c_int64), ("w", c_void_p), ("w_sn", c_int64), ("bias", c_void_p), ("y", c_void_p),
                ("y_sm", c_int64), ("N", c_int), ("tile_end", c_int)]


class _Gates(ctypes.Structure):
    _fields_ = [("A_log", c_void_p), ("dt_bias", c_void_p), ("H", c_int), ("Dk", c_int), ("logits", c_void_p),
                ("logits_row", c_int64), ("beta", c_void_p)]


@pytest.mark.parametrize("tile,K", [(7, 128), (8, 128), (1, 64)])
def test_a_forced_tile_that_does_not_serve_a_gated_product_is_refused(tile, K):
    """Not replaced by another: refused ahead of any launch (an internal function of the library, called by its C++ name)."""
    lib = _lib.load()
    fn = lib._ZN5daisy13proj_segmentsEPKNS_11ProjSegmentEiiiP12ihipStream_tiPKNS_8KdaGatesE
    fn.argtypes = [c_void_p, c_int, c_int, c_int, c_void_p, c_int, c_void_p]
    p = (ctypes.addressof(ctypes.create_string_buffer(64)) + 15) // 16 * 16        # (never read)
    seg, gates = _Segment(p, K, p, K, None, p, 128, 128, 0), _Gates(p, p, 2, 64, p, 8, p)
    assert fn(ctypes.byref(seg), 1, 4, K, None, tile, ctypes.byref(gates)) == -2
    assert "tile" in lib.daisy_last_error().decode()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,widths", [(1, 64, (13,)), (127, 128, (128, 128, 16)), (129, 192, (64, 5, 8, 3, 100, 72)), (300, 256, (256, 32)), (24001, 1024, (64, 20, 8))])
def test_narrow_products_in_one_tile_across(M, K, widths):
    """One tile for all columns (code 12) against tiles of 128 x 128 (6), which sum over K in the same order: the same bits; by rule at
    24001 rows; nothing behind a product's rows or columns is written.  Products that one tile does not hold are refused."""
    lib = _lib.load()
    fn = lib._ZN5daisy13proj_segmentsEPKNS_11ProjSegmentEiiiP12ihipStream_tiPKNS_8KdaGatesE
    fn.argtypes = [c_void_p, c_int, c_int, c_int, c_void_p, c_int, c_void_p]
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = [torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in widths]

    def call(tile, bias=None):
        y = [torch.full((M + 1, (n + 7) // 8 * 8 + 8), 7.0, dtype=torch.bfloat16, device="cuda") for n in widths]
        segs = (_Segment * len(widths))(*(_Segment(x.data_ptr(), K + 8, a.data_ptr(), K, bias, b.data_ptr(), b.shape[1], n, 0)
                                          for a, b, n in zip(w, y, widths)))
        return fn(ctypes.addressof(segs), len(widths), M, K, torch.cuda.current_stream().cuda_stream, tile, None), y

    results = [call(tile) for tile in (12, 6, 0)]
    assert [rc for rc, _ in results] == [0, 0, 0]
    for i, n in enumerate(widths):
        assert all(torch.equal(y[i][:M, :n], results[1][1][i][:M, :n]) for _, y in results)
        assert all((y[i][M] == 7).all() and (y[i][:, (n + 7) // 8 * 8:] == 7).all() for _, y in results)
        ref = x.float() @ w[i].float().T
        assert (results[0][1][i][:M, :n] - ref).abs().max() <= 2 ** -8 * ref.abs().max()
    assert call(12, bias=w[0].data_ptr())[0] == -2
    widths = (128, 128, 40)
    w = [torch.zeros(n, K, dtype=torch.bfloat16, device="cuda") for n in widths]
    assert call(12)[0] == -2


class _Normed(torch.nn.Module):
    def forward(self, x):
        return norm(x)


@pytest.mark.parametrize("record", [torch.fx.symbolic_trace, torch.jit.script], ids=["symbolic_trace", "script"])
@pytest.mark.parametrize("of", ["function", "module"])
def test_norm_is_recorded_as_the_librarys_call(record, of):
    """A stand-in for a tensor has no device and no dtype to ask for, and a script no extension to call."""
    recorded = record(norm if of == "function" else _Normed())
    assert "rms_norm" in str(getattr(recorded, "inlined_graph", recorded.graph))
    for x in (torch.randn(3, 24), torch.randn(2, 1, 40).bfloat16()):
        assert torch.equal(recorded(x), torch.nn.functional.rms_norm(x, (x.size(-1),)))


@pytest.mark.parametrize("groups", [1, 2, 5, 8, 10, 16, 40, 95, 96, 97, 768, 769, 800, 4000])
def test_low_rank_products_always_have_workgroups(groups):
    """Whole eights, one per XCD; of more groups of columns than fit the chip too."""
    fn = _lib.load()._ZN5daisy16low_rank_walkersEii
    for M in (1, 64, 65, 1000, 40000):
        walkers = fn(M, groups)
        assert walkers >= 8 and walkers % 8 == 0 and walkers * groups * 256 < 2 ** 31
        assert walkers <= (M + 511) // 512 * 8


def test_low_rank_products_walk_in_one_round():
    """Heads whose number does not divide 96: of 768 places no more workgroups than fit, where that fills five sixths of them."""
    fn = _lib.load()._ZN5daisy16low_rank_walkersEii
    for groups in range(1, 97):
        whole = 768 // groups // 8 * 8
        walkers = fn(1 << 20, groups)
        assert walkers == whole if whole * groups > 640 else whole <= walkers <= whole + 8
    assert [fn(40000, n) * n for n in (5, 7, 8, 10, 14, 16)] == [760, 728, 768, 720, 672, 768]


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,H,Dk", [(1, 64, 3, 64), (15, 128, 2, 128), (16, 64, 16, 40), (17, 128, 5, 8), (129, 64, 4, 128), (70, 64, 800, 128),
                                      (2100, 128, 10, 64)])
@pytest.mark.parametrize("bias", [False, True])
def test_low_rank_products_with_what_follows_them(M, K, H, Dk, bias):
    """The decay gate with beta, and the gated norm: rows that end inside a block of 16, columns inside a group of 128, more groups of columns
    than workgroups fit the chip.  Against 64 bits: one rounding of the product to bf16, one of the result; nothing behind the rows is written."""
    lib = _lib.load()
    gate = lib._ZN5daisy13low_rank_gateEPKtlS1_RKNS_8KdaGatesEPtiiiP12ihipStream_t
    gate.argtypes = [c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p]
    norm_of = lib._ZN5daisy13low_rank_normEPKtlS1_S1_S1_PtfiiiP12ihipStream_t
    norm_of.argtypes = [c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_void_p, ctypes.c_float, c_int, c_int, c_int, c_void_p]
    g = torch.Generator(device="cuda").manual_seed(M + H)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    # (u: half the spacing of bf16 numbers, 7 bits behind the first)
    stream, u, x = torch.cuda.current_stream().cuda_stream, 2.0 ** -8, rnd(M, K + 16).bfloat16()

    def product(w, b):                                       # in 64 bits, and how far its bf16 value may be from it
        z, size = x[:, :K].double() @ w.double().T + b, x[:, :K].double().abs() @ w.double().abs().T + abs(b)
        return z, u * z.abs() + K * 2.0 ** -24 * size

    w, logits = (rnd(H * Dk, K) / K ** 0.5).bfloat16(), rnd(M, (H + 7) // 8 * 8).bfloat16()
    A_log, dt_bias, beta = rnd(H), rnd(H * Dk), torch.full((M + 1, H), 7.0, device="cuda")
    y = torch.full((M + 1, H * Dk), 7.0, device="cuda").bfloat16()
    gates = _Gates(A_log.data_ptr(), dt_bias.data_ptr(), H, Dk, logits.data_ptr(), logits.shape[1], beta.data_ptr())
    assert gate(x.data_ptr(), K + 16, w.data_ptr(), ctypes.addressof(gates), y.data_ptr(), M, H * Dk, K, stream) == 0, lib.daisy_last_error()
    z, dz = product(w, 0.0)
    scale = A_log.double().exp().repeat_interleave(Dk)
    ref = -scale * torch.nn.functional.softplus(z + dt_bias.double())
    assert ((y[:M] - ref).abs() - (scale * dz + (u + 1e-5) * ref.abs()) * 1.01).max() <= 0   # (the gate's slope is at most its scale)
    ref = logits[:, :H].double().sigmoid()
    assert ((beta[:M] - ref).abs() - (u + 1e-5) * ref).max() <= 0
    assert (y[M] == 7).all() and (beta[M] == 7).all()

    w, weight, b = (rnd(H * K, K) / K ** 0.5).bfloat16(), rnd(K).bfloat16(), rnd(H * K).bfloat16() if bias else None
    o = torch.full((M + 1, H * K), 7.0, device="cuda").bfloat16()
    o[:M] = rnd(M, H * K)
    before = o[:M].double().view(M, H, K)
    assert norm_of(x.data_ptr(), K + 16, w.data_ptr(), b.data_ptr() if bias else None, weight.data_ptr(), o.data_ptr(), 1e-5, M, H * K, K, stream) == 0
    z, dz = product(w, b.double() if bias else 0.0)
    rows = (before * (before.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt() * weight.double()).view(M, H * K)
    ref = rows * z.sigmoid()
    assert ((o[:M] - ref).abs() - (rows.abs() * dz / 4 + (u + 1e-5) * ref.abs()) * 1.01).max() <= 0   # (the sigmoid's slope is at most 1 / 4)
    assert (o[M] == 7).all()
