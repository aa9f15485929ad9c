"""The KDA layer's one-call path against the layer's own Python path (the same kernels one by one), and the products that share a
launch against separate ones."""
import ctypes

import pytest
import torch

from daisy_amd import KimiLinearSelfAttention, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(H, D, expand_v, taps, conv_bias, dim=None):
    torch.manual_seed(H * D + taps)
    with torch.device(DEV):
        m = KimiLinearSelfAttention(dim or H * D, H, max_seq_len=1024, head_dim=D, expand_v=expand_v, conv_size=taps, conv_bias=conv_bias)
    with torch.no_grad():
        m.dt_bias.normal_()
        m.g_proj[1].bias.normal_(std=0.3)
        m.o_norm.weight.normal_(1, 0.2)
        for c in (m.q_conv1d, m.k_conv1d, m.v_conv1d):
            if c.bias is not None:
                c.bias.normal_(std=0.2)
    return m.eval()


@pytest.mark.parametrize("H,D,expand_v,taps,conv_bias", [(16, 128, 1.0, 4, False), (12, 64, 1.0, 4, True), (4, 64, 2.0, 3, True),
                                                         (4, 128, 0.5, 2, False), (12, 96, 4 / 3, 4, False), (8, 40, 1.6, 3, False)])
@pytest.mark.parametrize("B,T", [(1, 1), (1, 37), (3, 70), (33, 2)])
def test_layer_in_one_call_equals_its_kernels_one_by_one(H, D, expand_v, taps, conv_bias, B, T, monkeypatch):
    m = _layer(H, D, expand_v, taps, conv_bias)
    g = torch.Generator(device=DEV).manual_seed(B + T)
    x = torch.randn(B, T, H * D, generator=g, device=DEV).bfloat16()
    steps = torch.randn(3, B, 1, H * D, generator=g, device=DEV).bfloat16()

    @torch.no_grad()
    def run(fast):
        taken = []
        whole = KimiLinearSelfAttention._fast
        monkeypatch.setattr(KimiLinearSelfAttention, "_fast",
                            (lambda self, *a: taken.append(whole(self, *a)) or taken[-1]) if fast else (lambda self, *a: None))
        m._recurrent_state = m._conv_state = None
        m._state_homes = {}
        outs = [m(x, None), m.prefill(x, None)[0], m.prefill(x[:, :max(1, T // 2)], None)[0]]
        outs += [m.step(s, None, None, T + i, None, None)[0] for i, s in enumerate(steps)]
        outs += [t.clone() for t in m.state_tensors()]
        addresses = [t.data_ptr() for t in m.state_tensors()]
        m.reset_history()
        outs += [m.prefill(x, None)[0]] + [t.clone() for t in m.state_tensors()]
        assert [t.data_ptr() for t in m.state_tensors()] == addresses
        monkeypatch.undo()
        return outs, taken

    ref, _ = run(False)
    got, taken = run(True)
    served = m.head_v_dim % 64 == 0 and (H * D) % 64 == 0
    assert all((t is not None) == served for t in taken[:3]) and all(t is not None for t in taken[3:6])
    for a, b in zip(ref, got):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert ((a.float() - b.float()).norm() / a.float().norm().clamp_min(1e-9)).item() < 5e-3


@pytest.mark.parametrize("H,D,expand_v,taps,conv_bias", [(8, 8, 4.0, 4, True), (8, 72, 32 / 72, 2, True), (8, 120, 64 / 120, 3, False),
                                                         (16, 56, 128 / 56, 4, False)])
def test_step_whose_key_channels_end_inside_a_tile(H, D, expand_v, taps, conv_bias, monkeypatch):
    """Key widths that are no multiple of the 16 weight rows of a tile, from the smallest; every value width."""
    test_layer_in_one_call_equals_its_kernels_one_by_one(H, D, expand_v, taps, conv_bias, 5, 4, monkeypatch)


@pytest.mark.parametrize("M,K,Ns", [(1, 256, (256, 64, 12)), (4, 128, (100, 8, 1)), (5, 64, (64, 200)), (70, 768, (768, 64, 64, 12)),
                                    (300, 128, (2048, 2048)), (513, 2048, (128, 128, 16))])
def test_products_in_one_launch_equal_separate_ones(M, K, Ns):
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    ws = tuple(torch.randn(n, K, generator=g, device=DEV).bfloat16() for n in Ns)
    bs = tuple(torch.randn(n, generator=g, device=DEV).bfloat16() if M > 4 and i % 2 else None for i, n in enumerate(Ns))
    native = _lib.native()
    for tile in [0] + [t for t, bk in ((1, 128), (2, 128), (3, 128), (4, 64), (5, 64), (6, 64), (7, 64)) if K % bk == 0]:
        ys = native.linears(x, ws, bs, 4, tile)
        assert ys is not None
        for y, w, b in zip(ys, ws, bs):
            ref = x.float() @ w.float().T + (b.float() if b is not None else 0.0)
            assert ((y.float() - ref).abs() <= 2.0 ** -7 * ref.abs() + 1e-3 * K ** 0.5).all(), tile


def test_hooks_on_what_the_layer_calls_are_called():
    m = _layer(4, 64, 1.0, 4, False)
    x = torch.randn(2, 5, 256, device=DEV).bfloat16()
    seen = []
    with torch.no_grad():
        assert m._fast(x, False) is not None
        for add in (m.o_norm.register_forward_hook, m.g_proj[1].register_forward_pre_hook, torch.nn.modules.module.register_module_forward_hook):
            handle = add(lambda *a: seen.append(type(a[0])))
            m(x, None)
            handle.remove()
            assert {"GatedRMSNorm", "Linear"} & {t.__name__ for t in seen}
            seen.clear()


@pytest.mark.parametrize("B,T,H,D", [(1, 5, 4, 64), (5, 1, 12, 64), (2, 33, 4, 128), (1, 700, 12, 96), (1, 2000, 16, 128)])
@pytest.mark.parametrize("strided", [False, True])
def test_input_projections_of_a_layer_on_its_python_path(B, T, H, D, strided):
    """A layer that receives value embeddings, a padded batch: one launch up to the sizes where the library's products lead."""
    m = _layer(H, D, 1.0 if D != 96 else 4 / 3, 4, False)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(B, T, 2 * H * D if strided else H * D, generator=g, device=DEV).bfloat16()[..., :H * D]
    lins = (m.q_proj, m.k_proj, m.v_proj, m.f_proj[0], m.g_proj[0], m.b_proj)
    with torch.no_grad():
        served = _lib.native().linears(x, tuple(l.weight for l in lins), (None,) * 6, 4, 0) is not None
        assert served == (T < 2000)
        for y, l in zip(m._input_projections(x), lins):
            ref = x.float() @ l.weight.float().T
            assert y.shape == ref.shape and y.stride(-1) == 1
            assert ((y.float() - ref).abs() <= 2.0 ** -7 * ref.abs() + 1e-3 * (H * D) ** 0.5).all()
        mask = torch.ones(B, T, dtype=torch.long, device=DEV)
        mask[0, :T // 3] = 0
        if T > 1:
            y = m(x, None, attn_mask=mask)
            alone = m(x[:1, T // 3:].contiguous(), None)
            assert (y[0, :T // 3] == 0).all()
            assert ((y[:1, T // 3:].float() - alone.float()).norm() / alone.float().norm()).item() < 5e-3


@pytest.mark.parametrize("B,T,H,D", [(1, 680, 16, 128), (2, 1031, 8, 128), (1, 3896, 16, 128), (1, 3897, 16, 128), (1, 5201, 12, 64), (1, 7700, 8, 128)])
def test_input_projections_of_the_one_call_on_every_route(B, T, H, D, monkeypatch):
    """The six products in one launch (up to 25 million columns and rows: 3896 rows of 16 heads of 128), and beyond it the large ones by
    themselves, this library's (3897 rows) and the tensor library's (7700); against the layer's Python path."""
    m = _layer(H, D, 1.0, 4, False)
    x = torch.randn(B, T, H * D, generator=torch.Generator(device=DEV).manual_seed(T), device=DEV).bfloat16()
    with torch.no_grad():
        got = m._fast(x, False)
        assert got is not None
        monkeypatch.setattr(KimiLinearSelfAttention, "_fast", lambda self, *a: None)
        ref = m(x, None)
    # the same products with sums in another order ahead of their rounding to bf16, through the layer
    assert ((got.float() - ref.float()).norm() / ref.float().norm()).item() < 5e-3


@pytest.mark.parametrize("B,T,H,D,route", [(1, 3896, 16, 128, "one"), (1, 7700, 8, 128, "own"), (1, 8193, 8, 128, "library")])
def test_input_projections_of_the_one_call_as_the_rules_say(B, T, H, D, route, monkeypatch):
    """One launch, the large products by themselves in this library's kernel, or in the tensor library's: which, the rules that the call asks say."""
    dim, lib = H * D, _lib.load()
    one, own = lib._ZN5daisy17proj_layer_wantedEiii, lib._ZN5daisy11proj_wantedEiii
    one.restype = own.restype = ctypes.c_bool
    assert ("one" if one(B * T, (3 * dim + 2 * D + H + 7) // 8 * 8, dim) else "own" if own(B * T, dim, dim) else "library") == route
    test_input_projections_of_the_one_call_on_every_route(B, T, H, D, monkeypatch)


@pytest.mark.parametrize("what", ["value width", "norm weight"])
@torch.no_grad()
def test_a_call_that_is_given_back_has_not_touched_the_states(what):
    """A value width that the gated norm does not take, a norm weight off its 16-byte boundary: refused ahead of the
    convolutions, which write the windows where they are kept."""
    H, Dk, Dv, B, T = 2, 64, 192 if what == "value width" else 64, 2, 5
    dim, kd, vd = 128, H * Dk, H * Dv
    g = torch.Generator(device=DEV).manual_seed(3)

    def rnd(*shape, dtype=torch.bfloat16):
        return (torch.randn(*shape, generator=g, device=DEV) * 0.1).to(dtype)

    norm_w = rnd(Dv + 1)[1:] if what == "norm weight" else rnd(Dv)
    weights = (rnd(kd, dim), rnd(kd, dim), rnd(vd, dim), rnd(Dv, dim), rnd(Dv, dim), rnd(H, dim), rnd(kd, Dv), rnd(vd, Dv), rnd(vd), rnd(dim, vd),
               rnd(kd, 1, 4), rnd(kd, 1, 4), rnd(vd, 1, 4), None, None, None, rnd(H, dtype=torch.float32), rnd(kd, dtype=torch.float32), norm_w)
    state, windows = rnd(B, H, Dk, Dv, dtype=torch.float32), tuple(rnd(B, c, 4) for c in (kd, kd, vd))
    before = [t.clone() for t in (state, *windows)]
    assert _lib.native().kda_layer(rnd(B, T, dim), weights, H, Dk, Dv, 4, state, windows, (state, *windows), True, 1e-5, 4) is None
    for t, b in zip((state, *windows), before):
        assert torch.equal(t, b)


@pytest.mark.parametrize("B,T,H,D,expand_v,dim", [(1, 4099, 16, 64, 1.0, 1024), (2, 2061, 8, 128, 1.0, 1024), (1, 6251, 16, 40, 1.6, 640),
                                                  (1, 16385, 2, 128, 1.0, 256), (1, 81, 800, 64, 1.0, 64)])
def test_long_rows_take_the_low_rank_kernels(B, T, H, D, expand_v, dim, monkeypatch):
    """Rows that are no multiple of the 16 of a block, 640 columns (no multiple of 128) for the decay gate, fewer columns than an XCD has
    workgroups, more heads than workgroups fit the chip; against the layer's own path, which makes the products as tiles and the norm by itself."""
    m = _layer(H, D, expand_v, 4, False, dim)
    assert _lib.load()._ZN5daisy15low_rank_wantedEiii(B * T, H * D, m.head_v_dim) & 1
    x = torch.randn(B, T, dim, generator=torch.Generator(device=DEV).manual_seed(T), device=DEV).bfloat16()
    whole, taken = KimiLinearSelfAttention._fast, []
    with torch.no_grad():
        monkeypatch.setattr(KimiLinearSelfAttention, "_fast", lambda self, *a: taken.append(whole(self, *a)) or taken[-1])
        got = [m.prefill(x, None)[0]] + [t.clone() for t in m.state_tensors()]
        assert len(taken) == 1 and taken[0] is not None, "the one-call path gave the call back"
        m.reset_history()
        monkeypatch.setattr(KimiLinearSelfAttention, "_fast", lambda self, *a: None)
        ref = [m.prefill(x, None)[0]] + [t.clone() for t in m.state_tensors()]
    # the same products and gates; the norm's sum of squares in another order (fp32) ahead of one rounding to bf16
    for a, b in zip(ref, got):
        assert ((a.float() - b.float()).norm() / a.float().norm()).item() < 1e-3
        assert (a.float() - b.float()).abs().max().item() <= 2 ** -7 * a.float().abs().max().item()
