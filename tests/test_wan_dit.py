"""The Wan2.1 DiT harness (pasa_amd.wan_dit) on the CPU: closed forms of its RoPE grid,
timestep embedding and unpatchify, the installer on its pipeline shape, and the PASA
processor's dense branch against the harness's own dense processor."""
import cmath
import math

import pytest
import torch

from pasa_amd import wan_dit as W
from pasa_amd.processors import Wan_PASA_Processor, replace_wan_attention


def tiny_cfg(layers=2):
    return W.WanDiTConfig(text_dim=64, freq_dim=32, ffn_dim=512, num_layers=layers, num_attention_heads=2,
                          attention_head_dim=128, rope_max_seq_len=64)


def test_rope_grid_closed_form():
    rope = W.WanRotaryPosEmbed(128, (1, 2, 2), 64)
    lat = torch.zeros(1, 16, 3, 4, 6)
    f = rope(lat)
    assert f.shape == (1, 1, 3 * 2 * 3, 64) and f.dtype == torch.complex128
    for n in range(18):
        fr, y, x = n // 6, (n // 3) % 2, n % 3
        for j in range(64):
            if j < 22:
                ang = fr * 10000.0 ** (-2 * j / 44)
            elif j < 43:
                ang = y * 10000.0 ** (-2 * (j - 22) / 42)
            else:
                ang = x * 10000.0 ** (-2 * (j - 43) / 42)
            assert abs(complex(f[0, 0, n, j]) - cmath.exp(1j * ang)) < 1e-12


def test_timestep_embedding_closed_form():
    t = torch.tensor([0.0, 500.0])
    e = W.timestep_embedding(t, 8)
    assert torch.equal(e[0], torch.tensor([1.0, 1, 1, 1, 0, 0, 0, 0]))
    for i in range(4):
        w = math.exp(-math.log(10000.0) * i / 4)
        assert abs(float(e[1, i]) - math.cos(500 * w)) < 1e-4
        assert abs(float(e[1, 4 + i]) - math.sin(500 * w)) < 1e-4


def test_unpatchify_brute_force():
    nf, nh, nw, pt, ph, pw, C = 2, 3, 2, 1, 2, 2, 3
    x = torch.randn(1, nf * nh * nw, pt * ph * pw * C)
    out = W.unpatchify(x, (nf, nh, nw), (pt, ph, pw))
    assert out.shape == (1, C, nf * pt, nh * ph, nw * pw)
    for f in range(nf):
        for y in range(nh):
            for xx in range(nw):
                tok = (f * nh + y) * nw + xx
                for a in range(pt):
                    for i in range(ph):
                        for j in range(pw):
                            for c in range(C):
                                assert out[0, c, f * pt + a, y * ph + i, xx * pw + j] == \
                                    x[0, tok, ((a * ph + i) * pw + j) * C + c]


def test_forward_shape_and_latent_shape():
    torch.manual_seed(0)
    m = W.WanDiT(tiny_cfg())
    assert W.latent_shape(81, 480, 832) == (16, 21, 60, 104)
    lat = torch.randn(1, 16, 3, 4, 6)
    out = m(lat, torch.tensor([500]), torch.randn(1, 7, 64))
    assert out.shape == lat.shape and torch.isfinite(out).all()


def test_installer_on_pipeline_shape():
    torch.manual_seed(0)
    pipe = W.WanPipelineShape(W.WanDiT(tiny_cfg(3)))
    replace_wan_attention(pipe, height=32, width=48, num_frames=9, first_layers_fp=1, first_times_fp=900)
    for i, blk in enumerate(pipe.transformer.blocks):
        assert isinstance(blk.attn1.processor, Wan_PASA_Processor) and blk.attn1.processor.layer_idx == i
        assert isinstance(blk.attn2.processor, W.WanAttnProcessor)
    # latent [16, 3, 4, 6] -> 3 frames of 2 x 3 patches
    assert (Wan_PASA_Processor.num_frame, Wan_PASA_Processor.frame_size) == (3, 6)
    assert Wan_PASA_Processor.context_length == 0 and Wan_PASA_Processor.num_layers == 3


def test_pasa_dense_branch_matches_stock_processor():
    """With every timestep above first_times_fp the PASA processor attends densely; its
    projections, RMSNorm, head split and RoPE must then reproduce the stock processor."""
    torch.manual_seed(0)
    m = W.WanDiT(tiny_cfg())
    lat, ts, text = torch.randn(1, 16, 3, 4, 6), torch.tensor([500]), torch.randn(1, 7, 64)
    with torch.no_grad():
        ref = m(lat, ts, text)
        replace_wan_attention(W.WanPipelineShape(m), height=32, width=48, num_frames=9, first_layers_fp=0,
                              first_times_fp=0)
        out = m(lat, ts, text)
    torch.testing.assert_close(out, ref, rtol=1e-4, atol=1e-5)


def test_rope_survives_dtype_cast():
    """Casting the model to bf16 must leave the complex RoPE table complex128."""
    m = W.WanDiT(tiny_cfg(1)).to(torch.bfloat16)
    f = m.rope(torch.zeros(1, 16, 3, 4, 6))
    assert f.dtype == torch.complex128 and f.imag.abs().max() > 0.5


def test_fused_paths_leave_replaced_and_hooked_modules_alone():
    """The block's fused feed-forward and cross-attention step aside for anything that a module call
    would run and they would not: subclasses (adapters), hooks, another activation or processor."""
    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=64, text_dim=32, freq_dim=16)
    blk = W.WanBlock(cfg)

    class Adapter(torch.nn.Linear):
        pass

    assert W._plain(blk.ffn, torch.nn.Sequential) and W._plain(blk.ffn[0], torch.nn.Linear)
    assert not W._plain(Adapter(4, 4), torch.nn.Linear)
    handle = blk.attn2.register_forward_hook(lambda m, a, o: o)
    assert not W._plain(blk.attn2, W.WanAttention)
    handle.remove()
    assert W._plain(blk.attn2, W.WanAttention)
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, o: o)
    assert not W._plain(blk.attn2, W.WanAttention)
    handle.remove()
    blk.ffn[0].forward = lambda x: torch.nn.Linear.forward(blk.ffn[0], x) * 2
    with torch.no_grad():                                    # a wrapper set on the object runs
        torch.testing.assert_close(blk._ffn_fused(torch.ones(1, 3, 256)), blk.ffn(torch.ones(1, 3, 256)))
    assert not W._plain(blk.ffn[0], torch.nn.Linear)
    del blk.ffn[0].forward
    x, text = torch.randn(1, 3, 256), torch.randn(1, 5, 256)
    with torch.no_grad(), torch.autocast("cpu", torch.bfloat16):
        assert blk._ffn_fused(x).dtype == blk.ffn(x).dtype == torch.bfloat16
    assert not W._cross_fusable(blk.attn2, x, text)          # host tensors
    blk.ffn[1] = torch.nn.GELU()                             # the erf form has no fused counterpart
    with torch.no_grad():
        torch.testing.assert_close(blk._ffn_fused(x), blk.ffn(x))


def test_only_the_pasa_processor_is_given_the_timestep_on_the_host(monkeypatch):
    """The stock processor (whose forward may be captured in a graph) and any other one that takes a
    timestep see the caller's own tensor, unread; the PASA processors share one host copy."""
    class Takes(W.WanAttnProcessor):
        def __call__(self, attn, hidden_states, timestep=None, **kw):
            self.seen = timestep
            return super().__call__(attn, hidden_states, **kw)

    class Pasa(Wan_PASA_Processor):
        pass

    m = W.WanDiT(tiny_cfg(4))
    m.blocks[1].attn1.set_processor(Takes())
    m.blocks[2].attn1.set_processor(Wan_PASA_Processor(2))
    m.blocks[3].attn1.set_processor(Pasa(3))
    assert [W._reads_timestep_on_host(b) for b in m.blocks] == [False, False, True, False]
    m.blocks[2].attn1.register_forward_pre_hook(lambda *a: None)
    assert not W._reads_timestep_on_host(m.blocks[2])

    m = W.WanDiT(tiny_cfg(2))
    m.blocks[1].attn1.set_processor(Takes())
    copies = []
    for name in ("cpu", "tolist", "item"):
        monkeypatch.setattr(torch.Tensor, name, lambda self, name=name: copies.append(name))
    t = torch.tensor([500.0])
    with torch.no_grad():
        m(torch.randn(1, 16, 2, 4, 4), t, torch.randn(1, 5, m.cfg.text_dim))
    assert m.blocks[1].attn1.processor.seen is t and not copies


@pytest.mark.parametrize("text_shape, fused", [((2, 5, 256), True), ((1, 5, 256), False), ((2, 0, 256), False)])
def test_fused_cross_attention_takes_one_text_per_sample(monkeypatch, text_shape, fused):
    """A text that broadcasts over the samples, and an empty one, stay on the module's own route."""
    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=64, text_dim=32, freq_dim=16)
    attn = W.WanBlock(cfg).to(torch.bfloat16).attn2
    monkeypatch.setattr(W, "fusable", lambda *a: True)       # the device test, as on a GPU
    x, text = torch.zeros(2, 3, 256, dtype=torch.bfloat16), torch.zeros(text_shape, dtype=torch.bfloat16)
    assert W._cross_fusable(attn, x, text) is fused
    with torch.autocast("cpu", torch.bfloat16):
        assert not W._cross_fusable(attn, x, text)
    attn.to_k.float()
    assert not W._cross_fusable(attn, x, text)


class QuantisedLike(torch.Tensor):
    """A weight that reports bf16 and is only ever multiplied through F.linear."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        plain = [a.as_subclass(torch.Tensor) if isinstance(a, cls) else a for a in args]
        if func is torch.nn.functional.linear or func.__name__ in ("__get__", "dim", "size"):
            return func(*plain, **(kwargs or {}))
        raise NotImplementedError(str(func))


@pytest.mark.parametrize("name", ["weight", "bias"])
def test_fused_feed_forward_leaves_other_kinds_of_weights_to_the_module(name):
    """A plain Linear whose weight or bias is a tensor subclass (weight-only quantisation, distributed
    tensors) multiplies through F.linear alone."""
    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=64, text_dim=32, freq_dim=16)
    blk = W.WanBlock(cfg).to(torch.bfloat16)
    up = blk.ffn[0]
    w = getattr(up, name).detach().as_subclass(QuantisedLike)
    del up._parameters[name]
    object.__setattr__(up, name, w)
    x = torch.randn(1, 3, 256, dtype=torch.bfloat16)
    with torch.no_grad():
        assert torch.equal(blk._ffn_fused(x), blk.ffn(x))


def test_fused_feed_forward_keeps_the_shapes_that_modules_see(monkeypatch):
    """The down projection (a hook on it, an adapter in its place) is called with the module path's shape,
    and a batch without rows passes through."""
    monkeypatch.setattr(torch, "_addmm_activation",          # torch's own is the erf form on the CPU
                        lambda b, x, w, use_gelu: torch.nn.functional.gelu(torch.addmm(b, x, w), approximate="tanh"))
    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=64, text_dim=32, freq_dim=16)
    blk = W.WanBlock(cfg)
    seen = []
    blk.ffn[2].register_forward_pre_hook(lambda m, args: seen.append(tuple(args[0].shape)))
    with torch.no_grad():
        for shape in ((1, 3, 256), (2, 0, 256)):
            x = torch.randn(shape)
            a, b = blk._ffn_fused(x), blk.ffn(x)
            assert seen[-2] == seen[-1] == (*shape[:2], 64)
            torch.testing.assert_close(a, b)


def test_fused_cross_attention_wants_plain_projections(monkeypatch):
    """A projection that is not nn.Linear itself may return another type or width than the kernels take."""
    class Widening(torch.nn.Module):
        def __init__(self, lin):
            super().__init__()
            self.lin = lin

        def forward(self, x):
            return self.lin(x).float()

    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=64, text_dim=32, freq_dim=16)
    monkeypatch.setattr(W, "fusable", lambda *a: True)       # the device test, as on a GPU
    x, text = torch.zeros(2, 3, 256, dtype=torch.bfloat16), torch.zeros(2, 5, 256, dtype=torch.bfloat16)
    for name in ("to_q", "to_k", "to_v"):
        attn = W.WanBlock(cfg).to(torch.bfloat16).attn2
        assert W._cross_fusable(attn, x, text)
        lin = getattr(attn, name)
        setattr(attn, name, Widening(lin))
        assert not W._cross_fusable(attn, x, text)
        setattr(attn, name, torch.nn.Linear(256, 512, dtype=torch.bfloat16))
        assert not W._cross_fusable(attn, x, text)
        setattr(attn, name, lin)
        lin.register_forward_hook(lambda m, i, o: o.float())
        assert not W._cross_fusable(attn, x, text)


def test_feed_forward_of_another_make():
    """A feed-forward that is not the block's own three modules is called as it is."""
    class Mlp(torch.nn.Module):
        def forward(self, x):
            return x * 3

    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=64, text_dim=32, freq_dim=16)
    x = torch.randn(1, 3, 256)
    lin = lambda a, b: torch.nn.Linear(a, b)
    for ffn in (Mlp(), torch.nn.Sequential(lin(256, 256)), torch.nn.Sequential(),
                torch.nn.Sequential(lin(256, 64), torch.nn.GELU(approximate="tanh"), torch.nn.Dropout(0.0), lin(64, 256))):
        blk = W.WanBlock(cfg)
        blk.ffn = ffn
        with torch.no_grad():
            assert torch.equal(blk._ffn_fused(x), ffn(x))
