"""Dense attention with its output token-major (and to a different number of keys), and the head
merge of the processors, at the edges of the 128-row tiles.

Reference: softmax(scale q k^T) v in 64 bits.  P and the output are rounded once each to 8 (bf16)
or 11 (fp16) bits, so the relative error stays within twice half an ulp, 2^-8 or 2^-11, in the
2-norm."""
import pytest
import torch

from oracle import pisa_oracle as O
from pasa_amd import ops
from pasa_amd.processors.qknorm import merge_heads

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def make(B, H, S, L, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, H, S, 128, generator=g).to(dtype)
    k, v = (torch.randn(B, H, L, 128, generator=g).to(dtype) for _ in range(2))
    return q, k, v


@pytest.mark.parametrize("B,H,S,L,dtype", [(1, 1, 1, 1, torch.bfloat16), (2, 3, 129, 512, torch.bfloat16),
                                           (1, 2, 1000, 77, torch.float16), (1, 5, 127, 257, torch.bfloat16),
                                           (1, 1, 2048, 128, torch.float16), (1, 2, 300, 300, torch.bfloat16)])
def test_cross_attention(device, B, H, S, L, dtype):
    q, k, v = make(B, H, S, L, dtype, S + L)
    o = ops.cross_attention(q.to(device), k.to(device), v.to(device))
    assert o.shape == q.shape and o.transpose(1, 2).is_contiguous()
    ref = O.dense_attention(q, k, v, O.effective_scale(128 ** -0.5))
    err = float((o.cpu().double() - ref).norm() / ref.norm())
    print(f"[cross] B={B} H={H} S={S} L={L} {dtype}: rel {err:.2e}", flush=True)
    assert err <= TOL[dtype]


@pytest.mark.parametrize("B,H,T,text,valid,dtype", [(1, 3, 700, 0, None, torch.bfloat16),
                                                    (2, 2, 513, 100, 37, torch.float16)])
def test_dense_token_major_is_the_same(device, B, H, T, text, valid, dtype):
    q, k, v = (t.to(device) for t in make(B, H, T, T, dtype, T))
    a = ops.dense_attention(q, k, v, text_tokens=text, text_valid=valid)
    b = ops.dense_attention(q, k, v, text_tokens=text, text_valid=valid, token_major_out=True)
    assert b.transpose(1, 2).is_contiguous() and torch.equal(a, b)


@pytest.mark.parametrize("B,H,S,D", [(1, 12, 1000, 128), (2, 3, 5, 64), (1, 1, 7, 128), (1, 70, 9, 128)])
def test_merge_heads(device, B, H, S, D):
    x = torch.randn(B, H, S, D, device=device, dtype=torch.bfloat16)
    want = x.transpose(1, 2).flatten(2, 3)
    assert torch.equal(merge_heads(x), want)
    view = x.transpose(1, 2).contiguous().transpose(1, 2)   # token-major memory: a view suffices
    assert torch.equal(merge_heads(view), want) and merge_heads(view).data_ptr() == view.data_ptr()


@pytest.mark.parametrize("B,H,S,D", [(1, 12, 1000, 128), (2, 3, 5, 64), (1, 64, 9, 128), (1, 12, 4200, 128)])
def test_merge_heads_on_the_kernel(device, monkeypatch, B, H, S, D):
    """The layout pass itself at the sizes that the rule leaves to PyTorch, and one that it takes."""
    from pasa_amd.processors import qknorm
    calls = []
    prologue = qknorm.qkv_prologue
    monkeypatch.setattr(qknorm, "qkv_prologue", lambda *a, **k: calls.append(1) or prologue(*a, **k))
    x = torch.randn(B, H, S, D, device=device, dtype=torch.bfloat16)
    want = x.transpose(1, 2).flatten(2, 3)
    assert torch.equal(merge_heads(x), want)
    assert len(calls) == (x.numel() >= qknorm.MERGE_KERNEL_MIN)
    monkeypatch.setattr(qknorm, "MERGE_KERNEL_MIN", 0)
    assert torch.equal(merge_heads(x), want) and calls


def test_rejected_arguments(device):
    q, k, v = (t.to(device) for t in make(1, 2, 16, 8, torch.bfloat16, 0))
    with pytest.raises(ValueError):
        ops.cross_attention(q[:, :1].contiguous(), k, v)
    with pytest.raises(ValueError):
        ops.cross_attention(q.float(), k, v)
    with pytest.raises(ops._lib.PasaError):
        ops.cross_attention(q[..., :64].contiguous(), k[..., :64].contiguous(), v[..., :64].contiguous())


def test_block_with_and_without_the_fused_cross_attention(device):
    """One Wan block (2 heads x 128) whose feed-forward and cross-attention run fused, against the
    same block with a hook on each that makes it call the modules: two more bf16 roundings of
    intermediate rows (2^-9 each, relative) on the module route, two fewer on the fused one."""
    from pasa_amd import wan_dit as W
    torch.manual_seed(0)
    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=512, text_dim=64, freq_dim=16)
    blk = W.WanBlock(cfg).to(device, torch.bfloat16).eval()
    blk.fused_min_rows = 0
    x = torch.randn(1, 300, 256, device=device, dtype=torch.bfloat16)
    text = torch.randn(1, 37, 256, device=device, dtype=torch.bfloat16)
    temb = torch.randn(1, 6, 256, device=device, dtype=torch.bfloat16)
    with torch.no_grad():
        assert W._cross_fusable(blk.attn2, x, text)
        a = blk(x, text, temb, None)
        calls = []
        for m in (blk.attn2, blk.ffn):
            m.register_forward_hook(lambda m, i, o: calls.append(type(m).__name__))
        b = blk(x, text, temb, None)
    assert calls == ["WanAttention", "Sequential"]
    err = float((a.double() - b.double()).norm() / b.double().norm())
    print(f"[cross] block fused against modules: rel {err:.2e}", flush=True)
    assert err <= 2.0 ** -7


@pytest.mark.parametrize("B,S,least,fused", [(1, 300, 0, True), (2, 1025, 2048, True), (1, 300, 2048, False)])
def test_block_fuses_from_a_number_of_rows_on(device, monkeypatch, B, S, least, fused):
    """The routes of the same block by its rows, with the bound of the test above between the two."""
    from pasa_amd import wan_dit as W
    torch.manual_seed(0)
    cfg = W.WanDiTConfig(num_layers=1, num_attention_heads=2, ffn_dim=512, text_dim=64, freq_dim=16)
    blk = W.WanBlock(cfg).to(device, torch.bfloat16).eval()
    x = torch.randn(B, S, 256, device=device, dtype=torch.bfloat16)
    text = torch.randn(B, 37, 256, device=device, dtype=torch.bfloat16)
    temb = torch.randn(B, 6, 256, device=device, dtype=torch.bfloat16)
    calls = []
    cross = W._cross_attention_fused
    monkeypatch.setattr(W, "_cross_attention_fused", lambda *a: calls.append(1) or cross(*a))
    ffn = W.WanBlock._ffn_fused
    monkeypatch.setattr(W.WanBlock, "_ffn_fused", lambda self, x: calls.append(2) or ffn(self, x))
    with torch.no_grad():
        blk.fused_min_rows = B * S + 1
        b = blk(x, text, temb, None)
        assert not calls
        blk.fused_min_rows = least
        a = blk(x, text, temb, None)
    assert calls == ([1, 2] if fused else [])
    assert float((a.double() - b.double()).norm() / b.double().norm()) <= (2.0 ** -7 if fused else 0.0)
