"""The any-shape kernels at the edges of their tiles: head dims that are not whole 16-byte chunks
(the element-wise loads), tensors whose data is not 16-byte aligned, block counts that leave a
workgroup's last waves without a block, 16-row blocks two to a chunk (odd counts of them), groups
longer than one zero-order chunk, and the smallest sizes of each.

The attention stage runs on the GPU's own statistics and selection and is held to the oracle's
attention stage on that selection: fp32 to a relative 2-norm of 4e-6 (the longest fp32 chain here
has a few hundred terms of rounding 2^-24: sqrt(300) * 6e-8 = 1e-6 in the scores, which the
softmax passes on about once, and as much again in the products with V), 16 bits to 1.5 times the
error of the oracle run with the reference's own roundings, plus one ulp."""
import pytest
import torch

from oracle import pisa_oracle as O
from pasa_amd import ops

pytestmark = pytest.mark.gpu

B16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def make(heads, T, D, dtype, seed, shift=0):
    """q, k, v [1, heads, T, D] whose data starts ``shift`` elements into its storage."""
    g = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(3):
        buf = torch.randn(heads * T * D + shift, generator=g).to(dtype)
        out.append(buf[shift:].view(1, heads, T, D))
    return out


def to_dev(t, device, shift):
    buf = torch.empty(t.numel() + shift, dtype=t.dtype, device=device)
    view = buf[shift:].view(t.shape)
    view.copy_(t)
    assert view.is_contiguous()
    return view


# heads, T, D, BT, G, density, dtype, gamma, text, valid, shift
CASES = [
    (1, 16, 16, 16, 1, 1.0, F32, "literal", 0, 0, 0),          # one block, nothing approximated
    (2, 17, 1, 16, 32, 0.5, F32, "literal", 0, 0, 0),          # one feature, a block of one row
    (1, 700, 37, 64, 7, 0.2, F32, "consistent", 0, 0, 0),      # odd head dim, fp32
    (1, 700, 37, 32, 7, 0.2, B16, "literal", 0, 0, 0),         # odd head dim, 16 bits
    (2, 530, 96, 32, 16, 0.2, B16, "literal", 0, 0, 3),        # misaligned data
    (1, 530, 128, 64, 32, 0.2, F32, "literal", 0, 0, 1),       # misaligned data, fp32
    (1, 1111, 40, 16, 5, 0.11, F16, "literal", 0, 0, 0),       # 70 blocks of 16: 7 selected, an odd count
    (1, 1111, 100, 16, 64, 0.03, F32, "literal", 33, 5, 0),    # 16-row blocks in fp32, text and padding
    (1, 2079, 72, 16, 100, 0.05, B16, "consistent", 31, 31, 0),  # groups of 100: several zero-order chunks
    (2, 993, 64, 32, 64, 0.3, F32, "literal", 0, 0, 0),        # two waves per 32-row block
    (1, 1250, 112, 256, 2, 0.5, F16, "literal", 130, 70, 0),   # two tiles per block, text
    (3, 129, 128, 128, 8, 0.5, B16, "literal", 0, 0, 0),       # a last block of one row
    (1, 33000, 64, 128, 16, 0.02, B16, "literal", 0, 0, 0),    # enough blocks for 128-row tiles
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_attention_edges(device, case):
    heads, T, D, BT, G, density, dtype, gamma, text, valid, shift = case
    q, k, v = make(heads, T, D, dtype, T + D + BT)
    assert not ops.tuned_shape(dtype, D, BT, G, text)
    qd, kd, vd = (to_dev(t, device, shift) for t in (q, k, v))
    scale = D ** -0.5
    st = ops.block_stats(qd, kd, vd, BT, G, text_tokens=text)
    sel = ops.select_blocks(st, density, scale)
    out = to_dev(torch.zeros_like(v), device, shift)
    o = ops.sparse_attn(qd, kd, vd, st, sel, scale, BT, gamma, out=out, text_tokens=text, text_valid=valid,
                        group_size=G).cpu()
    kw = dict(gamma=gamma, indices=sel.idx.cpu(), text_tokens=text, text_valid=valid)
    ref = O.pisa_pg_attention(q, k, v, density, BT, G, scale, dtype=torch.float64, **kw)
    err = (o.double() - ref).norm() / ref.norm()
    print(f"[edges] {case}: rel {err:.2e}", flush=True)
    if dtype == F32:
        assert err <= 4e-6
        return
    rp = O.pisa_pg_attention(q, k, v, density, BT, G, scale, ref_precision=dtype, **kw).double()
    ulp = float(O.ulp(ref.abs().max(), dtype))
    assert float((o.double() - ref).abs().max()) <= 1.5 * float((rp - ref).abs().max()) + ulp
    assert err <= 1.5 * float((rp - ref).norm() / ref.norm())


@pytest.mark.parametrize("T,D,dtype,text,valid,shift", [(1, 5, F32, 0, 0, 0), (333, 72, B16, 0, 0, 1),
                                                       (200, 64, F32, 70, 1, 0), (33000, 96, F16, 0, 0, 0)])
def test_dense_edges(device, T, D, dtype, text, valid, shift):
    q, k, v = make(1, T, D, dtype, T + D)
    qd, kd, vd = (to_dev(t, device, shift) for t in (q, k, v))
    o = ops.dense_attention(qd, kd, vd, text_tokens=text, text_valid=valid).double().cpu()
    seg, es = T - text + valid, O.effective_scale(D ** -0.5)
    rows = torch.cat([torch.arange(0, min(seg, 100)), torch.arange(max(0, seg - 100), T)]).unique()
    a, b = rows[rows < seg], rows[rows >= seg]
    ref = torch.cat([O.dense_attention(q[..., r, :].double(), k[..., s, :].double(), v[..., s, :].double(), es)
                     for r, s in ((a, slice(0, seg)), (b, slice(seg, T))) if len(r)], dim=2)
    err = float((o[..., rows, :] - ref).norm() / ref.norm())
    print(f"[edges] dense T={T} D={D} {dtype}: rel {err:.2e}", flush=True)
    # 16 bits: P and o rounded once each to 8 (bf16) or 11 (fp16) bits
    assert err <= {F32: 4e-6, B16: 6e-3, F16: 1e-3}[dtype]


@pytest.mark.parametrize("case", ["finite_range", "minus_inf_score", "inf_value", "nan_row"])
@pytest.mark.parametrize("T,D", [(64, 64), (131, 37), (200, 128)])
def test_dense_fp32_range(device, T, D, case):
    """fp32 rows are multiplied as three bf16 parts each, and tiles that hold an infinity or NaN in
    fp32: the ends of the range and the infinities come out as fp32 products give them."""
    q, k, v = make(1, T, D, F32, 3 * T + D)
    q[..., 0] = q[..., 0].abs() + 0.1
    hot = T // 2  # the key, or the query row, that is special
    if case == "finite_range":
        v[..., 1] *= 2.0 ** 110      # sums of up to 200 weights <= 1 before they are normalised:
        v[..., 2] = 2.0 ** 119       # below 2^127
        v[..., 3] *= 2.0 ** -80      # and small ones
        k[..., hot, 0] = -3.0e38     # a weight of exactly 0
    elif case == "minus_inf_score":
        k[..., hot, 0] = -torch.inf  # a score of -inf in every row: that key has no weight
    elif case == "inf_value":
        v[..., hot, 1], v[..., hot, 2] = torch.inf, -torch.inf
    else:
        q[..., hot, 1] = torch.nan   # one row of NaN, the others as they were
    o = ops.dense_attention(*(to_dev(t, device, 0) for t in (q, k, v))).double().cpu()
    es = O.effective_scale(D ** -0.5)
    s = (q.double() @ k.double().transpose(-1, -2)) * es
    ref = torch.softmax(s, -1) @ v.double()
    if case == "finite_range":
        assert float((torch.softmax(s, -1)[..., hot]).max()) == 0.0
    assert torch.equal(torch.isnan(o), torch.isnan(ref)) and torch.equal(torch.isinf(o), torch.isinf(ref))
    assert torch.equal(o.isposinf(), ref.isposinf())
    ok = torch.isfinite(ref)
    for col in range(D):  # per feature: their magnitudes differ
        a, b = o[..., col][ok[..., col]], ref[..., col][ok[..., col]]
        if a.numel():
            assert float((a - b).norm() / b.norm()) <= 1e-5, col  # cancellation within one feature: 2.5x the bound above


def short_chain_scores(q, k):
    """q k^T in fp32 with one FMA chain per 16 features, the chains added pairwise."""
    x, y = q.double(), k.double()
    parts = []
    for f in range(0, q.shape[-1], 16):
        acc = torch.zeros(*q.shape[:-1], k.shape[-2], dtype=torch.float64)
        for d in range(f, min(f + 16, q.shape[-1])):
            acc = (x[..., :, None, d] * y[..., None, :, d] + acc).float().double()
        parts.append(acc)
    while len(parts) > 1:
        parts = [(sum(parts[i:i + 2])).float().double() for i in range(0, len(parts), 2)]
    return parts[0]


@pytest.mark.parametrize("BT", [16, 32])
@pytest.mark.parametrize("D,mq,mk", [(128, 1.0, 3.0), (128, 3.0, 3.0), (96, 1.0, 3.0), (64, 3.0, 3.0), (37, 1.0, 3.0)])
def test_fp32_scores_of_q_and_k_with_a_mean(device, BT, D, mq, mk):
    """fp32 below block 64, every block selected (so plain attention): q and k with a common mean give
    scores of about D mq mk / sqrt(D), whose rounding is then the whole error.  It is no larger than
    with chains of 16 features in 64-bit arithmetic otherwise, but for a quarter (the order within a chain
    is another) and what the exponentials and P V add (4e-7, as with no mean)."""
    q, k, v = make(1, 512, D, F32, D + BT)
    q, k = q + mq, k + mk
    d = [t.to(device) for t in (q, k, v)]
    scale = D ** -0.5
    st = ops.block_stats(*d, BT, 8)
    sel = ops.select_blocks(st, 1.0, scale)
    o = ops.sparse_attn(*d, st, sel, scale, BT, group_size=8).double().cpu()
    es = O.effective_scale(scale)
    ref = torch.softmax(q.double() @ k.double().transpose(-1, -2) * es, -1) @ v.double()
    short = torch.softmax(short_chain_scores(q, k) * es, -1) @ v.double()
    err, bound = (float((x - ref).norm() / ref.norm()) for x in (o, short))
    print(f"[edges] means {mq} {mk} BT={BT} D={D}: rel {err:.2e}, chains of 16 {bound:.2e}", flush=True)
    assert err <= 1.25 * bound + 4e-7


@pytest.mark.parametrize("D", [4, 5, 68, 100])
def test_fp32_split_product(device, D):
    """fp32 on the bf16 MFMA: one key of 64 has scores s = q a scale of -20 to -80, the others 0, so its
    weight is exp(s) / (63 + exp(s)) and shows the relative error of a single product times |s|.  That
    is at most 2^-24 for what the product leaves out, 2^-24 for its rounding and 2^-24 for that of
    s log2(e); a part cut instead of rounded leaves out up to 3.9 of 2^-24.  The exponential, the sum and
    the quotient round to 4 x 2^-23 more."""
    heads, T = 512, 64
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.zeros(1, heads, T, D) for _ in range(3))
    scale = 0.5
    q[..., D - 1] = 8 + 8 * torch.rand(1, heads, T, generator=g)
    k[..., T // 2, D - 1] = -5 - 5 * torch.rand(1, heads, generator=g)
    v[..., T // 2, 0] = 1.0
    o = ops.dense_attention(*(t.to(device) for t in (q, k, v)), scale=scale)[..., 0].double().cpu()
    s = q[..., D - 1].double() * k[..., T // 2, D - 1, None].double() * O.effective_scale(scale)
    ref = torch.exp(s) / (T - 1 + torch.exp(s))
    err = ((o / ref - 1).abs() - 4 * 2.0 ** -23) / (s.abs() * 2.0 ** -24)
    print(f"[edges] split product D={D}: {float(err.max()):.2f} of 2^-24 per unit of score", flush=True)
    assert float(err.max()) <= 3.1


@pytest.mark.parametrize("eq,ek,ev", [(0, 0, -112), (0, 0, -121), (-121, 121, 0), (121, -121, 0), (85, -85, -118),
                                      (-118, 90, 30), (0, 0, 100), (0, 0, -130), (0, 0, -140)])
@pytest.mark.parametrize("D,BT", [(64, 64), (37, 128), (128, 64)])
def test_fp32_range(device, D, BT, eq, ek, ev):
    """fp32 down to the subnormals and up to where the split sums leave the range: q, k and v times 2^eq,
    2^ek and 2^ev, with the scores' magnitude kept.  Relative error as for ordinary values, and for
    subnormal results half of 2^-149 each besides.  (Where v or the block
    moments k v are below 2^-121 only the dense call: the statistics' own sums are subnormal there.)"""
    T = 300
    q, k, v = make(1, T, D, F32, T + D)
    d = [(t * 2.0 ** e) for t, e in zip((q, k, v), (eq, ek, ev))]
    c = [t.to(device) for t in d]
    scale = D ** -0.5 * 2.0 ** -(eq + ek)

    def check(o, ref):
        err, n = float((o - ref).norm()), float(ref.norm())
        print(f"[edges] fp32 range D={D} BT={BT} 2^{eq} 2^{ek} 2^{ev}: rel {err / n:.2e}", flush=True)
        assert err <= 4e-6 * n + 2.0 ** -150 * o.numel() ** 0.5

    es = O.effective_scale(scale)
    ref = torch.softmax(d[0].double() @ d[1].double().transpose(-1, -2) * es, -1) @ d[2].double()
    check(ops.dense_attention(*c, scale=scale).double().cpu(), ref)
    if min(ev, ek + ev) < -121:
        return
    st = ops.block_stats(*c, BT, 2)
    sel = ops.select_blocks(st, 0.4, scale)
    o = ops.sparse_attn(*c, st, sel, scale, BT, group_size=2).double().cpu()
    check(o, O.pisa_pg_attention(*d, 0.4, BT, 2, scale, dtype=torch.float64, indices=sel.idx.cpu()))


def selection(rows, device):
    """The selection of one slice whose query block I selects the key blocks rows[I]."""
    NT = len(rows)
    m = torch.zeros(NT, (NT + 31) // 32, dtype=torch.int64)
    for i, js in enumerate(rows):
        for j in js:
            m[i, j // 32] |= 1 << (j % 32)
    idx = torch.tensor([sorted(js) for js in rows], dtype=torch.int32)[None, None]
    mask = torch.where(m >= 2 ** 31, m - 2 ** 32, m).to(torch.int32)[None, None].to(device)
    return ops.Selection(None, mask, None, idx.shape[-1]), idx


@pytest.mark.parametrize("BT,D,dtype", [(16, 72, F32), (16, 72, B16), (32, 40, F16), (32, 128, F32), (64, 72, F32),
                                        (64, 72, B16), (128, 37, F16), (64, 64, B16), (64, 128, B16), (64, 128, F16),
                                        (128, 128, B16), (128, 64, B16)])
def test_infinity_in_a_selected_group_stays_there(device, BT, D, dtype):
    """Two value rows of one group hold an infinity.  Query blocks that select the whole group do not
    approximate it: their output is infinite in those two features and what it was in all others, whatever
    other query blocks of their workgroup approximate."""
    G = 32 if ops.tuned_shape(dtype, D, BT) else 2
    NT = 2 * G + 6
    T = NT * BT - 3
    q, k, v = make(1, T, D, dtype, T + D)
    whole = set(range(G))                                   # the first group
    rows = [whole | {NT - 1, NT - 2} if i % 2 == 0 else set(range(NT - 1, NT - 1 - G - 2, -1)) for i in range(NT)]
    sel, idx = selection(rows, device)
    bad = v.clone()
    bad[0, 0, 3, 7], bad[0, 0, (G - 1) * BT + 5, 30] = torch.inf, -torch.inf
    scale = D ** -0.5
    d = [t.to(device) for t in (q, k, bad)]
    st = ops.block_stats(*d, BT, G)
    o = ops.sparse_attn(*d, st, sel, scale, BT, group_size=G).double().cpu()
    ref = O.pisa_pg_attention(q, k, v, 0.5, BT, G, scale, dtype=torch.float64, indices=idx)
    even = (torch.arange(T) // BT) % 2 == 0
    fine = [c for c in range(D) if c not in (7, 30)]
    assert bool((o[..., even, 7] == torch.inf).all()) and bool((o[..., even, 30] == -torch.inf).all())
    a, b = o[..., fine], ref[..., fine]
    err = float((a - b).norm() / b.norm())
    print(f"[edges] infinity BT={BT} D={D} {dtype}: rel {err:.2e}", flush=True)
    assert err <= {F32: 4e-6, B16: 1e-2, F16: 2e-3}[dtype]    # 16 bits: kc, vc, Hbar, P and o rounded once each


@pytest.mark.parametrize("BT,D", [(16, 72), (32, 128), (64, 72), (128, 40), (256, 96)])
def test_a_selected_block_whose_value_sum_leaves_fp16(device, BT, D):
    """Every query block selects block 4, whose values add up to more than fp16 holds; the other blocks of
    its group are approximated, and that sum, whose weight there is 0, does not show."""
    NT = 9
    T = NT * BT - 3
    q, k, v = make(1, T, D, F16, T + D)
    v[..., 4 * BT:5 * BT, :] += 8192.0
    sel, idx = selection([{4, i if i != 4 else 0} for i in range(NT)], device)
    scale = D ** -0.5
    d = [t.to(device) for t in (q, k, v)]
    st = ops.block_stats(*d, BT, 4)
    assert bool((st.vc[0, 0, 4] > 65520).all()) and bool((st.hgroup.abs() < 65504).all())
    o = ops.sparse_attn(*d, st, sel, scale, BT, group_size=4).double().cpu()
    ref = O.pisa_pg_attention(q, k, v, 0.5, BT, 4, scale, dtype=torch.float64, indices=idx)
    err = float((o - ref).norm() / ref.norm())
    print(f"[edges] fp16 value sum BT={BT} D={D}: rel {err:.2e}", flush=True)
    assert err <= 2e-3


@pytest.mark.parametrize("heads,T,D,BT,G,dtype", [(2, 1024, 64, 64, 32, F32), (1, 777, 37, 16, 50, F16),
                                                  (3, 1000, 96, 32, 16, B16), (1, 300, 128, 256, 2, F32),
                                                  (2, 3001, 64, 64, 32, B16), (1, 4099, 64, 128, 32, B16)])
def test_block_stats_split_any(device, heads, T, D, BT, G, dtype):
    """A group split over several workgroups (any-shape kernels and the head_dim 64 ones): the per-block statistics are the unsplit call's bit for
    bit, and the group moment differs by the order of at most G sums (G 2^-24 of the sum of their
    magnitudes).  A workspace smaller than asked for is used as far as it reaches."""
    from pasa_amd import _lib
    q, k, v = (t.to(device) for t in make(heads, T, D, dtype, T + D))
    lib = _lib.load()
    need = lib.pasa_block_stats_workspace_bytes_dtype(heads, T, 0, D, BT, G, ops._DTYPES[dtype])
    assert need > 0
    one = ops.block_stats(q, k, v, BT, G, split=False)
    runs = [ops.block_stats(q, k, v, BT, G)]
    for nbytes in (need // 2, 4):
        st = ops.BlockStats(*(torch.full_like(getattr(one, n), float("nan"))
                              for n in ("qc", "kc", "vc", "hnorm", "hgroup")))
        ws = torch.empty(need, dtype=torch.uint8, device=device)
        _lib.call("pasa_block_stats_ws", q.data_ptr(), k.data_ptr(), v.data_ptr(), st.qc.data_ptr(), st.kc.data_ptr(),
                  st.vc.data_ptr(), st.hnorm.data_ptr(), st.hgroup.data_ptr(), heads, T, 0, D, BT, G,
                  ops._DTYPES[dtype], ws.data_ptr(), nbytes, ops._stream(q))
        torch.cuda.synchronize()
        runs.append(st)
    ref = O.block_stats(*(t.cpu().reshape(heads, T, D) for t in (q, k, v)), BT, dtype=torch.float64)
    bound = G * 2.0 ** -24 * O.group_moment(ref.hc.abs(), G) + 1e-6
    for st in runs:
        for n in ("qc", "kc", "vc", "hnorm"):
            assert torch.equal(getattr(st, n), getattr(one, n)), n
        diff = (st.hgroup - one.hgroup).abs().double().cpu().reshape(bound.shape)
        assert bool((diff <= bound).all())


@pytest.mark.parametrize("heads,NT,D", [(1, 1, 1), (2, 63, 127), (1, 65, 96), (2, 130, 38), (1, 64, 100)])
def test_scores_any(device, heads, NT, D):
    """Selection scores at the edges of the 64 x 64 tile and at head dims that are not whole 16-byte
    pieces, against 64 bits: a chain of D fused multiply-adds, each rounding at most 2^-24 of the
    running sum's bound sum |q k|, and the log and the two additions about as much again."""
    g = torch.Generator().manual_seed(NT + D)
    qc, kc = (torch.randn(1, heads, NT, D, generator=g) for _ in range(2))
    hn = torch.rand(1, heads, NT, generator=g) + 0.5
    st = ops.BlockStats(qc.to(device), kc.to(device), torch.empty(0), hn.to(device), torch.empty(0))
    sel = ops.select_blocks(st, 0.3, 0.37, return_scores=True)
    ref = O.select_scores(qc.double(), kc.double(), hn.double(), 0.37)
    mag = O.select_scores(qc.double().abs(), kc.double().abs(), hn.double(), 0.37, use_cov_bias=False)
    assert bool(((sel.scores.cpu().double() - ref).abs() <= (D + 8) * 2.0 ** -24 * (mag + 1)).all())
    idx = O.topk_indices(sel.scores.cpu(), sel.ns)
    assert torch.equal(idx.reshape(sel.idx.shape), sel.idx.cpu())


@pytest.mark.parametrize("T, BT, shift", [(64, 64, 1), (1000, 64, 3), (1000, 128, 4), (4500, 64, 5), (4500, 128, 1)])
def test_head_dim_64_takes_misaligned_data(device, T, BT, shift):
    """bf16 head dim 64 on data that is not 16-byte aligned: staged through registers, the same bits."""
    q, k, v = make(2, T, 64, B16, T + BT)
    outs = []
    for n in (0, shift):
        d = [to_dev(t, device, n) for t in (q, k, v)]
        st = ops.block_stats(*d, BT)
        sel = ops.select_blocks(st, 0.2, 64 ** -0.5)
        outs.append((st.qc, st.kc, st.vc, st.hnorm, st.hgroup, ops.sparse_attn(*d, st, sel, 64 ** -0.5, BT)))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T, BT, text, valid, dtype, shift", [(128, 128, 0, 0, B16, 1), (1000, 128, 0, 0, F16, 4),
                                                              (1000, 64, 0, 0, B16, 3), (4500, 64, 70, 9, F16, 5),
                                                              (4500, 128, 200, 130, B16, 2), (5000, 128, 0, 0, B16, 7)])
def test_head_dim_128_takes_misaligned_data(device, T, BT, text, valid, dtype, shift):
    """16-bit head dim 128 on data that is not 16-byte aligned: staged through registers, the same bits."""
    q, k, v = make(2, T, 128, dtype, T + BT)
    outs = []
    for n in (0, shift):
        d = [to_dev(t, device, n) for t in (q, k, v)]
        st = ops.block_stats(*d, BT, text_tokens=text)
        sel = ops.select_blocks(st, 0.2, 128 ** -0.5)
        kw = dict(text_tokens=text, text_valid=valid)
        outs.append((st.qc, st.kc, st.vc, st.hnorm, st.hgroup, ops.sparse_attn(*d, st, sel, 128 ** -0.5, BT, **kw),
                     ops.dense_attention(*d, **kw), ops.dense_attention(*d, token_major_out=True, **kw),
                     ops.cross_attention(d[0], *(to_dev(t[:, :, :77].contiguous(), device, n) for t in (k, v)))))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype, shift", [(B16, 1), (F16, 6)])
def test_placed_call_takes_misaligned_data(device, dtype, shift):
    """The same for the frame-major call: its inputs, and the token-major k and v its second half reads."""
    frames, size, text = 5, 210, 40
    q, k, v = make(2, frames * size + text, 128, dtype, 5)
    pl = ops.Placement(frames, size)
    outs = []
    for n in (0, shift):
        d = [to_dev(t, device, n) for t in (q, k, v)]
        st = ops.block_stats(*d, 128, text_tokens=text, placement=pl)
        sel = ops.select_blocks(st, 0.3, 128 ** -0.5)
        pack = ops.pack_phase2(d[0], st, 128, text)
        tm = [to_dev(t, device, n) for t in (st.k_tm, st.v_tm)]
        o = ops.sparse_attn_packed(d[0], *tm, pack, sel, 128 ** -0.5, 128, text_tokens=text, placement=pl)
        outs.append((st.qc, st.kc, st.vc, st.hnorm, st.hgroup, st.k_tm, st.v_tm, o))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T, D, BT, dtype, shift", [(700, 64, 64, B16, 8), (700, 64, 128, B16, 2), (700, 128, 64, F16, 4),
                                                    (4500, 128, 128, B16, 12)])
def test_pack_takes_any_address(device, T, D, BT, dtype, shift):
    """A phase-2 pack (or workspace) that is not 16-byte aligned: the same bits."""
    q, k, v = (t.to(device) for t in make(2, T, D, dtype, T + BT))
    st = ops.block_stats(q, k, v, BT)
    sel = ops.select_blocks(st, 0.2, D ** -0.5)
    pack = ops.pack_phase2(q, st, BT)
    moved = torch.empty(pack.numel() + shift, dtype=torch.uint8, device=device)[shift:]
    ops._lib.call("pasa_pack_phase2", st.kc.data_ptr(), st.vc.data_ptr(), st.hgroup.data_ptr(), moved.data_ptr(),
                  moved.numel(), 2, T, 0, D, BT, 32, ops._DTYPES[dtype], ops._stream(q))
    a, b = (ops.sparse_attn_packed(q, k, v, p, sel, D ** -0.5, BT) for p in (pack, moved))
    assert torch.equal(a, b)


@pytest.mark.parametrize("D, shift", [(64, 1), (128, 2), (128, 3)])
def test_scores_take_any_address(device, D, shift):
    """Block means that are not 16-byte aligned, at the head dims of the tuned score kernel: the bound of
    test_scores_any against 64 bits."""
    g = torch.Generator().manual_seed(D + shift)
    qc, kc = (torch.randn(1, 2, 130, D, generator=g) for _ in range(2))
    hn = torch.rand(1, 2, 130, generator=g) + 0.5
    st = ops.BlockStats(to_dev(qc, device, shift), to_dev(kc, device, shift), torch.empty(0), to_dev(hn, device, shift),
                        torch.empty(0))
    sel = ops.select_blocks(st, 0.3, 0.37, return_scores=True)
    ref = O.select_scores(qc.double(), kc.double(), hn.double(), 0.37)
    mag = O.select_scores(qc.double().abs(), kc.double().abs(), hn.double(), 0.37, use_cov_bias=False)
    assert bool(((sel.scores.cpu().double() - ref).abs() <= (D + 8) * 2.0 ** -24 * (mag + 1)).all())


@pytest.mark.parametrize("case", ["nan_row", "infinite_unselected", "infinite_selected", "out_of_scaled_range"])
@pytest.mark.parametrize("BT,D,G", [(64, 64, 3), (64, 128, 32), (128, 100, 2), (256, 37, 1)])
def test_fp32_tiles_done_again(device, BT, D, G, case):
    """Sparse fp32 calls whose tiles are not finite in the split form and are computed again in fp32, after
    phase 2 has used their LDS for the sums and moments: the rows and features that are finite come out as
    the oracle's, the others are not finite."""
    NT = 9
    T = NT * BT - 5
    q, k, v = make(1, T, D, F32, T + D)
    rows = [{3, *[j % NT for j in (i, i + 2, i + 5, i + 4) if j % NT not in (3, 6)][:2]} for i in range(NT)]
    sel, idx = selection(rows, device)
    bad_rows = torch.zeros(T, dtype=torch.bool)
    bad_cols = torch.zeros(D, dtype=torch.bool)
    qb, vb = q.clone(), v.clone()
    if case == "nan_row":
        qb[0, 0, 2 * BT + 1, 0] = torch.nan
        bad_rows[2 * BT + 1] = True
    elif case == "out_of_scaled_range":
        vb = v = v * 2.0 ** 95                               # finite, but not times 2^56
    else:
        vb[0, 0, (6 if case == "infinite_unselected" else 3) * BT + 7, 11] = torch.inf
        bad_cols[11] = True
    scale = D ** -0.5
    d = [t.to(device) for t in (qb, k, vb)]
    st = ops.block_stats(*d, BT, G)
    o = ops.sparse_attn(*d, st, sel, scale, BT, group_size=G).double().cpu()[0, 0]
    ref = O.pisa_pg_attention(q, k, v, 0.5, BT, G, scale, dtype=torch.float64, indices=idx)[0, 0]
    assert bool(torch.isnan(o[bad_rows]).all())
    a, b = o[~bad_rows][:, ~bad_cols], ref[~bad_rows][:, ~bad_cols]
    err = float((a - b).norm() / b.norm())
    print(f"[edges] fp32 again BT={BT} D={D} G={G} {case}: rel {err:.2e}", flush=True)
    assert err <= 4e-6
    if bad_cols.any():
        assert not bool(torch.isfinite(o[:, bad_cols]).any())
