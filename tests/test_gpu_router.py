"""GPU parity of the MoE-router entry points (deltanet.metal:863-900,
2229-2329). qff_q8_dequant must be bit-exact with the closed form.
qff_router_top8: logits within rel 1e-5 (max-abs over max |logit|) of the
fp64 dense product; indices equal to the oracle's top-8 rule applied to the
kernel's own logits, and to the oracle's logits where the eight winners are
separated from the rest by more than the logit tolerance; scores within
1e-6 of the oracle's on the kernel's logits."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, bf16_tensor, f16_tensor, f32_tensor, to_np
from oracle import oracle as O
from qff import synth

pytestmark = pytest.mark.gpu


def _w_gpu(w, s, b, sb):
    conv = f16_tensor if sb == "f16" else bf16_tensor
    return torch.from_numpy(w.view(np.int32)).to(DEV), conv(s), conv(b)


@pytest.mark.parametrize("rows,cols,sb", [(256, 2048, "bf16"), (17, 64, "f16"), (40, 4096, "bf16")])
def test_q8_dequant_bit_exact(hip, rows, cols, sb):
    import qff
    print(f"q8_dequant {rows}x{cols} {sb}", flush=True)
    w, s, b = synth.q8_weight(rows, cols, seed=rows + cols, sb_dtype=sb)
    ctx = qff.Context(max_batch=1, max_ctx=64, max_prefill_tokens=1)
    out = qff.q8_dequant(ctx, *_w_gpu(w, s, b, sb))
    torch.cuda.synchronize()
    ref = O.q8_dequant(w, s, b, O.F16 if sb == "f16" else O.BF16)
    assert np.array_equal(to_np(out).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("batch,experts,cols,xdt", [(1, 256, 2048, "f32"), (5, 256, 2048, "bf16"),
                                                    (32, 256, 2048, "f32"), (300, 256, 2048, "f32"),
                                                    (3, 64, 1024, "f32"), (2, 8, 4096, "bf16"),
                                                    (9, 100, 192, "f32")])
def test_router_top8(hip, batch, experts, cols, xdt):
    import qff
    print(f"router_top8 batch={batch} experts={experts} cols={cols} x={xdt}", flush=True)
    w, s, b = synth.q8_weight(experts, cols, seed=experts + cols + batch)
    rng = np.random.default_rng(batch)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    if xdt == "bf16":
        x = O.round_bf16(x)
        xt = bf16_tensor(O.f32_to_bf16(x))
    else:
        xt = f32_tensor(x)
    ctx = qff.Context(max_batch=1, max_ctx=64, max_prefill_tokens=1)
    idx, sc, lg = qff.router_top8(ctx, *_w_gpu(w, s, b, "bf16"), xt)
    torch.cuda.synchronize()
    idx, sc, lg = idx.cpu().numpy(), sc.cpu().numpy(), lg.cpu().numpy()
    dense = O.q8_dequant(w, s, b, O.BF16).astype(np.float64)
    ref_lg = x.astype(np.float64) @ dense.T
    tol = 1e-5 * np.max(np.abs(ref_lg))
    assert np.max(np.abs(lg - ref_lg)) <= tol
    for m in range(batch):
        oi, os_ = O.router_top8(lg[m])
        assert np.array_equal(idx[m], oi)
        assert np.allclose(sc[m], os_, atol=1e-6)
        # against the oracle's own logits where the ranking is unambiguous
        ol = O.router_logits(w, s, b, x[m], O.BF16)
        srt = np.sort(ol.astype(np.float64))[::-1]
        gaps = np.diff(srt[:9])
        if np.all(np.abs(gaps) > 4 * tol):
            assert np.array_equal(idx[m], O.router_top8(ol)[0])


@pytest.mark.parametrize("batch,experts,cols,xdt,sb", [
    (2, 256, 2048, "f32", "bf16"), (17, 256, 2048, "bf16", "f16"),     # one tile per workgroup, a ragged token block
    (257, 40, 4096, "f32", "bf16"), (300, 256, 64, "f32", "f16"),      # two tiles; one group of columns
    (600, 250, 2048, "bf16", "bf16"), (1000, 8, 1088, "f32", "bf16"),  # four tiles; fewer experts than a tile
    (2577, 256, 2048, "f32", "bf16"), (2600, 100, 576, "bf16", "f16")  # whole blocks; a ragged slab of columns
])
def test_router_top8_many_tokens(hip, batch, experts, cols, xdt, sb):
    """The matrix-core logits at the edges of their tiles, with tokens scaled
    by 2^-60 .. 2^60 and an all-zero token: every token within 1e-6 of the
    fp64 product relative to its own sum of |W x| (fp32 sums of exact
    products: a few 2^-24), the ranking that of the kernel's own logits."""
    import qff
    print(f"router_top8 batch={batch} experts={experts} cols={cols} x={xdt} scales={sb}", flush=True)
    w, s, b = synth.q8_weight(experts, cols, seed=experts + cols + batch, sb_dtype=sb)
    rng = np.random.default_rng(batch)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x *= np.exp2(rng.integers(-60, 61, (batch, 1))).astype(np.float32)
    x[batch // 2] = 0.0
    if xdt == "bf16":
        x = O.round_bf16(x)
    xt = bf16_tensor(O.f32_to_bf16(x)) if xdt == "bf16" else f32_tensor(x)
    ctx = qff.Context(max_batch=1, max_ctx=64, max_prefill_tokens=1)
    idx, sc, lg = qff.router_top8(ctx, *_w_gpu(w, s, b, sb), xt)
    torch.cuda.synchronize()
    idx, sc, lg = idx.cpu().numpy(), sc.cpu().numpy(), lg.cpu().numpy()
    dense = O.q8_dequant(w, s, b, O.F16 if sb == "f16" else O.BF16).astype(np.float64)
    err = np.abs(lg - x.astype(np.float64) @ dense.T)
    assert np.all(err <= 1e-6 * (np.abs(x).astype(np.float64) @ np.abs(dense).T))
    order = np.argsort(-lg, axis=1, kind="stable")[:, :8]
    assert np.array_equal(idx, order)
    top = np.take_along_axis(lg, order, 1).astype(np.float64)
    p = np.exp(top - top[:, :1])
    assert np.allclose(sc, p / p.sum(1, keepdims=True), atol=1e-6)


@pytest.mark.parametrize("batch,xdt", [(2, "f32"), (17, "bf16"), (40, "f32"), (40, "bf16"), (300, "f32"),
                                       (300, "bf16"), (1000, "f32"), (1000, "bf16"), (2600, "f32"), (2600, "bf16")])
def test_router_logits_keep_every_bit_of_x(hip, batch, xdt):
    """Scale 1, bias -128 and bytes of 128 except one 129 per expert: the
    logit is one element of x. With (q - 128) x exact it is that element bit
    for bit, also where it sits 2^-110 below the rest of its 64 columns."""
    import qff
    print(f"router exact x batch={batch} x={xdt}", flush=True)
    E, C = 256, 2048
    rng = np.random.default_rng(batch)
    q = np.full((E, C), 128, np.uint8)
    col = rng.permutation(C)[:E]
    q[np.arange(E), col] = 129
    x = (rng.uniform(1, 2, (batch, C)) * np.exp2(rng.integers(-110, 1, (batch, C)))).astype(np.float32)
    x *= rng.choice(np.float32([-1, 1]), (batch, C))
    if xdt == "bf16":
        x = O.round_bf16(x)
    xt = bf16_tensor(O.f32_to_bf16(x)) if xdt == "bf16" else f32_tensor(x)
    one, bias = (bf16_tensor(O.f32_to_bf16(np.full((E, C // 64), v, np.float32))) for v in (1.0, -128.0))
    ctx = qff.Context(max_batch=1, max_ctx=64, max_prefill_tokens=1)
    _, _, lg = qff.router_top8(ctx, torch.from_numpy(q.view(np.int32)).to(DEV), one, bias, xt)
    torch.cuda.synchronize()
    assert np.array_equal(lg.cpu().numpy(), x[:, col])


@pytest.mark.parametrize("batch,experts,cols,xdt,sb", [(4, 256, 2048, "f32", "bf16"), (40, 256, 4096, "bf16", "f16"),
                                                       (300, 250, 2048, "bf16", "bf16"), (300, 256, 64, "f32", "f16"),
                                                       (1000, 256, 2048, "f32", "bf16"), (1000, 40, 320, "bf16", "f16"),
                                                       (2600, 256, 2048, "f32", "f16"), (2600, 100, 576, "bf16", "bf16")])
def test_router_special_tokens(hip, batch, experts, cols, xdt, sb):
    """Tokens with infinities or NaN in a batch: their logits and ranking are
    bit for bit those of a call with that token alone, and the other tokens'
    those of a batch that has zeros in their place. A token of magnitudes up to
    2^126: finite wherever that call's logit is, and within 1e-6 of the fp64
    product relative to its sum of |W x| wherever finite."""
    import qff
    print(f"router special tokens batch={batch} experts={experts} cols={cols} x={xdt} scales={sb}", flush=True)
    w, s, b = synth.q8_weight(experts, cols, seed=experts + cols + batch, sb_dtype=sb)
    rng = np.random.default_rng(batch + cols)
    conv = f16_tensor if sb == "f16" else bf16_tensor
    # biases of both signs: q x and b sum(x) both infinite, of one sign or two
    bf = rng.choice(np.float32([-0.2, 0.05]), b.shape)
    wt = (torch.from_numpy(w.view(np.int32)).to(DEV), conv(s), conv(O.f32_to_f16(bf) if sb == "f16" else O.f32_to_bf16(bf)))
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    spec = sorted({0, 1, batch // 2, batch - 1} if batch > 4 else {0, 1, 2})
    plain = x.copy()
    plain[spec] = 0.0
    x[spec[0], 5] = np.inf
    x[spec[1], [3, cols - 1]] = np.inf, -np.inf
    x[spec[2]] = np.clip(x[spec[2]], -3, 3) * 2.0 ** (118 if batch % 20 else 124)
    if len(spec) > 3:
        x[spec[3], cols // 2] = np.nan
    mk = (lambda v: bf16_tensor(O.f32_to_bf16(v))) if xdt == "bf16" else f32_tensor
    ctx = qff.Context(max_batch=1, max_ctx=64, max_prefill_tokens=1)
    xt = mk(x)
    idx, sc, lg = (t.cpu().numpy() for t in qff.router_top8(ctx, *wt, xt))
    pidx, _, plg = (t.cpu().numpy() for t in qff.router_top8(ctx, *wt, mk(plain)))
    rest = np.setdiff1d(np.arange(batch), spec)
    assert np.array_equal(lg[rest], plg[rest]) and np.array_equal(idx[rest], pidx[rest])
    huge = spec.pop(2)
    l1 = qff.router_top8(ctx, *wt, xt[huge:huge + 1].clone())[2].cpu().numpy()[0]
    dense = O.q8_dequant(w, s, O.f32_to_f16(bf) if sb == "f16" else O.f32_to_bf16(bf),
                         O.F16 if sb == "f16" else O.BF16).astype(np.float64)
    xh = xt[huge].double().cpu().numpy()
    fin = np.isfinite(lg[huge])
    assert np.all(fin[np.isfinite(l1)])
    assert np.all(np.abs(lg[huge] - dense @ xh)[fin] <= 1e-6 * (np.abs(dense) @ np.abs(xh))[fin])
    for m in spec:
        i1, s1, l1 = (t.cpu().numpy()[0] for t in qff.router_top8(ctx, *wt, xt[m:m + 1].clone()))
        assert np.array_equal(lg[m], l1, equal_nan=True), m
        assert np.array_equal(idx[m], i1) and np.array_equal(sc[m], s1, equal_nan=True)
    assert np.isinf(lg[spec[0]]).any()   # where the bias is positive


def test_router_rejects_bad_calls(hip):
    import qff
    from qff._lib import lib
    ctx = qff.Context(max_batch=1, max_ctx=64, max_prefill_tokens=1)
    w, s, b = _w_gpu(*synth.q8_weight(300, 128, seed=1), "bf16")
    x = torch.zeros(1, 128, device=DEV)
    with pytest.raises(qff.QffError) as e:
        qff.router_top8(ctx, w, s, b, x)           # 300 experts > 256
    assert e.value.status == -2
    L = lib()
    assert L.qff_router_top8(ctx.handle, None, w.data_ptr(), s.data_ptr(), b.data_ptr(), 1, x.data_ptr(), 0,
                             None, None, None, 256, 128, 1) == -1
