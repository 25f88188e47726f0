"""The SDPA adapter's dense forward, in place through strides, against the
packed path on the same inputs (the same kernels on packed copies)."""

import pytest
import torch

from tests.helpers import REF_ATOL, randn

pytestmark = pytest.mark.gpu


def _tensor(layout, B, H, N, D, dtype, g):
    if layout == "bhnd":
        return randn((B, H, N, D), dtype, g).cuda()
    if layout == "bnhd":                      # a projection's [B, N, H, D], transposed
        return randn((B, N, H, D), dtype, g).cuda().transpose(1, 2)
    if layout == "slice":                     # rows and heads inside a wider tensor
        return randn((B, H, N + 3, D + 16), dtype, g).cuda()[:, :, 2:N + 2, 8:D + 8]
    return randn((1, H, N, D), dtype, g).cuda().expand(B, H, N, D)    # "shared": one batch for all


@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nkv,D,dtype,layout,mask,causal", [
    (2, 8, 2, 300, 300, 128, torch.bfloat16, "bhnd", None, True),
    (3, 4, 4, 257, 257, 64, torch.float16, "bnhd", None, False),
    (1, 16, 4, 1025, 1025, 64, torch.bfloat16, "bnhd", None, True),
    (2, 4, 4, 33, 129, 80, torch.float16, "slice", None, False),
    (2, 8, 8, 100, 700, 128, torch.float16, "shared", None, True),
    (2, 4, 2, 64, 64, 96, torch.bfloat16, "bhnd", None, True),
    (2, 4, 4, 70, 70, 88, torch.bfloat16, "bnhd", "bool", False),
    (2, 8, 1, 130, 128, 128, torch.bfloat16, "bnhd", "float", False),
    (2, 8, 2, 130, 131, 64, torch.float16, "bhnd", "heads", False),
    (40, 16, 16, 512, 512, 128, torch.bfloat16, "bhnd", None, False),   # beyond the small-grid kernels
])
def test_dense_matches_packed(monkeypatch, B, Hq, Hkv, Nq, Nkv, D, dtype, layout, mask, causal):
    import mtlattn_amd as mt
    print(f"\n[case] dense {layout} {B}x{Hq}/{Hkv} {Nq}x{Nkv} D={D} {dtype} mask={mask} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(2)
    q = _tensor("bnhd" if layout == "shared" else layout, B, Hq, Nq, D, dtype, g)
    k, v = (_tensor(layout, B, Hkv, Nkv, D, dtype, g) for _ in range(2))
    m = None
    if mask == "bool":
        m = torch.rand(B, 1, Nq, Nkv, generator=g).cuda() < 0.6
        m[..., 0] = True
    elif mask == "float":
        m = torch.randn(Nq, Nkv, generator=g).cuda()
    elif mask == "heads":
        m = torch.randn(B, Hq, Nq, Nkv, generator=g).cuda()
    with torch.no_grad():
        assert mt._dense(q, k, v, 0.1, causal,
                         bias=None if m is None else mt._sdpa_mask_to_bias(m, B, Hq, Nq, Nkv)) is not None
        out = mt.sdpa(q, k, v, m, is_causal=causal)
        monkeypatch.setattr(mt, "_dense", lambda *a, **kw: None)
        ref = mt.sdpa(q, k, v, m, is_causal=causal)
    assert out.is_contiguous() and out.shape == ref.shape
    assert torch.equal(out, ref)


@pytest.mark.parametrize("B,Hq,Hkv,N,D,dtype,layout,causal", [
    (4, 8, 8, 257, 64, torch.bfloat16, "bhnd", False),
    (5, 8, 2, 300, 128, torch.float16, "bnhd", True),
    (3, 4, 4, 64, 80, torch.bfloat16, "slice", False),
])
def test_dense_padding_matches_packed(monkeypatch, B, Hq, Hkv, N, D, dtype, layout, causal):
    """Key-padding lengths (0, 1, a tile's edge, all): padded query rows are 0."""
    import mtlattn_amd as mt
    print(f"\n[case] dense padding {layout} {B}x{Hq}/{Hkv}x{N} D={D} {dtype} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(4)
    q = _tensor(layout, B, Hq, N, D, dtype, g)
    k, v = (_tensor(layout, B, Hkv, N, D, dtype, g) for _ in range(2))
    lens = torch.tensor([N, 0, 1, 32, N - 1][:B], device="cuda")
    m = (torch.arange(N, device="cuda")[None] < lens[:, None])[:, None, None, :]
    assert mt._dense(q, k, v, 0.1, causal, lens.int()) is not None
    out = mt._try_padding_varlen(q, k, v, m, causal, 0.1)
    monkeypatch.setattr(mt, "_dense", lambda *a, **kw: None)
    ref = mt._try_padding_varlen(q, k, v, m, causal, 0.1)
    assert torch.equal(out, ref)
    for b in range(B):
        assert not out[b, :, lens[b]:].any()


def test_dense_refusals():
    """Calls the dense kernels do not take go through the packed path."""
    import mtlattn_amd as mt
    x = lambda *s, dt=torch.bfloat16: torch.randn(s, device="cuda").to(dt)   # noqa: E731
    q = x(2, 4, 64, 128)
    assert mt._dense(q, q, q, 0.1, False) is not None
    for a, kw in (((q.float(),) * 3, {}), ((x(2, 4, 64, 72),) * 3, {}), ((x(2, 4, 64, 256),) * 3, {}),
                  ((x(2, 4, 8, 128),) * 3, {}), ((x(2, 4, 64, 136)[..., 1:129],) * 3, {}),
                  ((x(2, 4, 128, 64).transpose(2, 3),) * 3, {}), ((q, q, x(2, 4, 65, 128)), {}),
                  ((q.clone().requires_grad_(), q, q), {})):
        assert mt._dense(*a, 0.1, False, **kw) is None, [tuple(t.shape) for t in a]
    assert mt._dense(q, q, q, -0.1, False) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_padding_mask_rewritten_or_made_in_inference_mode(dtype):
    """Under replace_sdpa() a key-padding mask is taken as it is at each call:
    rewritten through .data (the version counter stays), made under
    inference_mode (it has none), turned into another kind of mask; and a call
    recorded into a graph repeats what it recorded. Valid rows against the
    original on fp32 copies."""
    import mtlattn_amd as mt
    print(f"\n[case] padding mask content {dtype}", flush=True)
    B, H, N, D = 3, 4, 130, 64
    g = torch.Generator().manual_seed(9)
    q, k, v = (randn((B, H, N, D), dtype, g).cuda() for _ in range(3))
    j = torch.arange(N, device="cuda")
    orig = torch.nn.functional.scaled_dot_product_attention

    def prefix(lens):
        return (j[None] < torch.tensor(lens, device="cuda")[:, None])[:, None, None, :]

    def check(m, lens):
        out = torch.nn.functional.scaled_dot_product_attention(q, k, v, attn_mask=m)
        ref = orig(q.float().cpu(), k.float().cpu(), v.float().cpu(), attn_mask=prefix(lens).cpu()).cuda()
        for b, n in enumerate(lens):
            assert (out[b, :, :n].float() - ref[b, :, :n]).abs().max() < (2e-2 if dtype == torch.bfloat16 else 1e-5)
            assert not out[b, :, n:].any()
        return out

    mt.replace_sdpa(min_seqlen=64)
    try:
        with torch.no_grad():
            m = prefix([130, 64, 1])
            for _ in range(3):
                check(m, [130, 64, 1])
            m.data.copy_(prefix([100, 130, 33]))
            for _ in range(2):
                want = check(m, [100, 130, 33])
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = torch.nn.functional.scaled_dot_product_attention(q, k, v, attn_mask=m)
            for _ in range(3):
                out.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, want)
                check(m, [100, 130, 33])
            m.data[:, :, :, 0] = False                      # no prefix any more: padded rows attend too
            got = torch.nn.functional.scaled_dot_product_attention(q, k, v, attn_mask=m)
            assert torch.equal(got, orig(q, k, v, attn_mask=m))
        with torch.inference_mode():
            m = prefix([5, 130, 70])
            for _ in range(2):
                check(m, [5, 130, 70])
    finally:
        mt.restore_sdpa()


@pytest.mark.parametrize("layout,D,dtype", [("bhnd", 64, torch.bfloat16), ("bnhd", 128, torch.float16)])
def test_dense_nan(monkeypatch, layout, D, dtype):
    """NaN in padding rows of q, k and v reaches nothing; NaN in a token's k
    reaches the rows that see it, as on the packed path."""
    import mtlattn_amd as mt
    print(f"\n[case] dense NaN {layout} D={D} {dtype}", flush=True)
    B, H, N = 3, 4, 200
    g = torch.Generator().manual_seed(6)
    q, k, v = (_tensor(layout, B, H, N, D, dtype, g) for _ in range(3))
    lens = torch.tensor([200, 65, 0], device="cuda", dtype=torch.int32)
    pad = (torch.arange(N, device="cuda")[None] >= lens[:, None])[:, None, :, None]
    for causal in (False, True):
        ref = mt._dense(q, k, v, 0.1, causal, lens)
        bad = [t.masked_fill(pad, float("nan")) for t in (q, k, v)]
        assert torch.equal(mt._dense(*bad, 0.1, causal, lens), ref)
        bad[1][0, 2, 150, 3] = float("nan")
        out = mt._dense(*bad, 0.1, causal, lens)
        want = torch.zeros_like(out, dtype=torch.bool)
        want[0, 2, 150 if causal else 0:] = True
        assert torch.equal(out.isnan(), want)
        # (at D = 64 a NaN row makes its wave take the row maxima again: other roundings of P)
        assert (out.nan_to_num() - ref.masked_fill(want, 0)).abs().max().item() < REF_ATOL[dtype]


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4099, 1 << 20, (9 << 20) + 5])
@pytest.mark.parametrize("skew", [0, 3])
def test_content_differs(n, skew):
    """One byte of difference anywhere is found: first, last, at the edges of
    the 16-byte part; the bytes around the tensors do not count."""
    from mtlattn_amd import _C
    print(f"\n[case] content_differs {n} bytes at +{skew}", flush=True)
    g = torch.Generator().manual_seed(n)
    x = torch.randint(0, 256, (n + skew + 8,), generator=g, dtype=torch.uint8).cuda()
    y = x.clone()
    y[n + skew:] += 1
    a, b = x[skew:skew + n], y[skew:skew + n]

    def differs():
        flag = torch.zeros((), dtype=torch.int32, pin_memory=True)
        _C.content_differs(a, b, flag)
        torch.cuda.synchronize()
        return flag.item()

    assert differs() == 0
    for i in sorted({0, n // 2, n - 1, max(0, n // 16 * 16 - 1), min(n - 1, n // 16 * 16)}):
        b[i] += 1
        assert differs() == 1, i
        b[i] -= 1
    assert differs() == 0
