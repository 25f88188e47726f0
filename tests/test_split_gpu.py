"""The forward's work splits on small grids: one-workgroup decode (whole
sequences, and chunks of a short stream) and the flash forward's key pieces,
against the oracle and against the unsplit flash forward."""

import ctypes
import math

import pytest
import torch

import oracle
from mtlattn_amd import capi
from tests.helpers import LSE_TOL, REF_ATOL, cu_of, randn

pytestmark = pytest.mark.gpu


def _inputs(q_lens, kv_lens, Hq, Hkv, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return (randn((sum(q_lens), Hq, D), dtype, g), randn((sum(kv_lens), Hkv, D), dtype, g),
            randn((sum(kv_lens), Hkv, D), dtype, g))


def _fwd(q, k, v, cq, ck, max_q, causal, window, bias, workspace):
    """(out, lse, workspace bytes) of mtlattn_varlen_fwd on NaN-filled outputs,
    with the queried workspace (NaN-filled) or none."""
    Hq, D, Hkv = q.shape[1], q.shape[2], k.shape[1]
    p = capi.problem_for(q, k, cq, ck, max_q, 1.0 / math.sqrt(D), causal=causal, window=window, bias=bias)
    need = capi.lib().mtlattn_varlen_fwd_workspace_size(ctypes.byref(p))
    n = need if workspace else 0
    ws = torch.full((max(n // 4, 1),), float("nan"), dtype=torch.float32, device="cuda")
    out = torch.full_like(q, float("nan"))
    lse = torch.full((q.shape[0], Hq), float("nan"), dtype=torch.float32, device="cuda")
    capi.call("mtlattn_varlen_fwd", p, q.data_ptr(), Hq * D, k.data_ptr(), Hkv * D, v.data_ptr(), Hkv * D,
              out.data_ptr(), lse.data_ptr(), ws.data_ptr() if n else None, n, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out.cpu(), lse.cpu(), need


def _check(name, out, lse, ref, ref_lse, dtype):
    fin = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse), fin), f"{name}: LSE -inf pattern"
    assert torch.isfinite(out.float()).all(), name
    assert (out.float() - ref).abs().max().item() < REF_ATOL[dtype], name
    assert (lse[fin] - ref_lse[fin]).abs().max().item() < LSE_TOL[dtype], name


@pytest.mark.parametrize("q_lens,kv_lens,Hq,Hkv,D,dtype,causal,window,bias", [
    ([1] * 9, [1, 31, 32, 33, 127, 128, 129, 0, 1000], 8, 2, 128, torch.bfloat16, True, 0, None),
    ([1, 0, 4, 16, 7], [300, 50, 9, 16, 513], 16, 2, 128, torch.float16, True, 0, None),
    ([3, 5], [260, 700], 12, 12, 64, torch.bfloat16, False, 0, None),
    ([1] * 70, list(range(1, 281, 4)), 32, 8, 64, torch.float16, True, 0, None),       # more than one item per CU
    ([1, 2, 1], [900, 1500, 40], 8, 8, 128, torch.bfloat16, True, 100, None),
    ([2, 1], [700, 333], 16, 4, 128, torch.float16, True, 0, "head"),
    ([1, 3], [530, 1200], 8, 2, 64, torch.bfloat16, True, 300, "broadcast"),
    ([1], [1999], 8, 2, 128, torch.bfloat16, True, 0, None),                            # few sequences: chunks
    ([2, 1], [5000, 2047], 16, 16, 128, torch.float16, True, 0, None),
    ([1], [40000], 8, 2, 64, torch.bfloat16, True, 0, None),
])
def test_decode_workgroup(q_lens, kv_lens, Hq, Hkv, D, dtype, causal, window, bias):
    """Few-query calls on one workgroup per item: key counts around a tile and
    around the waves' share, empty sequences, rows with no key (more queries
    than keys), head groups of several rows, windows, biases, chunked calls.
    O and LSE against the oracle; a call without a workspace (whole sequences)
    where fewer than 2048 keys a sequence allow one."""
    print(f"\n[case] decode workgroup D={D} {dtype} {q_lens[:5]} {kv_lens[:9]} window={window} bias={bias}", flush=True)
    q, k, v = _inputs(q_lens, kv_lens, Hq, Hkv, D, dtype, 3)
    cq, ck = cu_of(q_lens), cu_of(kv_lens)
    b = None
    if bias:
        b = torch.randn(sum(q_lens), 1 if bias == "broadcast" else Hq, max(kv_lens),
                        generator=torch.Generator().manual_seed(4))
    ref, ref_lse = oracle.varlen_forward(q, k, v, cq, ck, 1.0 / math.sqrt(D), causal, window, b)
    dev = [t.cuda() for t in (q, k, v, cq, ck)]
    bd = None if b is None else b.cuda()
    for ws in (True, False):
        if not ws and sum(kv_lens) // len(kv_lens) >= 2048:
            continue
        out, lse, need = _fwd(*dev, max(q_lens), causal, window, bd, ws)
        _check(f"workspace={ws} ({need} bytes)", out, lse, ref, ref_lse, dtype)


@pytest.mark.parametrize("n,q,kv,Hq,Hkv,D,window,flash", [
    (32, 9, 100, 16, 2, 128, 0, False),      # 512 items of one head: the most
    (33, 9, 100, 16, 2, 128, 0, True),
    (130, 16, 70, 8, 4, 128, 50, True),
    (130, 16, 70, 8, 4, 64, 0, False),       # D = 64
    (180, 12, 60, 6, 2, 128, 0, False),      # odd group
    (70, 8, 60, 16, 2, 128, 0, False),       # two heads a group
])
def test_short_calls_of_many_rows(monkeypatch, n, q, kv, Hq, Hkv, D, window, flash):
    """The line between one workgroup per head group and the flash forward on
    short calls of up to 16 queries: the flash side is the flash forward,
    bitwise, the other is not; both against the oracle."""
    print(f"\n[case] {n} x {q} queries, {kv} keys, {Hq}/{Hkv} heads D={D} window={window}", flush=True)
    qs, k, v = _inputs([q] * n, [kv] * n, Hq, Hkv, D, torch.bfloat16, 9)
    cq, ck = cu_of([q] * n), cu_of([kv] * n)
    dev = [t.cuda() for t in (qs, k, v, cq, ck)]
    out, lse, _ = _fwd(*dev, q, True, window, None, True)
    ref, ref_lse = oracle.varlen_forward(qs, k, v, cq, ck, 1.0 / math.sqrt(D), True, window)
    _check("short", out, lse, ref, ref_lse, torch.bfloat16)
    monkeypatch.setenv("MTLATTN_NO_SPLITKV", "1")
    fout, flse, _ = _fwd(*dev, q, True, window, None, True)
    assert (torch.equal(out, fout) and torch.equal(lse, flse)) == flash


@pytest.mark.parametrize("q_lens,kv_lens,Hq,Hkv,D,dtype,max_q,window,bias", [
    ([1, 40, 0, 17], [200, 300, 9, 17], 8, 2, 128, torch.bfloat16, 1, 0, None),     # whole sequences
    ([5, 16, 33], [700, 16, 0], 8, 8, 64, torch.float16, 4, 0, None),               # (one without keys)
    ([3, 18], [400, 600], 8, 2, 128, torch.bfloat16, 2, 100, "head"),
    ([1] * 40 + [20], [50] * 41, 32, 8, 128, torch.float16, 3, 0, None),
    ([20], [1999], 8, 2, 128, torch.bfloat16, 1, 0, None),                          # chunks
    ([2, 17, 18], [5100, 0, 900], 4, 4, 64, torch.float16, 2, 0, "broadcast"),
])
def test_short_calls_with_too_small_max_seqlen_q(q_lens, kv_lens, Hq, Hkv, D, dtype, max_q, window, bias):
    """Below 2048 keys a sequence max_seqlen_q only routes: sequences with more
    queries than it says are attended in full."""
    print(f"\n[case] max_seqlen_q {max_q} for {q_lens[-4:]} D={D} {dtype} {kv_lens[-4:]}", flush=True)
    q, k, v = _inputs(q_lens, kv_lens, Hq, Hkv, D, dtype, 8)
    cq, ck = cu_of(q_lens), cu_of(kv_lens)
    b = None
    if bias:
        b = torch.randn(sum(q_lens), 1 if bias == "broadcast" else Hq, max(kv_lens),
                        generator=torch.Generator().manual_seed(4))
    ref, ref_lse = oracle.varlen_forward(q, k, v, cq, ck, 1.0 / math.sqrt(D), True, window, b)
    dev = [t.cuda() for t in (q, k, v, cq, ck)]
    for ws in (True, False):
        out, lse, need = _fwd(*dev, max_q, True, window, None if b is None else b.cuda(), ws)
        _check(f"workspace={ws} ({need} bytes)", out, lse, ref, ref_lse, dtype)


@pytest.mark.parametrize("q_lens,kv_lens,Hq,Hkv,D,dtype,causal,window", [
    ([512, 130], [4096, 9000], 8, 2, 128, torch.bfloat16, True, 0),
    ([32], [6000], 16, 2, 128, torch.float16, True, 0),
    ([17, 0, 65], [3000, 5, 5000], 8, 8, 64, torch.bfloat16, True, 0),
    ([100], [5001], 12, 12, 64, torch.float16, False, 0),
    ([257], [4100], 8, 2, 128, torch.bfloat16, True, 2100),
    ([70, 40], [4097, 3071], 8, 2, 80, torch.float16, True, 0),
    ([60], [5000], 8, 8, 96, torch.bfloat16, False, 0),
    ([90], [3500], 8, 2, 160, torch.bfloat16, True, 0),
    ([1, 65], [4000, 2999], 8, 2, 256, torch.float16, True, 0),
])
def test_forward_key_pieces(q_lens, kv_lens, Hq, Hkv, D, dtype, causal, window):
    """The flash forward on row tiles too few for the GPU cuts their keys into
    pieces (with the queried workspace) and merges them; without a workspace it
    runs unsplit. Row and key remainders, an empty sequence, keys below one
    piece, a window, every head dim's kernel; NaN in the workspace and trailing
    rows that no sequence owns stay out; equal on a second call, bitwise."""
    print(f"\n[case] forward key pieces D={D} {dtype} {q_lens} {kv_lens} window={window}", flush=True)
    q, k, v = _inputs(q_lens, kv_lens, Hq, Hkv, D, dtype, 5)
    cq, ck = cu_of(q_lens), cu_of(kv_lens)
    ref, ref_lse = oracle.varlen_forward(q, k, v, cq, ck, 1.0 / math.sqrt(D), causal, window)
    n = q.shape[0]
    dev = [torch.cat([q, q[:3]]).cuda(), torch.cat([k, k[:3]]).cuda(), torch.cat([v, v[:3]]).cuda(), cq.cuda(), ck.cuda()]
    runs = [_fwd(*dev, max(q_lens), causal, window, None, ws) for ws in (True, True, False)]
    assert runs[0][2] > 0, "expected a split workspace for this small grid"
    for out, lse, _ in runs:
        _check("pieces", out[:n], lse[:n], ref, ref_lse, dtype)
        assert out[n:].isnan().all() and lse[n:].isnan().all(), "rows outside every sequence were written"
    assert torch.equal(runs[0][0][:n], runs[1][0][:n]) and torch.equal(runs[0][1][:n], runs[1][1][:n])


@pytest.mark.parametrize("q_lens,kv_lens,Hq,Hkv,D,dtype,bad_key", [
    ([1, 3, 2], [300, 40, 700], 8, 2, 128, torch.bfloat16, 900),        # whole sequences (the last one's key)
    ([1, 2], [2100, 1999], 8, 2, 64, torch.float16, 600),               # chunks of one workgroup
    ([40, 17], [5000, 2100], 8, 2, 128, torch.bfloat16, 4975),          # key pieces, rows 15 and up
    ([70], [4000], 4, 4, 80, torch.float16, 10),
])
def test_split_forwards_keep_nan_and_infinity(q_lens, kv_lens, Hq, Hkv, D, dtype, bad_key):
    """A NaN or an infinite logit in one part of a row's keys makes the merged
    row NaN, as a softmax over all of them does, and no other row; a key of
    logit -inf drops out. Rows without a key stay 0, LSE -inf."""
    print(f"\n[case] NaN in split forwards {q_lens} {kv_lens} D={D} {dtype}", flush=True)
    q, k, v = _inputs(q_lens, kv_lens, Hq, Hkv, D, dtype, 12)
    q[0, 1, 5] = float("nan")                       # one row of one head
    k[bad_key, 0, 3] = float("nan")                 # the rows of kv head 0 that see it
    k[bad_key + 5, Hkv - 1, 7] = float("inf")       # logits +inf or -inf, by the sign of q
    cq, ck = cu_of(q_lens), cu_of(kv_lens)
    ref, ref_lse = oracle.varlen_forward(q, k, v, cq, ck, 1.0 / math.sqrt(D), True)
    want = ref.isnan().any(-1)
    assert want.any() and not want.all()
    dev = [t.cuda() for t in (q, k, v, cq, ck)]
    for ws in (True, False):
        if not ws and max(q_lens) <= 16 and sum(kv_lens) // len(kv_lens) >= 2048:
            continue
        out, lse, need = _fwd(*dev, max(q_lens), True, 0, None, ws)
        assert torch.equal(out.isnan().any(-1), want) and torch.equal(out.isnan().all(-1), want), f"workspace={ws}"
        assert lse[ref_lse.isnan()].isnan().all()
        assert (out.float() - ref)[~want].abs().max().item() < REF_ATOL[dtype]
        assert (lse - ref_lse)[~want].abs().max().item() < LSE_TOL[dtype]


@pytest.mark.parametrize("last", [33, 64])
def test_forward_key_pieces_at_the_most_tiles(last):
    """256 row tiles are the most that a split launch numbers; with one more
    the forward runs unsplit."""
    print(f"\n[case] forward key pieces, {255 + last // 33} tiles", flush=True)
    q_lens, kv_lens = [64] * 127 + [last], [1500 + 13 * i for i in range(128)]
    q, k, v = _inputs(q_lens, kv_lens, 2, 1, 64, torch.bfloat16, 13)
    cq, ck = cu_of(q_lens), cu_of(kv_lens)
    ref, ref_lse = oracle.varlen_forward(q, k, v, cq, ck, 0.125, True)
    out, lse, need = _fwd(*[t.cuda() for t in (q, k, v, cq, ck)], 64, True, 0, None, True)
    assert (need > 0) == (last == 33)
    _check("tiles", out, lse, ref, ref_lse, torch.bfloat16)


def _bwd(q, k, v, do, out, lse, cq, ck, max_q, causal, nbytes, skew=0):
    """(dq, dk, dv) of mtlattn_varlen_bwd on NaN-filled outputs with a
    NaN-filled workspace of nbytes that starts `skew` bytes past an aligned
    address, and the queried size."""
    Hq, D, Hkv = q.shape[1], q.shape[2], k.shape[1]
    p = capi.problem_for(q, k, cq, ck, max_q, 1.0 / math.sqrt(D), causal=causal)
    need = capi.lib().mtlattn_varlen_bwd_workspace_size(ctypes.byref(p))
    nbytes = need if nbytes is None else nbytes
    ws = torch.full((nbytes // 4 + 4,), float("nan"), dtype=torch.float32, device="cuda")
    g = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    capi.call("mtlattn_varlen_bwd", p, q.data_ptr(), Hq * D, k.data_ptr(), Hkv * D, v.data_ptr(), Hkv * D,
              out.data_ptr(), Hq * D, do.data_ptr(), Hq * D, lse.data_ptr(), g[0].data_ptr(), g[1].data_ptr(),
              g[2].data_ptr(), ws.data_ptr() + skew, nbytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return [t.cpu() for t in g], need


@pytest.mark.parametrize("last", [256, 384])
def test_dkv_pieces_at_the_most_tiles(last):
    """As above for dK/dV: 256 key blocks in pieces, 257 unsplit."""
    print(f"\n[case] dK/dV pieces, {255 + last // 256 + last // 384} tiles", flush=True)
    q_lens, kv_lens = [600 - i for i in range(127)], [128] * 126 + [last]
    q, k, v = _inputs(q_lens, kv_lens, 4, 1, 64, torch.bfloat16, 14)
    do = randn(q.shape, torch.bfloat16, torch.Generator().manual_seed(15))
    cq, ck = cu_of(q_lens), cu_of(kv_lens)
    dev = [t.cuda() for t in (q, k, v, do, cq, ck)]
    qd, kd, vd, dod, cqd, ckd = dev
    out, lse, _ = _fwd(qd, kd, vd, cqd, ckd, 600, False, 0, None, True)
    grads, need = _bwd(qd, kd, vd, dod, out.cuda(), lse.cuda(), cqd, ckd, 600, False, None)
    assert (need > lse.numel() * 4) == (last == 256)
    _, _, *refs = oracle.varlen_forward_backward(q, k, v, do, cq, ck, 0.125, False)
    for nm, a, r in zip(("dq", "dk", "dv"), grads, refs):
        assert torch.isfinite(a.float()).all(), nm
        assert ((a.float() - r).norm() / r.norm()).item() < 8e-3, nm     # P, dS and the output in bf16, 2^-9 each


@pytest.mark.parametrize("lens,Hq,Hkv,D,dtype", [
    ([700, 90], 8, 2, 128, torch.bfloat16),
    ([1000], 8, 2, 64, torch.float16),
    ([500], 4, 2, 256, torch.bfloat16),
])
def test_split_dkv_keeps_nan_and_takes_any_workspace(lens, Hq, Hkv, D, dtype):
    """dK/dV in pieces (the queried workspace) against the unsplit kernel (a
    workspace of delta only): NaN rows of dout reach the same gradients. A
    workspace that is not 16-byte aligned runs unsplit, bitwise, here and in the
    forward's key pieces."""
    print(f"\n[case] split dK/dV NaN {lens} {Hq}/{Hkv} D={D} {dtype}", flush=True)
    q, k, v = _inputs(lens, lens, Hq, Hkv, D, dtype, 16)
    do = randn(q.shape, dtype, torch.Generator().manual_seed(17))
    cq, ck = cu_of(lens), cu_of(lens)
    qd, kd, vd, cqd, ckd = (t.cuda() for t in (q, k, v, cq, ck))
    out, lse, _ = _fwd(qd, kd, vd, cqd, ckd, max(lens), True, 0, None, True)
    args = (out.cuda(), lse.cuda(), cqd, ckd, max(lens), True)
    delta = lse.numel() * 4
    for bad in (False, True):
        if bad:
            do[300, 1] = float("nan")               # (its query head's kv head, the keys it sees)
        split, need = _bwd(qd, kd, vd, do.cuda(), *args, None)
        whole, _ = _bwd(qd, kd, vd, do.cuda(), *args, delta)
        skewed, _ = _bwd(qd, kd, vd, do.cuda(), *args, need, skew=4)
        assert need > delta
        for nm, a, b, c in zip(("dq", "dk", "dv"), split, whole, skewed):
            assert torch.equal(b.isnan(), c.isnan()) and torch.equal(b.nan_to_num(), c.nan_to_num()), nm
            assert torch.equal(a.isnan(), b.isnan()) and a.isnan().any().item() == bad, nm
            err = (a.float() - b.float()).nan_to_num().norm() / b.float().nan_to_num().norm()
            assert err.item() < 8e-3, nm


def test_forward_key_pieces_need_an_aligned_workspace():
    print("\n[case] forward key pieces, workspace alignment", flush=True)
    q, k, v = _inputs([40], [5000], 8, 2, 128, torch.bfloat16, 18)
    q, k, v, cq, ck = (t.cuda() for t in (q, k, v, cu_of([40]), cu_of([5000])))
    ref, _, need = _fwd(q, k, v, cq, ck, 40, True, 0, None, False)
    assert need > 0
    p = capi.problem_for(q, k, cq, ck, 40, 1.0 / math.sqrt(128), causal=True)
    ws = torch.empty(need // 4 + 4, dtype=torch.float32, device="cuda")
    out = torch.full_like(q, float("nan"))
    capi.call("mtlattn_varlen_fwd", p, q.data_ptr(), 1024, k.data_ptr(), 256, v.data_ptr(), 256, out.data_ptr(), None,
              ws.data_ptr() + 4, need, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(out.cpu(), ref)


@pytest.mark.parametrize("stride", [(1 << 24) - 8, (1 << 24) + 8])
def test_row_strides_around_the_tile_limit(stride):
    """128-row tiles reach 32-bit byte offsets at row strides of 2^24 elements:
    below, the last row of a tile; at and above, the portable kernels. Against
    the same rows packed."""
    import mtlattn as mt
    print(f"\n[case] row stride {stride}", flush=True)
    n, H, D = 130, 2, 96                             # (head dims 80 to 96: 128-key tiles)
    g = torch.Generator().manual_seed(19)
    q, k, v = (randn((n, H, D), torch.bfloat16, g).cuda() for _ in range(3))
    cu = cu_of([n], "cuda")
    wide = torch.empty((n - 1) * stride + 2 * H * D, dtype=torch.bfloat16, device="cuda")
    ks, vs = (wide.as_strided((n, H, D), (stride, D, 1), i * H * D) for i in range(2))
    ks.copy_(k)
    vs.copy_(v)
    with torch.no_grad():
        for causal in (False, True):
            ref = mt.varlen_attention(q, k, v, cu, cu, n, causal=causal)
            out = mt.varlen_attention(q, ks, vs, cu, cu, n, causal=causal)
            assert (out.float() - ref.float()).abs().max().item() < REF_ATOL[torch.bfloat16]
