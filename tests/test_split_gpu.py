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
