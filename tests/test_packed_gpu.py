"""The packed wrappers' gradients, written in place by the backward kernels
through row strides, against the separate-tensor entry on the same inputs."""

import pytest
import torch

from tests.helpers import cu_of, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,Hq,Hkv,D,dtype,causal,window", [
    ([37, 256, 1, 700], 8, 8, 128, torch.bfloat16, True, 0),       # split dK/dV
    ([5], 4, 2, 128, torch.float16, True, 0),
    ([1], 4, 4, 64, torch.bfloat16, False, 0),                     # one row
    ([130, 64, 0, 500], 8, 4, 64, torch.float16, False, 0),
    ([300, 90], 8, 8, 80, torch.bfloat16, True, 100),
    ([257], 4, 4, 160, torch.float16, True, 0),
    ([129, 70], 4, 2, 256, torch.bfloat16, True, 0),
    ([40, 33], 4, 4, 72, torch.bfloat16, True, 0),                 # portable kernels: stacked
    ([100, 29], 4, 2, 64, torch.float32, True, 0),                 # fp32 kernels: stacked
    ([2048] * 12, 16, 16, 64, torch.bfloat16, False, 0),           # unsplit dK/dV
    ([2048] * 8, 32, 8, 128, torch.float16, True, 0),
])
def test_packed_gradients_in_place(lens, Hq, Hkv, D, dtype, causal, window):
    """Bitwise the gradients of varlen_attention on the unbound tensors: the
    same kernels with other row strides. Two trailing rows belong to no
    sequence and get zeros."""
    import mtlattn as mt
    print(f"\n[case] packed gradients {lens[:4]} {Hq}/{Hkv} D={D} {dtype}", flush=True)
    g = torch.Generator().manual_seed(3)
    M = sum(lens) + 2
    cu = cu_of(lens, "cuda")
    q = randn((M, Hq, D), dtype, g).cuda()
    kv = randn((M, 2, Hkv, D), dtype, g).cuda()
    do = randn((M, Hq, D), dtype, g).cuda()
    do[-2:] = 0
    leaves = [t.detach().clone().requires_grad_() for t in (q, kv[:, 0], kv[:, 1])]
    ref = mt.varlen_attention(*leaves, cu, cu, max(lens), causal=causal, window=window)
    rq, rk, rv = torch.autograd.grad(ref, leaves, do)
    q1, kv1 = q.clone().requires_grad_(), kv.clone().requires_grad_()
    out = mt.flash_attn_varlen_kvpacked_func(q1, kv1, cu, cu, max(lens), max(lens), causal=causal, window=window)
    dq, dkv = torch.autograd.grad(out, (q1, kv1), do)
    n = sum(lens)
    assert torch.equal(out[:n], ref[:n]) and torch.equal(dq, rq)
    assert torch.equal(dkv, torch.stack((rk, rv), 1))
    assert not dq[n:].any() and not dkv[n:].any()
    if Hq == Hkv:
        qkv = torch.cat((q[:, None], kv), 1).requires_grad_()
        out = mt.flash_attn_varlen_qkvpacked_func(qkv, cu, max(lens), causal=causal, window=window)
        d, = torch.autograd.grad(out, qkv, do)
        assert torch.equal(out[:n], ref[:n]) and torch.equal(d, torch.stack((rq, rk, rv), 1))


def test_packed_gradient_memory():
    """Where the gradients are stacked (fp32), the backward holds no tensor for
    writing in place besides: the three gradients, the stack of them, workspace."""
    import mtlattn_amd as mt
    print("\n[case] packed fp32 gradient memory", flush=True)
    M, H, D = 20000, 8, 64
    qkv = torch.randn(M, 3, H, D, device="cuda", requires_grad=True)
    q, kv = (torch.randn(M, *s, H, D, device="cuda", requires_grad=True) for s in ((), (2,)))
    cu = torch.tensor([0, M // 2, M], dtype=torch.int32, device="cuda")
    for call, leaves in ((lambda: mt.flash_attn_varlen_qkvpacked_func(qkv, cu, M // 2), [qkv]),
                         (lambda: mt.flash_attn_varlen_kvpacked_func(q, kv, cu, cu, M // 2, M // 2), [q, kv])):
        out = call()
        do = torch.randn_like(out)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        grads = torch.autograd.grad(out, leaves, do)
        # in tensors of out's size; the half is for delta, a 64th (no split
        # partials at this size)
        stacked = 3 if len(leaves) == 1 else 2
        assert torch.cuda.max_memory_allocated() - before < (3 + stacked + 0.5) * out.numel() * 4
        del grads, out
