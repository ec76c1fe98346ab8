"""The bf16 gradient kernel's own paths, against the float64 oracle and against
the same kernels on one key head or one sequence alone."""
import numpy as np
import pytest
import torch

from oracle import gdn
from pseudobrain_amd import gated_deltanet as gd
from pseudobrain_amd.workloads import cu_seqlens_of, generate, to_numpy

pytestmark = pytest.mark.gpu
DEV = "cuda"


def make(batch, length, hk, hv, dk, dv, seed, dtype=torch.bfloat16, nseq=None):
    q, k, v, g, beta, h0 = generate(batch, length, hk, hv, dk, dv, dtype, 0.05, seed=seed, nstates=nseq)
    gen = torch.Generator().manual_seed(seed + 1)
    do = (torch.randn(batch, length, hv, dv, generator=gen) * 0.1).to(dtype)
    dht = torch.randn(nseq or batch, hv, dk, dv, generator=gen) * 0.1
    return q, k, v, g, beta, h0, do, dht


@pytest.mark.parametrize("batch,length,nseq,hk,hv,dk,dv,dtype", [
    (8, 200, None, 16, 32, 128, 128, torch.bfloat16),
    (1, 130, None, 2, 4, 128, 64, torch.bfloat16),     # per value head in the workspace
    (1, 300, 3, 2, 2, 64, 128, torch.bfloat16),
    (1, 300, 3, 1, 2, 64, 64, torch.float16),
    (2, 65, None, 1, 2, 128, 128, torch.float32),
])
def test_the_workspace_is_not_overrun(monkeypatch, batch, length, nseq, hk, hv, dk, dv, dtype):
    """A call with the bytes its dtype needs writes nothing behind them."""
    q, k, v, g, beta, h0, do, dht = (x.to(DEV) for x in make(batch, length, hk, hv, dk, dv, 5, dtype, nseq))
    cu = None if nseq is None else cu_seqlens_of([100, 0, 200]).to(DEV)
    guards, empty = [], torch.empty

    def guarded(*size, **kw):
        if kw.get("dtype") != torch.uint8:
            return empty(*size, **kw)
        x = empty(size[0] + 4096, **kw)
        x[size[0]:] = 0xA5
        guards.append(x[size[0]:])
        return x[:size[0]]

    with monkeypatch.context() as m:
        m.setattr(torch, "empty", guarded)
        gd._chunk_bwd(q, k, v, g, beta, 0.1, h0, cu, do, dht)
    torch.cuda.synchronize()
    assert len(guards) == 1 and bool((guards[0] == 0xA5).all())


def test_decay_sums_are_in_float32():
    """dg where the state's decay terms make it up (chunks of 4 tokens, states and
    final gradients of bf16 values, so that their pairs are exact). U and dX carry
    the rounding of one bf16 pair each (2^-18 of an element at most, from beta X
    and dU); a sum over the columns that takes them as pairs again rounds both
    once more and drops the low by low products: three roundings of that size in
    quadrature for one. The 2-norm error over three seeds measures 2.4e-6 with
    float32 sums and 3.3e-6 with pairs."""
    errs = []
    for seed in (1, 2, 3):
        print(f"[decay sums, seed {seed}]", flush=True)
        q, k, v, g, beta, h0 = generate(32, 4, 4, 8, 128, 128, torch.bfloat16, 0.05, seed=seed)
        gen = torch.Generator().manual_seed(seed)
        do = (torch.randn(32, 4, 8, 128, generator=gen) * 0.1).to(torch.bfloat16)
        dht = (torch.randn(32, 8, 128, 128, generator=gen) * 0.1).to(torch.bfloat16).float()
        h0 = (torch.randn(h0.shape, generator=gen) * 0.05).to(torch.bfloat16).float()
        got = gd.chunk_bwd(*(x.to(DEV) for x in (q, k, v, g, beta)), 128 ** -0.5, h0.to(DEV), do.to(DEV), dht.to(DEV))
        ref = gdn.gated_delta_rule_backward(*(to_numpy(x.double()) for x in (q, k, v, g, beta)), 128 ** -0.5,
                                            to_numpy(h0.double()), to_numpy(do.double()), to_numpy(dht.double()))[3]
        errs.append(np.linalg.norm(to_numpy(got[3].double()) - ref) / np.linalg.norm(ref))
    print(errs, flush=True)
    assert np.mean(errs) < 2.8e-6
