"""The bf16 gradient kernel's own paths, against the float64 oracle and against
the same kernels on one key head or one sequence alone."""
import numpy as np
import pytest
import torch

from oracle import gdn
from pseudobrain_amd import _lib
from pseudobrain_amd import gated_deltanet as gd
from pseudobrain_amd.workloads import cu_seqlens_of, generate, to_numpy
from tests.test_gpu_backward import check, oracle_grads

pytestmark = pytest.mark.gpu
DEV = "cuda"


def make(batch, length, hk, hv, dk, dv, seed, dtype=torch.bfloat16, nseq=None):
    q, k, v, g, beta, h0 = generate(batch, length, hk, hv, dk, dv, dtype, 0.05, seed=seed, nstates=nseq)
    gen = torch.Generator().manual_seed(seed + 1)
    do = (torch.randn(batch, length, hv, dv, generator=gen) * 0.1).to(dtype)
    dht = torch.randn(nseq or batch, hv, dk, dv, generator=gen) * 0.1
    return q, k, v, g, beta, h0, do, dht


def sums_in_registers(batch, length, nseq, hk, hv, dk, dv):
    """The gradient kernel takes whole groups of value heads: the call's workspace
    has no float32 dq and dk per value head."""
    records = batch * -(-length // 64) if nseq is None else length // 64 + nseq + 1
    floats = records * hv * (2 * 64 * 64 + 2 * 64 + 2 * dk * dv)
    return _lib.lib().pbgdn_chunk_bwd_workspace_size_dtype(
        _lib.BF16, batch, length, -1 if nseq is None else nseq, hk, hv, dk, dv) == 4 * floats + 256


def one_element_off(x, **kw):
    return torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("batch,length,hk,hv,dk,dv", [
    (8, 200, 16, 32, 128, 128),  # two items a workgroup, the last chunk of 8 tokens
    (8, 200, 8, 32, 128, 64),    # four value heads an item
    (16, 193, 8, 32, 64, 128),   # a chunk of one token
    (8, 200, 16, 32, 64, 64),
])
def test_value_heads_summed_in_registers(monkeypatch, batch, length, hk, hv, dk, dv, aligned):
    """Key heads' gradients where one workgroup takes a key head's value heads in
    turn and sums dq and dk over them: some key heads against the oracle, and
    against a call of that key head alone, whose items are one value head each
    (everything but that sum the same bits; dq and dk within their rounding)."""
    with monkeypatch.context() as m:
        if not aligned:
            m.setattr(torch, "empty_like", one_element_off)
        check_value_heads_summed_in_registers(batch, length, hk, hv, dk, dv)


def check_value_heads_summed_in_registers(batch, length, hk, hv, dk, dv):
    assert sums_in_registers(batch, length, None, hk, hv, dk, dv)
    args = make(batch, length, hk, hv, dk, dv, seed=hk + dv)
    q, k, v, g, beta, h0, do, dht = (x.to(DEV) for x in args)
    scale, group = dk ** -0.5, hv // hk
    got = gd.chunk_bwd(q, k, v, g, beta, scale, h0, do, dht)
    torch.cuda.synchronize()
    for n, kh in ((0, 0), (batch // 2, hk // 2), (batch - 1, hk - 1)):
        print(f"[row {n}, key head {kh}]", flush=True)
        one, keys, heads = slice(n, n + 1), slice(kh, kh + 1), slice(kh * group, (kh + 1) * group)
        part = lambda x, hd: x[one, :, hd].contiguous()  # noqa: E731
        sub = [part(q, keys), part(k, keys), part(v, heads), part(g, heads), part(beta, heads)]
        mine = [part(x, hd) for x, hd in zip(got, (keys, keys, heads, heads, heads))] + [got[5][one, heads]]
        alone = gd.chunk_bwd(*sub, scale, h0[one, heads], part(do, heads), dht[one, heads])
        assert not sums_in_registers(1, length, None, 1, group, dk, dv)
        for name, a, b in zip(("dv", "dg", "dbeta", "dh0"), mine[2:], alone[2:]):
            assert torch.equal(a, b), f"{name} of row {n}, key head {kh}"
        for name, a, b in zip(("dq", "dk"), mine, alone):  # two bf16 roundings of sums that differ in their last bits
            diff = (a.double() - b.double()).abs()
            assert (diff <= 2 ** -7 * b.double().abs() + 1e-6).all(), f"{name} of row {n}, key head {kh}"
        ref = oracle_grads(*(x.cpu() for x in sub), scale, h0[one, heads].cpu(), part(do, heads).cpu(),
                           dht[one, heads].cpu())
        check(f"row {n} key head {kh}", mine, ref, dict(dq=q.dtype, dk=q.dtype, dv=q.dtype, dg=torch.float32,
                                                        dbeta=torch.float32, dh0=torch.float32))


def test_value_heads_summed_in_registers_packed():
    """The same of packed sequences: each against a batched call of it alone."""
    lengths = [200, 64, 0, 1, 321, 450, 65, 499]
    nseq, total, hk, hv, dk, dv = len(lengths), sum(lengths), 16, 32, 128, 128
    assert sums_in_registers(1, total, nseq, hk, hv, dk, dv)
    q, k, v, g, beta, h0, do, dht = (x.to(DEV) for x in make(1, total, hk, hv, dk, dv, seed=3, nseq=nseq))
    cu = cu_seqlens_of(lengths).to(DEV)
    got = torch.ops.pbgdn.gated_delta_chunk_packed_backward(q, k, v, g, beta, h0, cu, do, dht, 0.1)
    torch.cuda.synchronize()
    for n, (lo, hi) in enumerate(zip(cu.tolist(), cu.tolist()[1:])):
        if lo == hi:
            assert torch.equal(got[5][n], dht[n])
            continue
        sl = slice(lo, hi)
        alone = gd.chunk_bwd(*(x[:, sl] for x in (q, k, v, g, beta)), 0.1, h0[n:n + 1], do[:, sl], dht[n:n + 1])
        for name, a, b in zip(("dv", "dg", "dbeta"), got[2:], alone[2:]):
            assert torch.equal(a[:, sl], b), f"{name} of sequence {n}"
        assert torch.equal(got[5][n], alone[5][0]), f"dh0 of sequence {n}"
        for name, a, b in zip(("dq", "dk"), got, alone):
            diff = (a[:, sl].double() - b.double()).abs()
            assert (diff <= 2 ** -7 * b.double().abs() + 1e-6).all(), f"{name} of sequence {n}"


@pytest.mark.parametrize("batch,length,nseq,hk,hv,dk,dv,dtype", [
    (8, 200, None, 16, 32, 128, 128, torch.bfloat16),  # dq and dk summed in registers
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
