"""The packed backward (pbgdn_chunk_bwd_packed) against the batched backward of
each sequence alone: the same kernels on the same rows, so bit for bit, in
every head width and dtype; rows that belong to no sequence get zeros, an empty
sequence's dh0 is its final gradient, and a call split into groups of sequences
(its workspace bounded) returns what one call returns."""
import pytest
import torch

from pseudobrain_amd import gated_deltanet as gd
from pseudobrain_amd.workloads import generate

pytestmark = pytest.mark.gpu
DEV = "cuda"


def make(bounds, total, hk, hv, dk, dv, dtype, seed):
    nseq = len(bounds) - 1
    q, k, v, g, beta, h0 = (x.to(DEV) for x in generate(1, total, hk, hv, dk, dv, dtype, 0.05, seed=seed, nstates=nseq))
    gen = torch.Generator().manual_seed(seed)
    do = (torch.randn(1, total, hv, dv, generator=gen) * 0.1).to(dtype).to(DEV)
    dht = (torch.randn(nseq, hv, dk, dv, generator=gen) * 0.1).to(DEV)
    return q, k, v, g, beta, h0, do, dht, torch.tensor(bounds, dtype=torch.int32, device=DEV)


def packed(q, k, v, g, beta, h0, do, dht, cu, scale=0.1):
    return torch.ops.pbgdn.gated_delta_chunk_packed_backward(q, k, v, g, beta, h0, cu, do, dht, scale)


@pytest.mark.parametrize("bounds,total,hk,hv,dk,dv,dtype", [
    ([0, 1, 1, 64, 129, 300], 300, 1, 2, 128, 128, torch.bfloat16),     # 1-token, empty, 63-, 65- and 171-token
    ([3, 70, 198], 211, 2, 2, 64, 128, torch.bfloat16),                 # rows before and after every sequence
    ([0, 64, 128, 192], 192, 1, 3, 128, 64, torch.bfloat16),            # whole chunks
    (list(range(0, 71 * 9, 9)), 70 * 9, 1, 1, 64, 64, torch.bfloat16),  # 70 sequences: past one wave's count
    ([0, 100, 100, 250], 260, 2, 4, 64, 64, torch.float16),
    ([5, 40, 170], 171, 1, 2, 128, 128, torch.float32),
])
def test_packed_equals_each_sequence_alone(bounds, total, hk, hv, dk, dv, dtype):
    print(f"[{bounds[:6]} {hk}->{hv} K={dk} V={dv} {dtype}]", flush=True)
    q, k, v, g, beta, h0, do, dht, cu = make(bounds, total, hk, hv, dk, dv, dtype, seed=len(bounds))
    got = packed(q, k, v, g, beta, h0, do, dht, cu)
    for n, (lo, hi) in enumerate(zip(bounds, bounds[1:])):
        sl = slice(lo, hi)
        if hi == lo:
            assert torch.equal(got[5][n], dht[n])
            continue
        ref = gd.chunk_bwd(*(x[:, sl] for x in (q, k, v, g, beta)), 0.1, h0[n:n + 1], do[:, sl], dht[n:n + 1])
        for name, a, b in zip(("dq", "dk", "dv", "dg", "dbeta"), got, ref):
            assert torch.equal(a[:, sl], b), f"{name} of sequence {n}"
        assert torch.equal(got[5][n], ref[5][0]), f"dh0 of sequence {n}"
    for a in got[:5]:
        assert not a[:, :bounds[0]].any() and not a[:, bounds[-1]:].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("total", [70, 0])
def test_no_sequence(dtype, total):
    """cu_seqlens of one bound: every row gets zeros, and there is no dh0."""
    q, k, v, g, beta, h0, do, dht, cu = make([0], total, 1, 2, 64, 64, dtype, seed=8)
    leaves = [x.requires_grad_() for x in (q, k, v, g, beta)]
    o, final = gd.gated_delta_rule(*leaves, 0.1, h0, "hip", cu)
    grads = torch.autograd.grad([o, final], leaves, [do.to(o.dtype), dht])
    torch.cuda.synchronize()
    for x, grad in zip(leaves, grads):
        assert grad.shape == x.shape and not grad.any()
    assert packed(*(x.detach() for x in leaves), h0, do, dht, cu)[5].shape == (0, 2, 64, 64)


def test_groups_of_sequences_equal_one_call(monkeypatch):
    bounds = [2, 90, 90, 300, 301, 420]
    args = make(bounds, 450, 1, 2, 64, 64, torch.bfloat16, seed=4)
    q, k, v, g, beta, h0, do, dht, cu = args
    want = packed(*args)
    monkeypatch.setattr(gd, "PACKED_BWD_WORKSPACE", 1 << 20)
    got = gd._packed_backward(q, k, v, g, beta, h0, cu, do, dht, 0.1)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("bounds", [[1000, 1090, 1090, 1300, 1301, 1420], [0, 200], [3900, 4000], [77], [0, 40, 90]])
def test_groups_hold_no_rows_of_no_sequence(monkeypatch, bounds):
    """Each group's workspace stays within the limit however long the buffer is
    around the sequences, and the result is one call's."""
    limit = 1 << 20  # (about 280 rows of these heads)
    args = make(bounds, 4000, 1, 2, 64, 64, torch.bfloat16, seed=5)
    q, k, v, g, beta, h0, do, dht, cu = args
    want = packed(*args)
    sizes, empty = [], torch.empty

    def recorded(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            sizes.append(size[0])
        return empty(*size, **kw)

    monkeypatch.setattr(gd, "PACKED_BWD_WORKSPACE", limit)
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", recorded)
        got = gd._packed_backward(q, k, v, g, beta, h0, cu, do, dht, 0.1)
    torch.cuda.synchronize()
    assert all(size <= limit for size in sizes) and (len(bounds) == 1 or sizes)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a, b)


def test_out_of_memory_leaves_each_sequence_alone(monkeypatch):
    """A call whose workspace for all sequences cannot be had still runs if the
    longest sequence's can."""
    bounds = [0, 90, 90, 300, 301, 420]
    args = make(bounds, 450, 1, 2, 64, 64, torch.bfloat16, seed=9)
    q, k, v, g, beta, h0, do, dht, cu = args
    want = packed(*args)
    refused, empty = [], torch.empty

    def small_only(*size, **kw):
        if kw.get("dtype") == torch.uint8 and size[0] > 1 << 20:
            refused.append(size[0])
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    with monkeypatch.context() as m:
        m.setattr(torch, "empty", small_only)
        got = packed(*args)
    torch.cuda.synchronize()
    assert len(refused) == 1
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dk,dv", [(128, 128), (64, 64), (128, 64)])
def test_many_heads_equal_few(dk, dv):
    """Scans of 64 value columns a workgroup (enough sequences and heads for
    the device) against those of 32 (one sequence alone): the same sums, so bit
    for bit, with chunks of one token and of 63."""
    batch, heads = 8, 32
    for length in (63, 129):
        q, k, v, g, beta, h0 = (x.to(DEV) for x in generate(batch, length, heads, heads, dk, dv, torch.bfloat16, 0.05,
                                                            seed=length))
        gen = torch.Generator().manual_seed(length)
        do = (torch.randn(batch, length, heads, dv, generator=gen) * 0.1).to(torch.bfloat16).to(DEV)
        dht = (torch.randn(batch, heads, dk, dv, generator=gen) * 0.1).to(DEV)
        got = gd.chunk_bwd(q, k, v, g, beta, 0.1, h0, do, dht)
        for n in (0, batch - 1):
            one = slice(n, n + 1)
            ref = gd.chunk_bwd(*(x[one, :, :2] for x in (q, k, v, g, beta)), 0.1, h0[one, :2], do[one, :, :2],
                               dht[one, :2])
            for name, a, b in zip(("dq", "dk", "dv", "dg", "dbeta"), got, ref):
                assert torch.equal(a[one, :, :2], b), f"{name} of row {n}, length {length}"
            assert torch.equal(got[5][one, :2], ref[5])


@pytest.mark.parametrize("hk,hv", [(2, 2), (1, 2)])
def test_outputs_of_any_alignment(monkeypatch, hk, hv):
    """dq, dk and dv at addresses that are no multiple of 8 bytes: the same values."""
    q, k, v, g, beta, h0 = (x.to(DEV) for x in generate(1, 100, hk, hv, 128, 128, torch.bfloat16, 0.05, seed=6))
    gen = torch.Generator().manual_seed(6)
    do = (torch.randn(1, 100, hv, 128, generator=gen) * 0.1).to(torch.bfloat16).to(DEV)
    want = gd.chunk_bwd(q, k, v, g, beta, 0.1, h0, do)

    def one_element_off(x, **kw):
        return torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)

    with monkeypatch.context() as m:
        m.setattr(torch, "empty_like", one_element_off)
        got = gd.chunk_bwd(q, k, v, g, beta, 0.1, h0, do)
    torch.cuda.synchronize()
    assert got[0].data_ptr() % 8 == 2
    for a, b in zip(got, want):
        assert torch.equal(a, b)
