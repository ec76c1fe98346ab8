"""float32 o of 16-bit inputs, written by the scan kernels themselves: rounded
to the input dtype it is the 16-bit o bit for bit (the same sums, stored before
and after the one rounding), on every scan the device gate routes to: the wide
scan (many sequences at K = 128), the narrow one (few; K = 64; V no multiple of
128) and the 256-wide one, with ragged ends and packed sequences."""
import pytest
import torch

from pseudobrain_amd import gated_deltanet as gd
from pseudobrain_amd.workloads import cu_seqlens_of, generate

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,lengths,hk,hv,dk,dv", [
    (4, [130], 16, 32, 128, 128),         # wide: 128 workgroups, a chunk of 2 tokens
    (1, [1, 64, 0, 77, 191], 16, 32, 128, 128),  # wide, packed, an empty sequence
    (2, [65], 32, 32, 128, 256),          # wide, two column groups a head
    (1, [300], 2, 4, 128, 128),           # narrow
    (2, [63], 2, 2, 64, 48),              # narrow, K = 64
    (1, [100], 1, 2, 256, 64),            # 256-wide keys
])
def test_float32_o_rounds_to_the_16_bit_o(dtype, batch, lengths, hk, hv, dk, dv):
    packed = len(lengths) > 1
    q, k, v, g, beta, h0 = generate(batch, sum(lengths), hk, hv, dk, dv, dtype, 0.05, seed=dk + len(lengths),
                                    nstates=len(lengths) if packed else None)
    cu = cu_seqlens_of(lengths).to(DEV) if packed else None
    args = [x.to(DEV) for x in (q, k, v, g, beta)] + [dk ** -0.5, h0.to(DEV), cu]
    o16, s16 = gd.chunk_fwd(*args)
    o32, s32 = gd.chunk_fwd(*args, out_dtype=torch.float32)
    entry, final = gd.gated_delta_rule(*args[:-1], "hip", cu)
    torch.cuda.synchronize()
    assert o32.dtype == torch.float32 and o16.dtype == dtype
    assert torch.equal(o32.to(dtype), o16) and torch.equal(s32, s16)
    assert torch.equal(entry, o32) and torch.equal(final, s32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dk,dv,grad", [(128, 100, False), (64, 33, False), (256, 40, False), (96, 120, False),
                                        (128, 100, True), (64, 33, True)])
def test_padded_value_widths_cut_a_16_bit_o(dtype, dk, dv, grad):
    """V no width of the kernels: o is the 16-bit o's columns, widened, contiguous."""
    q, k, v, g, beta, h0 = (x.to(DEV) for x in generate(2, 130, 2, 4, dk, dv, dtype, 0.05, seed=dv))
    with torch.set_grad_enabled(grad):
        if grad:
            q.requires_grad_()
        o, final = gd.gated_delta_rule(q, k, v, g, beta, 0.1, h0, "hip")
        kp, vp = gd._chunk_widths(dk, dv, grad)
    with torch.no_grad():
        o16, s16 = gd.chunk_fwd(gd._pad_last(q, kp), gd._pad_last(k, kp), gd._pad_last(v, vp), g, beta, 0.1,
                                gd._pad_state(h0, kp, vp))
    assert vp > dv and o.dtype == torch.float32 and o.is_contiguous() and o.requires_grad == grad
    assert torch.equal(o, o16[..., :dv].float()) and torch.equal(final, s16[..., :dk, :dv])
