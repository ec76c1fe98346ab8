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
