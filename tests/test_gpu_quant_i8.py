"""The int8 conversion of the Q / K quantisers on what random rows do not hold: exact ties, values at the bounds, NaN
and infinities. A NaN product (a NaN input, or an infinity times the reciprocal 0 of its group) gives -128; the amax
skips NaN."""
import pytest
import torch

from oracle import emu

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_quant_q_ties_bounds_nonfinite(dtype):
    from lingbot_world_v2_realtime_amd import kernels
    g = torch.Generator().manual_seed(3)
    q = torch.randn(1, 128, 4, 128, generator=g).to(dtype)
    # head 0, group 0: amax 127, so recip = 1 and k + 1/2 are ties; both bounds
    q[0, :32, 0] = torch.randint(-126, 126, (32, 128), generator=g).to(dtype) + 0.5
    q[0, 0, 0, 0], q[0, 1, 0, 1] = 127.0, -127.0
    q[0, 40, 0, 5] = float("nan")                                # group 1: a NaN among finite values
    q[0, 70, 0, 9], q[0, 71, 0, 3] = float("inf"), -float("inf")  # group 2
    q8, qs, _ = kernels.quant_q(q.to(DEV))
    torch.cuda.synchronize()
    clean = q.clone()
    clean[0, 40, 0, 5] = 0.0             # the amax skips a NaN
    want, scale = emu.quant_q(clean.nan_to_num(posinf=0.0, neginf=0.0))
    want[0, 40, 5] = -128
    want[0, 64:96] = 0                   # an infinite group: reciprocal 0
    want[0, 70, 9] = want[0, 71, 3] = -128
    scale[0, 2] = float("inf")
    assert torch.equal(q8.cpu(), want) and torch.equal(qs.cpu(), scale)
    tie = (q[0, 2:32, 0].float() * 2) % 2 == 1   # head 0, group 0: the quotient is the value itself
    assert bool(tie.all()) and bool((want[0, 2:32] % 2 == 0).all())
