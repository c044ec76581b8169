"""Expert-indexed products over sorts of every size: round the pairs and experts
up to which the sort runs in LDS, the 64 experts it sums at a time, experts
without pairs, one expert with all of them, and pairs that name no expert.  The
weights are exact in bf16 (scale 1, bias -8), so that whichever kernel multiplies,
a result is off by float32 sums alone."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts", [1, 63, 65, 200, 1024, 1025])
@pytest.mark.parametrize("pairs", [2, 17, 64, 65, 1023, 1025, 4096, 4097])
@pytest.mark.parametrize("skew", [False, True])
def test_sort(pairs, experts, skew):
    n, k = 24, 1088
    g = torch.Generator(device="cuda").manual_seed(pairs + experts)
    w = torch.randint(-2**31, 2**31 - 1, (experts, n, k // 8), dtype=torch.int32, device="cuda", generator=g)
    s = torch.ones((experts, n, k // 64), device="cuda").bfloat16()
    x = torch.randn((pairs, k), device="cuda", generator=g).bfloat16()
    rhs = torch.randint(-1, experts + 1, (pairs,), device="cuda", generator=g, dtype=torch.int32)
    if skew:
        rhs = torch.where(torch.rand((pairs,), device="cuda", generator=g) < 0.9, experts - 1, rhs).int()
    lhs = torch.randperm(pairs, device="cuda", generator=g).int()
    y = K.gather_qmm(x, w, s, -8 * s, lhs, rhs, out_dtype=torch.float32)
    ok = (rhs >= 0) & (rhs < experts)
    full = K.dequantize(w, s, -8 * s, out_dtype=torch.float32)
    rows, ids = x[lhs.long()].float(), rhs.long()
    want = torch.zeros((pairs, n), device="cuda", dtype=torch.float64)
    for e in ids[ok].unique().tolist():
        at = ok & (ids == e)
        want[at] = rows[at].double() @ full[e].double().T
    if bool(ok.any()):
        assert ((y[ok].double() - want[ok]).norm() / want[ok].norm()).item() <= 2e-5
