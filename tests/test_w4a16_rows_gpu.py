"""The w4a16 product's row forms (1, 2, 4 or 8 staged rows up to M = 8, one or two tiles of 32 above): each row of a batch
carries the bits the same form gives it alone in its place -- a form's rows past M are neither staged nor read, so what the
LDS held must not show -- with A staged in several chunks whose last is not whole, and A at two-byte alignment. Rows of up
to 8 also carry the single-row launch's bits (one MFMA form, one order of sums)."""
import numpy as np
import pytest

from r4dx_amd import workloads as WL

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from r4dx_amd import api  # noqa: E402
from gpu_util import banner, dev  # noqa: E402


@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 7, 8, 9, 31, 32, 33, 63, 64])
@pytest.mark.parametrize("K", [64, 11328])
def test_rows(group, M, K):
    banner("w4a16 rows", group, M, K)
    N = 272
    wq, wsz = WL.w4a16_packed(N, K, group, 3)
    wq, wsz = dev(wq), dev(wsz)
    a = dev(WL.activations_f16(64, K, 4).view(np.uint16))[:M].clone()
    poison = torch.full_like(a, 0x7E00)          # NaN rows through the same form: whatever they leave in LDS is NaN
    run = lambda x: api.w4a16_gemm(x, wq, wsz, K, N, group, f32=True)
    run(poison)
    got = run(a)
    odd = torch.empty(M * K + 1, dtype=torch.int16, device="cuda")[1:]
    odd.copy_(a.view(-1))
    again = run(odd.view(M, K))
    assert bool(torch.isfinite(got).all())
    assert torch.equal(got.view(torch.int32), again.view(torch.int32))
    for r in sorted({0, M // 2, M - 1}):
        one = torch.zeros_like(a)
        one[r] = a[r]
        alone = run(one)
        assert torch.equal(alone[r].view(torch.int32), got[r].view(torch.int32))
        if M <= 8:
            assert torch.equal(run(a[r:r + 1].contiguous())[0].view(torch.int32), got[r].view(torch.int32))
