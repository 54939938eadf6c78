"""The trellis int8 GEMM's tail split: with skg > 1 and more column groups than compute units, the groups beyond the last
whole round are cut along K. Sizes around its edges: one group over, a remainder of two pieces, a remainder too large to cut
(the K split as asked), K blocks fewer than and not divisible by the pieces, two input parts met inside the remainder.

Bars: the whole groups carry the bits of the skg = 1 launch; a cut group's sums differ from it by the order of at most 8 fp32
additions, so its bf16 results by at most one place (2^-7 of the value at a binade's edge) plus 2^-20 of the row's rms for
cancelled sums. The coarse form's pieces are whole numbers and carry the skg = 1 launch's bits in every group."""
import numpy as np
import pytest

from r4dx_amd import workloads as WL

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from r4dx_amd import api  # noqa: E402
from gpu_util import banner, dev  # noqa: E402


@pytest.mark.parametrize("coarse", [False, True])
@pytest.mark.parametrize("extra,K,KB,parts", [(1, 512, 4, False), (16, 2560, 5, True), (100, 1536, 4, True), (128, 512, 5, False),
                                              (200, 512, 4, False)])
def test_tail_split(extra, K, KB, parts, coarse):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    G = cus + extra
    N = 128 * G
    banner("int8 tail split", extra, K, KB, parts, coarse)
    g = torch.Generator(device="cuda").manual_seed(extra + K)
    w = torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)
    svh = dev(WL.svh_scales(N, 5))
    sw = api.trellis_i8_table(w, K, N, KB, coarse=coarse)
    a = [api.i8_quant(torch.randn(256, K, device="cuda", generator=g).half(), blk=not coarse) for _ in range(2)]
    two = dict(a8_1=a[1][0], sa_1=a[1][1], n_split=128 * (cus + extra // 2 + 1) if extra > 1 else 128) if parts else {}
    run = lambda skg: api.trellis_gemm_i8(a[0][0], a[0][1], w, sw, svh, K, N, KB, coarse=coarse, skg=skg, out_scale=0.1,
                                          ws=torch.full((max(1, skg) * 256 * N,), float("nan"), device="cuda"), **two)
    one, got, again = run(1), run(2), run(2)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), again.view(torch.int16))
    if extra <= 128:
        assert torch.equal(got[:, :128 * cus].view(torch.int16), one[:, :128 * cus].view(torch.int16))
    if coarse:
        assert torch.equal(got.view(torch.int16), one.view(torch.int16))
    x, y = got.double(), one.double()
    tol = y.abs() * 2.0**-7 + y.pow(2).mean(1, keepdim=True).sqrt() * 2.0**-20
    assert bool(((x - y).abs() <= tol).all())
    assert float((got.view(torch.int16) != one.view(torch.int16)).double().mean()) < 0.01
