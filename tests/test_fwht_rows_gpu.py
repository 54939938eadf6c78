"""The input transform's two forms (two or eight elements per lane, chosen by the number of 128-blocks) and the fused
int8 quantizers on operands at the element types' own alignment, against the oracle: the sizes around the choice, odd row
counts, a last wave that is not full, and a gate_up row stride that leaves every row misaligned."""
import numpy as np
import pytest

import oracle_lib as O
from r4dx_amd import workloads as WL

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from r4dx_amd import api  # noqa: E402
from gpu_util import banner, dev, host_u16  # noqa: E402


# 4095 | 4096 | 4097 blocks meet the two forms' boundary; 3 outputs and 1
@pytest.mark.parametrize("M,K,nout", [(1, 128, 1), (13, 40320, 1), (32, 16384, 3), (241, 2176, 2), (37, 5120, 3), (5, 6144, 2)])
@pytest.mark.parametrize("shift", [0, 1])
def test_transform_forms(M, K, nout, shift):
    banner("input transform", M, K, nout, shift)
    x = WL.activations_f16(M, K, M + K, outlier_frac=0.01)
    suh = [WL.signs(K, 7 + o) for o in range(nout)]
    xd = torch.empty(M * K + shift, dtype=torch.int16, device="cuda")[shift:]
    xd.copy_(dev(x.view(np.uint16)).view(-1))
    sd = []
    for s in suh:
        t = torch.empty(K + shift, dtype=torch.float32, device="cuda")[shift:]
        t.copy_(dev(s))
        sd.append(t)
    outs = [torch.empty(M * K + shift, dtype=torch.float16, device="cuda")[shift:].view(M, K) for _ in range(nout)]
    api.trellis_input(xd.view(M, K), sd, -3, bf16=False, outs=outs)
    torch.cuda.synchronize()
    for s, o in zip(suh, outs):
        assert np.array_equal(host_u16(o), O.transform_input(x.view(np.uint16), False, s, -3))


@pytest.mark.parametrize("rows,inter,extra", [(3, 1280, 1), (256, 2176, 3)])
def test_silu_misaligned_rows(rows, inter, extra):
    banner("silu + transform, row stride", 2 * inter + extra)
    g = torch.Generator(device="cuda").manual_seed(rows)
    wide = (torch.randn(rows, 2 * inter + extra, device="cuda", generator=g) * 3).bfloat16()
    suh = dev(WL.signs(inter, 3))
    packed = wide[:, :2 * inter].contiguous()
    for quant in (None, "blk", "row") if rows == 256 else (None,):
        got = api.silu_mul_trellis(wide, inter, suh, quant=quant)
        want = api.silu_mul_trellis(packed, inter, suh, quant=quant)
        torch.cuda.synchronize()
        for a, b in zip(got if quant else (got,), want if quant else (want,)):
            assert torch.equal(a, b)
    two = api.trellis_input(api.silu_mul(wide, inter), [suh])[0]
    assert torch.equal(api.silu_mul_trellis(wide, inter, suh).view(torch.int16), two.view(torch.int16))
