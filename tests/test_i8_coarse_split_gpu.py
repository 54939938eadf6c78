"""The coarse trellis int8 GEMM's K sum under a grid split: exact int32 sums over the fewest slices that give 128 workgroups
(r4d_mi355x_i8_skg), whatever larger skg the launch is cut by -- no tolerance: the bits of that many slices, and of the
oracle's epilogue over the exact sum where it is one slice."""
import numpy as np
import pytest

import oracle_lib as O
from r4dx_amd import plan
from r4dx_amd import workloads as WL

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from r4dx_amd import api  # noqa: E402
from r4dx_amd.loader import lib  # noqa: E402
from gpu_util import banner, dev  # noqa: E402

OUT_SCALE = float(np.float32(0.1))


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def _run(a, w, sw, svh, K, N, KB, skg, n_split=None):
    two = dict(a8_1=a[1][0], sa_1=a[1][1], n_split=n_split) if n_split else {}
    ws = torch.full((max(1, skg) * 256 * N,), float("nan"), device="cuda")
    out = api.trellis_gemm_i8(a[0][0], a[0][1], w, sw, svh, K, N, KB, coarse=True, skg=skg, out_scale=OUT_SCALE, ws=ws, **two)
    torch.cuda.synchronize()
    return out


# (K, columns -- or, negative, column groups beyond the CUs -- KB, two parts): 1, 1, 2, 4, 4, 1 and 1 slices; the last two
# have a remainder to cut and one too large to cut
@pytest.mark.parametrize("K,N,KB,two", [(2560, 128 * 128, 4, True), (1536, 128 * 130, 5, False), (2048, 8192, 4, False),
                                        (4096, 2048, 5, True), (4096, 128 * 33, 4, False), (2560, -16, 4, True),
                                        (1024, -150, 5, False)])
def test_bits_do_not_depend_on_the_split(K, N, KB, two):
    if N < 0:
        N = 128 * (_cus() - N)
    banner("coarse int8 splits", K, N, KB, two)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    w = torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)
    svh = WL.svh_scales(N, 5)
    sw = api.trellis_i8_table(w, K, N, KB, coarse=True)
    x = [torch.randn(256, K, device="cuda", generator=g).half() for _ in range(2)]
    a = [api.i8_quant(v, blk=False) for v in x]
    n_split = 128 * (N // 256) if two else None
    base = lib().r4d_mi355x_i8_skg(K, N)
    assert plan.plan_trellis_i8(N, K, KB, coarse=True).SKG >= base
    want = _run(a, w, sw, dev(svh), K, N, KB, base, n_split).view(torch.int16)
    skgs = [s for s in (2, 4, 8) if s > base and (K // 128) % (2 * s) == 0]
    assert skgs
    for skg in skgs:
        same = torch.equal(_run(a, w, sw, dev(svh), K, N, KB, skg, n_split).view(torch.int16), want)
        assert same, skg
    if base > 1:
        return
    wp = api.trellis_i8_dump(w, sw, K, N, KB, True)[1]
    for grp in (0, N // 256, N // 128 - 1):
        c = slice(128 * grp, 128 * grp + 128)
        q, sa = api.i8_quant(x[1 if two and 128 * grp >= n_split else 0], blk=False, ref_layout=False)
        acc = q.view(256, K).double() @ wp[c].double().t()              # whole numbers below 2^53: exact
        raw = acc.float() * (sa[:, None] * sw[c][None, :])
        ref = O.epilogue_from_raw(raw.cpu().numpy(), svh[c], OUT_SCALE)
        assert np.array_equal(want[:, c].cpu().numpy().view(np.uint16), ref)


def test_long_k_keeps_the_slices_asked_for():
    """K 135168 with every product at its largest: a whole column's sum (135168 * 127^2) is past int32, that of each of the
    two slices asked for is not, so they are scaled one by one."""
    K, KB = 135168, 4
    N = 128 * (_cus() + 1)
    banner("coarse int8, long K", K, N)
    w = torch.zeros(K * N * KB // 32, dtype=torch.int32, device="cuda")       # every weight the same value: all 127 or -127
    sw = api.trellis_i8_table(w, K, N, KB, coarse=True)
    a = [api.i8_quant(torch.ones(256, K, device="cuda").half(), blk=False)]
    out = _run(a, w, sw, torch.ones(N, device="cuda"), K, N, KB, 2).float().view(256, N // 128, 128)
    q = api.trellis_reconstruct(torch.zeros(128 * 128 * KB // 32, dtype=torch.int32, device="cuda"), 128, 128, KB)
    y = 128.0 * K * q.view(torch.float16)[0, 0].item() * OUT_SCALE            # the Hadamard of 128 equal sums: one column
    # the int8 rounding of the weight's scale and the bf16 rounding of the result, 2^-8 each
    worst, rest = float((out[:, :, 0] / y - 1).abs().max()), float(out[:, :, 1:].abs().max())
    assert worst < 2.0**-7 and rest == 0.0
