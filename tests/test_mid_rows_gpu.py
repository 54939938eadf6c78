"""r4d_gemm_trellis_nt_m64 for 17..64 rows (trellis_mid.hip) at the sizes where its staging, its row tiles and its balanced
form can go wrong: each row must carry the bits the same launch gives it in a batch of at most 16 rows (another kernel), in
both summation orders, at every rate, for slices whose last step is not whole, parts that are empty or shorter than the
others, cut units, two input parts and more than 8 slices; and the launch leaves its tickets zero."""
import numpy as np
import pytest

from r4dx_amd import workloads as WL

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from r4dx_amd import api  # noqa: E402
from gpu_util import banner, dev  # noqa: E402

CASES = [   # (M, K, N, KB, SKG, sk)
    (17, 128, 128, 4, 1, 2), (32, 128, 256, 4, 2, 2), (33, 640, 128, 5, 8, 2), (48, 1152, 256, 3, 1, 2),
    (49, 1152, 256, 3, 9, 2), (64, 2048, 384, 5, 16, 2), (64, 5120, 128, 4, 1, 1), (31, 4992, 256, 4, 3, 2),
    (18, 128, 128, 4, 1, 0), (32, 640, 256, 5, 5, 4), (48, 384, 128, 3, 3, 0), (49, 2304, 256, 5, 2, 0),
    (64, 4992, 256, 4, 1, 0), (57, 1152, 128, 4, 9, 0), (64, 128, 128, 5, 8, 0),
    # balanced: more units than CUs and not a multiple of them (40 steps a unit), at one and more slices
    (29, 2560, 128 * 257, 4, 1, 2), (64, 2560, 128 * 300, 4, 1, 2), (37, 5120, 128 * 140, 5, 2, 2),
]


def _run(a, w, svh, K, N, KB, skg, sk, a1=None, n_split=None):
    M = a.shape[0]
    ws = torch.full((max(1, skg * M * N),), float("nan"), dtype=torch.float32, device="cuda")
    tk = api.TicketBuffer(N).t
    out = [api.trellis_gemm_m64(a, w, svh, K, N, KB, skg=skg, a1=a1, n_split=n_split, ws=ws, tickets=tk, out_scale=0.1,
                                sk=sk).view(torch.int16) for _ in range(2)]
    raw = api.trellis_gemm_m64(a, w, None, K, N, KB, skg=skg, a1=a1, n_split=n_split, ws=ws, tickets=tk, raw=True, sk=sk)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
    assert int(tk.abs().sum()) == 0
    return out[0], raw.view(torch.int32)


@pytest.mark.parametrize("M,K,N,KB,skg,sk", CASES)
def test_rows_equal_small_batches(M, K, N, KB, skg, sk):
    banner("17..64 rows", M, K, N, KB, skg, sk)
    g = torch.Generator(device="cuda").manual_seed(M * 7 + K)
    w = torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)
    svh = dev(WL.svh_scales(N, 3))
    a = torch.randn(M, K, device="cuda", generator=g).half()
    two = N > 128 and K % 3 != 0                  # two input parts where there are two column groups
    a1 = torch.randn(M, K, device="cuda", generator=g).half() if two else None
    n_split = 128 if two else None
    got, raw = _run(a, w, svh, K, N, KB, skg, sk, a1, n_split)
    for r in range(0, M, 16):
        part = a[r:r + 16].contiguous()
        p1 = a1[r:r + 16].contiguous() if two else None
        ref, ref_raw = _run(part, w, svh, K, N, KB, skg, sk, p1, n_split)
        assert torch.equal(got[r:r + 16], ref), f"rows {r}.."
        assert torch.equal(raw[r:r + 16], ref_raw), f"raw rows {r}.."


@pytest.mark.parametrize("M,K,KB,skg,sk", [(1, 40960, 4, 1, 0), (5, 20480, 3, 2, 2), (9, 10880, 5, 2, 0), (13, 5120, 4, 1, 2),
                                           (16, 13952, 4, 4, 4)])
def test_long_slices_up_to_16_rows(M, K, KB, skg, sk):
    """A slice of A past what the M <= 16 kernel stages whole goes through the chunked form: each row carries the bits it has
    alone (one row of the same slice fits, or is itself past the limit at 40960), and the raw sums are those of the decoded
    weights."""
    N = 256
    g = torch.Generator(device="cuda").manual_seed(K)
    w = torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)
    svh = dev(WL.svh_scales(N, 3))
    a = torch.randn(M, K, device="cuda", generator=g).half()
    got, raw = _run(a, w, svh, K, N, KB, skg, sk)
    for r in range(M):
        one, one_raw = _run(a[r:r + 1].contiguous(), w, svh, K, N, KB, skg, sk)
        assert torch.equal(got[r:r + 1], one) and torch.equal(raw[r:r + 1], one_raw)
    q = api.trellis_reconstruct(w, K, N, KB).view(torch.float16).double()
    ref = a.double() @ q
    # fp32 sums of K products: error below K 2^-24 of the terms' magnitudes' sum, here within 1e-5 of the rms
    assert float((raw.view(torch.float32).double() - ref).abs().max()) < 2e-5 * float(ref.pow(2).mean().sqrt())


def test_unsplit_without_ws():
    """SKG = 1 with no ws: data-parallel, the bits of the launch that has one."""
    K, N, M = 2560, 128 * 258, 21
    g = torch.Generator(device="cuda").manual_seed(5)
    w = torch.randint(-2**31, 2**31, (K * N // 8,), dtype=torch.int32, device="cuda", generator=g)
    svh = dev(WL.svh_scales(N, 3))
    a = torch.randn(M, K, device="cuda", generator=g).half()
    got = api.trellis_gemm_m64(a, w, svh, K, N, 4, skg=1, out_scale=0.1, sk=2).view(torch.int16)
    assert torch.equal(got, _run(a, w, svh, K, N, 4, 1, 2)[0])
