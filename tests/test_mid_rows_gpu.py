"""r4d_gemm_trellis_nt_m64 above 16 rows, and below where a K slice of A is past 48 KiB: the chunked kernel (trellis_mid.hip)
and the forms of two and more row tiles that stage the slice whole, at the sizes where their staging, their row tiles and
the balanced form can go wrong. Each row must carry the bits the same launch
gives it in a batch of at most 16 whose slice of A stays within 48 KiB -- one row tile, A staged whole: neither the chunks nor
the cuts -- in both summation orders, at every rate, for slices whose last step is not whole, parts that are empty or shorter
than the others, two input parts and more than 8 slices. The balanced form (cut units) at every number of row tiles and every
rate, at one slice and at two; unsplit, it must also match the launch without ws and tickets, which cuts nothing, and stay
inside ws_bytes and tickets_bytes. Every launch leaves its tickets zero."""
import numpy as np
import pytest

from r4dx_amd import workloads as WL

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from r4dx_amd import api  # noqa: E402
from r4dx_amd.loader import lib  # noqa: E402
from gpu_util import banner, dev  # noqa: E402

CASES = [   # (M, K, N, KB, SKG, sk)
    (17, 128, 128, 4, 1, 2), (32, 128, 256, 4, 2, 2), (33, 640, 128, 5, 8, 2), (48, 1152, 256, 3, 1, 2),
    (49, 1152, 256, 3, 9, 2), (64, 2048, 384, 5, 16, 2), (64, 5120, 128, 4, 1, 1), (31, 4992, 256, 4, 3, 2),
    (18, 128, 128, 4, 1, 0), (32, 640, 256, 5, 5, 4), (48, 384, 128, 3, 3, 0), (49, 2304, 256, 5, 2, 0),
    (64, 4992, 256, 4, 1, 0), (57, 1152, 128, 4, 9, 0), (64, 128, 128, 5, 8, 0),
    # slices whose last step is not whole, in the chunked kernel: past 48 KiB, and parts of an even number of steps
    (64, 3456, 256, 5, 8, 2), (40, 5760, 128, 4, 8, 2), (23, 9856, 128, 3, 8, 1), (50, 1664, 256, 4, 8, 0), (20, 3456, 128, 4, 8, 0),
    (32, 3456, 256, 5, 8, 4),
    # balanced (40 steps a unit): columns -n are column groups such that there are n SKG more units than CUs (rounded down)
    (29, 2560, -1, 4, 1, 2), (64, 2560, -44, 4, 1, 2), (37, 2560, -5, 3, 1, 2), (13, 2560, -3, 5, 1, 2), (10, 2560, -2, 4, 1, 1),
    (58, 2560, -2, 5, 1, 1), (37, 5120, -12, 5, 2, 2), (57, 5120, -3, 4, 2, 2), (20, 5120, -2, 3, 2, 1), (16, 5120, -5, 4, 2, 2),
    (45, 5120, -1, 4, 2, 2),
]


def _cols(N, skg):
    return N if N > 0 else 128 * (torch.cuda.get_device_properties(0).multi_processor_count // skg - N)


def _whole_rows(K, skg, sk):
    """The most rows whose slice of A the whole-staging kernel takes: 32 bytes per row and k-tile of the four parts' (SK 1, 2:
    one part's) whole steps, 48 KiB in all."""
    steps, parts = -(-(K // 16 // skg) // 4), 1 if sk in (1, 2) else 4
    rows = 48 * 1024 // (32 * 4 * parts * -(-steps // parts))
    assert rows > 0
    return min(rows, 16)


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
    N = _cols(N, skg)
    banner("chunked rows", M, K, N, KB, skg, sk)
    g = torch.Generator(device="cuda").manual_seed(M * 7 + K)
    w = torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)
    svh = dev(WL.svh_scales(N, 3))
    a = torch.randn(M, K, device="cuda", generator=g).half()
    two = N > 128 and K % 3 != 0                  # two input parts where there are two column groups
    a1 = torch.randn(M, K, device="cuda", generator=g).half() if two else None
    n_split = 128 if two else None
    got, raw = _run(a, w, svh, K, N, KB, skg, sk, a1, n_split)
    step = _whole_rows(K, skg, sk)
    for r in range(0, M, step):
        part = a[r:r + step].contiguous()
        p1 = a1[r:r + step].contiguous() if two else None
        ref, ref_raw = _run(part, w, svh, K, N, KB, skg, sk, p1, n_split)
        same = torch.equal(got[r:r + step], ref), torch.equal(raw[r:r + step], ref_raw)
        assert same == (True, True), f"rows {r}.."
    if skg == 1 and sk in (1, 2):
        bare = api.trellis_gemm_m64(a, w, svh, K, N, KB, skg=1, a1=a1, n_split=n_split, out_scale=0.1, sk=sk)
        same = torch.equal(bare.view(torch.int16), got)
        assert same


@pytest.mark.parametrize("M,KB", [(64, 4), (29, 5), (12, 3)])
def test_unsplit_stays_inside_its_workspace(M, KB):
    """SKG 1 in the SK 1 / 2 order with ws and tickets, cut units or not: nothing outside ws_bytes(M, N, 1) and
    tickets_bytes(N) is written, the tickets end at zero."""
    L, K = lib(), 2560
    for N in (_cols(-7, 1), 512):
        banner("unsplit workspace", M, K, N, KB)
        g = torch.Generator(device="cuda").manual_seed(N)
        w = torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)
        a = torch.randn(M, K, device="cuda", generator=g).half()
        nw, nt = L.r4d_gemm_trellis_nt_m64_ws_bytes(M, N, 1) // 4, L.r4d_gemm_trellis_nt_m64_tickets_bytes(N) // 4
        ws = torch.full((nw + 8192,), -1, dtype=torch.int32, device="cuda")
        tk = torch.full((nt + 8192,), 7, dtype=torch.int32, device="cuda")
        tk[4096:4096 + nt] = 0
        out = api.trellis_gemm_m64(a, w, dev(WL.svh_scales(N, 3)), K, N, KB, skg=1, ws=ws[4096:4096 + nw],
                                   tickets=tk[4096:4096 + nt], sk=2)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(out.float()).all())
        assert int((ws[:4096] != -1).sum()) == 0 and int((ws[4096 + nw:] != -1).sum()) == 0
        assert int((tk[:4096] != 7).sum()) == 0 and int((tk[4096 + nt:] != 7).sum()) == 0
        assert int(tk[4096:4096 + nt].abs().sum()) == 0


@pytest.mark.parametrize("M,K,KB,skg,sk", [(1, 40960, 4, 1, 0), (5, 20480, 3, 2, 2), (9, 10880, 5, 2, 0), (13, 5120, 4, 1, 2),
                                           (16, 13952, 4, 4, 4)])
def test_long_slices_up_to_16_rows(M, K, KB, skg, sk):
    """A slice of A past 48 KiB at up to 16 rows: each row carries the bits it has
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
    # fp32 sums of K products round off about sqrt(K) 2^-24 of their rms, 1.2e-5 at K 40960; twice that is allowed
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
