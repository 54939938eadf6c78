"""The work this framework is used for, as timed cases: the blocks of a decoder layer over quantized weights.

Sizes are those of the 27B-class hybrid layer and LM head that bench.py times (r4dx_amd/workloads.py: hidden 5120, MLP
17408, attention q | k | v = 6144 | 1024 | 1024, GDN qkv | z = 10240 | 6144, inner 6144, vocabulary 248320), with the
row counts an engine meets: 1 (decode), a handful (verified drafts), up to 64 (a batch, or the tail of a prompt) and
128 / 256 (a prompt chunk). Drawn cases take other widths, such as a tensor-parallel share's or a smaller model's.

Kinds:
  linear   one trellis linear: input transform, product
  mlp      gate | up as one linear, silu(gate) * up fused with down's input transform, down
  attn     q | k | v as one linear; the output gate fused with o's input transform, o
  gdn      qkv | z as one linear; out's input transform, out
  mlp_i8 / gdn_i8   the same blocks over int8 activations (M = 256): "coarse" row scales, else per-128 scales
  head     the w4a16 LM head: fp32 logits and their argmax per row

The attention and the recurrence between a block's two projections are not part of the framework: their results are
inputs here. Every buffer a program keeps per layer (outputs, ws, tickets) is made once, in prepare().
"""
import math

import torch

from r4dx_amd import api, plan

F64 = torch.float64


# ---- the cases ----------------------------------------------------------------------------------------------------
def listed():
    return [
        # the narrowest projection of the layer (attn.k) for one token: launch latency is most of it
        dict(name="linear_k_m1", kind="linear", M=1, KB=4, H=5120, N=1024),
        # one decode step's MLP: two thirds of the layer's weight bytes
        dict(name="mlp_m1", kind="mlp", M=1, KB=4, H=5120, I=17408),
        # one decode step's GDN projections at the higher rate, the input transform inside the product
        dict(name="gdn_m1_kb5_fused", kind="gdn", M=1, KB=5, H=5120, n0=10240, n1=6144, n2=0, D=6144, fused=True),
        # verifying a draft of seven tokens plus one
        dict(name="attn_m8", kind="attn", M=8, KB=4, H=5120, n0=6144, n1=1024, n2=1024, D=6144, fused=False),
        # a batch of 29 sequences, or the end of a prompt
        dict(name="mlp_m29", kind="mlp", M=29, KB=4, H=5120, I=17408),
        # the 49-row end of a prompt at the higher rate
        dict(name="gdn_m49_kb5", kind="gdn", M=49, KB=5, H=5120, n0=10240, n1=6144, n2=0, D=6144, fused=False),
        # a prompt chunk, f16 activations
        dict(name="mlp_m256", kind="mlp", M=256, KB=4, H=5120, I=17408),
        dict(name="attn_m256_kb5", kind="attn", M=256, KB=5, H=5120, n0=6144, n1=1024, n2=1024, D=6144, fused=False),
        # a prompt chunk, int8 activations: row scales, and the finer per-128 scales
        dict(name="mlp_i8_coarse", kind="mlp_i8", M=256, KB=4, H=5120, I=17408, coarse=True),
        dict(name="gdn_i8_per128", kind="gdn_i8", M=256, KB=4, H=5120, n0=10240, n1=6144, D=6144, coarse=False),
        # the logits and the greedy token of one decode step, and of a batch of 24 at the finer group
        dict(name="head_m1_g64", kind="head", M=1, group=64, H=5120, V=248320),
        dict(name="head_m24_g32", kind="head", M=24, group=32, H=5120, V=248320),
    ]


def _log(rng, lo, hi, step):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "mlp", "attn", "gdn", "mlp", "attn", "gdn", "mlp_i8", "gdn_i8", "head"])
    if kind == "head":
        return dict(kind=kind, M=_log(rng, 1, 64, 1), group=rng.choice([32, 64]), H=_log(rng, 1024, 5120, 64),
                    V=_log(rng, 16384, 248320, 16))
    M = 256 if kind.endswith("_i8") else rng.choice([_log(rng, 1, 16, 1), _log(rng, 1, 64, 1), _log(rng, 17, 64, 1), 128, 256])
    KB = rng.choice([4, 5]) if kind.endswith("_i8") else rng.choice([3, 4, 4, 5, 5])
    step = 256 if kind.endswith("_i8") else 128   # the int8 products take K in pairs of 128-blocks
    H = _log(rng, 1024, 6144, step)
    c = dict(kind=kind, M=M, KB=KB, H=H)
    if kind == "linear":
        c.update(N=_log(rng, 512, 17408, 128))
    elif kind in ("mlp", "mlp_i8"):
        c.update(I=_log(rng, 2048, 17408, step) if H <= 5120 else _log(rng, 2048, 14336, step))
    else:
        D = _log(rng, 1024, 6144, step)
        if kind == "attn":
            kv = _log(rng, 256, 1024, 128)
            c.update(n0=D, n1=kv, n2=kv, D=D)
        else:
            c.update(n0=_log(rng, 2048, 10240, 128), n1=D, n2=0, D=D)
            if kind == "gdn_i8":
                del c["n2"]
    if kind in ("attn", "gdn"):
        c.update(fused=M <= 2 and rng.random() < 0.5)
    if kind.endswith("_i8"):
        c.update(coarse=rng.random() < 0.5)
    return c


# ---- inputs -------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _words(g, K, N, KB):
    """Every 32-bit word is a valid part of a trellis ring."""
    return torch.randint(-2**31, 2**31, (K * N * KB // 32,), dtype=torch.int32, device="cuda", generator=g)


def _signs(g, n):
    return (torch.rand(n, device="cuda", generator=g) < 0.5).float() * 2 - 1


def _svh(g, n):
    """Signed log-normal channel scales around 0.01, f16 numbers as a container stores them."""
    s = torch.exp(math.log(0.01) + 0.3 * torch.randn(n, device="cuda", generator=g)) * _signs(g, n)
    return s.half().float()


def _act(g, M, K, outliers=True):
    """bf16 activations: normal, one channel in 64 an outlier channel."""
    x = torch.randn(M, K, device="cuda", generator=g)
    if outliers:
        x = x * torch.where(torch.rand(K, device="cuda", generator=g) < 1 / 64, 8.0, 1.0)
    return x.bfloat16()


def _lin(g, K, N, KB, parts=1):
    return dict(K=K, N=N, KB=KB, w=_words(g, K, N, KB), suh=[_signs(g, K) for _ in range(parts)], svh=_svh(g, N))


def _inputs(case, seed):
    """The tensors of a case from the seed alone."""
    g = _gen(seed)
    c, kind = case, case["kind"]
    if kind == "head":
        V, H, G = c["V"], c["H"], c["group"]
        wq = torch.randint(-2**31, 2**31, (V * H // 8,), dtype=torch.int32, device="cuda", generator=g)
        n = V * H // G
        sc = torch.exp(math.log(0.02) + 0.3 * torch.randn(n, device="cuda", generator=g)).half()
        nz = -(1024.0 + torch.randint(0, 16, (n,), device="cuda", generator=g).float())
        wsz = (sc.view(torch.int16).int() & 0xFFFF) | (nz.half().view(torch.int16).int() << 16)
        return dict(a=torch.randn(c["M"], H, device="cuda", generator=g).half(), wq=wq, wsz=wsz)
    s = dict(x=_act(g, c["M"], c["H"]))
    if kind == "linear":
        s["l0"] = _lin(g, c["H"], c["N"], c["KB"])
    elif kind in ("mlp", "mlp_i8"):
        s["l0"] = _lin(g, c["H"], 2 * c["I"], c["KB"], 2)
        s["l1"] = _lin(g, c["I"], c["H"], c["KB"])
    else:
        ns = [n for n in (c["n0"], c["n1"], c.get("n2", 0)) if n]
        s["l0"] = _lin(g, c["H"], sum(ns), c["KB"], len(ns))
        s["l1"] = _lin(g, c["D"], c["H"], c["KB"])
        s["mix"] = _act(g, c["M"], c["D"], False)
        if kind == "attn":
            s["gate"] = _act(g, c["M"], c["D"], False)
    return s


OUT_SCALE = 1.0 / math.sqrt(128.0)


def _bufs(lin, M, ns=None):
    """What a program keeps per linear: its launch plan, output, ws and tickets."""
    K, N, KB = lin["K"], lin["N"], lin["KB"]
    L = api.lib()
    lin["M"] = M
    if M <= 64:
        if ns:          # same-input projections in one launch: this build's split for the decode kernel
            lin["sk"], lin["skg"] = 0, api.trellis_gemv_skg(K, N, KB)
        else:
            p = plan.linear_tuning(N, K, KB, M)
            lin["sk"], lin["skg"] = p.SK, p.SKG
        nbytes = L.r4d_gemm_trellis_nt_m64_ws_bytes(M, N, lin["skg"])
    else:
        lin["sk"], lin["skg"] = 2, api.trellis_m256_skg(K, N, KB)
        nbytes = L.r4d_gemm_trellis_nt_m256_ws_bytes(M, N, lin["skg"])
    lin["out"] = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    lin["ws"] = torch.empty(max(1, nbytes // 4), dtype=torch.float32, device="cuda")
    lin["tickets"] = api.TicketBuffer(N).t
    lin["a"] = [torch.empty((M, K), dtype=torch.float16, device="cuda") for _ in lin["suh"]]
    if ns:
        lin["n0"] = [sum(ns[:i]) for i in range(len(ns))]


def _bufs_i8(lin, parts_n, coarse):
    """The int8 form's: the weight scale table (made at load), the plan, the quantized activations' buffers."""
    K, N, KB = lin["K"], lin["N"], lin["KB"]
    lin["sw"] = api.trellis_i8_table(lin["w"], K, N, KB, coarse=coarse)
    p = plan.plan_trellis_i8(N, K, KB, parts=2 if parts_n else 1, part_n0=parts_n, coarse=coarse)
    lin["skw"], lin["skg"] = p.skw, p.SKG
    lin["out"] = torch.empty((256, N), dtype=torch.bfloat16, device="cuda")
    lin["ws"] = torch.empty(max(1, api.lib().r4d_gemm_trellis_nt_i8_ws_bytes(256, N, p.SKG) // 4), dtype=torch.float32,
                            device="cuda")
    lin["a8"] = [(torch.empty(256 * K, dtype=torch.int8, device="cuda"),
                  torch.empty(256 if coarse else (K // 128) * 256, dtype=torch.float32, device="cuda")) for _ in lin["suh"]]
    lin["n_split"] = parts_n


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, M = case["kind"], case["M"]
    s["kind"], s["case"] = kind, dict(case)
    if kind == "head":
        s["logits"] = torch.empty((M, case["V"]), dtype=torch.float32, device="cuda")
        s["idx"] = torch.empty(M, dtype=torch.int32, device="cuda")
        s["val"] = torch.empty(M, dtype=torch.float32, device="cuda")
    elif kind == "linear":
        _bufs(s["l0"], M)
    elif kind == "mlp":
        _bufs(s["l0"], M)
        _bufs(s["l1"], M)
    elif kind in ("attn", "gdn"):
        ns = [n for n in (case["n0"], case["n1"], case["n2"]) if n]
        _bufs(s["l0"], M, ns)
        _bufs(s["l1"], M)
    elif kind == "mlp_i8":
        _bufs_i8(s["l0"], case["I"], case["coarse"])
        _bufs_i8(s["l1"], None, case["coarse"])
    else:
        _bufs_i8(s["l0"], case["n0"], case["coarse"])
        _bufs_i8(s["l1"], None, case["coarse"])
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------
def _product(lin, a, n_split=None):
    a1 = a[1] if len(a) > 1 else None
    f = api.trellis_gemm_m64 if lin["M"] <= 64 else api.trellis_gemm_m256
    return f(a[0], lin["w"], lin["svh"], lin["K"], lin["N"], lin["KB"], skg=lin["skg"], a1=a1, n_split=n_split,
             out=lin["out"], ws=lin["ws"], tickets=lin["tickets"], out_scale=OUT_SCALE, sk=lin["sk"])


def _product_parts(lin, a):
    f = api.trellis_gemm_m64_parts if lin["M"] <= 64 else api.trellis_gemm_m256_parts
    return f(a, lin["n0"], lin["w"], lin["svh"], lin["K"], lin["N"], lin["KB"], skg=lin["skg"], out=lin["out"],
             ws=lin["ws"], tickets=lin["tickets"], out_scale=OUT_SCALE)


def _product_i8(lin, a, coarse):
    two = len(a) > 1
    return api.trellis_gemm_i8(a[0][0], a[0][1], lin["w"], lin["sw"], lin["svh"], lin["K"], lin["N"], lin["KB"],
                               coarse=coarse, a8_1=a[1][0] if two else None, sa_1=a[1][1] if two else None,
                               n_split=lin["n_split"], skw=lin["skw"], skg=lin["skg"], out=lin["out"], ws=lin["ws"],
                               out_scale=OUT_SCALE)


def run(state):
    s, c, kind = state, state["case"], state["kind"]
    if kind == "head":
        return list(api.w4a16_gemm_argmax(s["a"], s["wq"], s["wsz"], c["H"], c["V"], group=c["group"], out=s["logits"],
                                          out_idx=s["idx"], out_val=s["val"]))
    l0 = s["l0"]
    if kind == "linear":
        return _product(l0, api.trellis_input(s["x"], l0["suh"], outs=l0["a"]))
    l1 = s["l1"]
    if kind == "mlp":
        gu = _product(l0, api.trellis_input(s["x"], l0["suh"], outs=l0["a"]), c["I"])
        return _product(l1, [api.silu_mul_trellis(gu, c["I"], l1["suh"][0], out=l1["a"][0])])
    if kind in ("attn", "gdn"):
        if c["fused"]:
            y0 = api.trellis_gemv_xf_parts(s["x"], l0["suh"], l0["n0"], l0["w"], l0["svh"], l0["K"], l0["N"], l0["KB"],
                                           bf16=True, out=l0["out"], ws=l0["ws"], tickets=l0["tickets"],
                                           out_scale=OUT_SCALE)
        else:
            y0 = _product_parts(l0, api.trellis_input(s["x"], l0["suh"], outs=l0["a"]))
        if kind == "attn":
            a = [api.attn_gate_mul_trellis(s["mix"], s["gate"], l1["suh"][0], out=l1["a"][0])]
        else:
            a = api.trellis_input(s["mix"], l1["suh"], outs=l1["a"])
        return [y0, _product(l1, a)]
    coarse = c["coarse"]
    y0 = _product_i8(l0, api.trellis_input_i8(s["x"], l0["suh"], row_scale=coarse, outs=l0["a8"]), coarse)
    if kind == "mlp_i8":
        a = [api.silu_mul_trellis(y0, c["I"], l1["suh"][0], quant="row" if coarse else "blk", out=l1["a8"][0])]
        return _product_i8(l1, a, coarse)
    return [y0, _product_i8(l1, api.trellis_input_i8(s["mix"], l1["suh"], row_scale=coarse, outs=l1["a8"]), coarse)]


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def work(case):
    c, kind, M = case, case["kind"], case["M"]
    if kind == "head":
        V, H = c["V"], c["H"]
        return {"bytes": V * H // 2 + V * (H // c["group"]) * 4 + M * H * 2 + M * V * 4 + M * 8, "flops": 2 * M * V * H}
    H, KB = c["H"], c["KB"]

    def lin(K, N, parts, table):   # words, sign vectors, channel scales, int8 weight scales
        return K * N * KB // 8 + 4 * K * parts + 4 * N + table
    i8, fine = kind.endswith("_i8"), kind.endswith("_i8") and not c["coarse"]
    tab = lambda K, N: 0 if not i8 else (K // 128) * N * 4 if fine else N * 4
    if kind == "linear":
        return {"bytes": lin(H, c["N"], 1, 0) + M * (H + c["N"]) * 2, "flops": 2 * M * H * c["N"]}
    if kind in ("mlp", "mlp_i8"):
        I = c["I"]
        return {"bytes": lin(H, 2 * I, 2, tab(H, 2 * I)) + lin(I, H, 1, tab(I, H)) + M * (H + H) * 2,
                "flops": 2 * M * H * 3 * I}
    ns = [n for n in (c["n0"], c["n1"], c.get("n2", 0)) if n]
    N, D = sum(ns), c["D"]
    mix = D * (2 if kind == "attn" else 1)
    return {"bytes": lin(H, N, len(ns), tab(H, N)) + lin(D, H, 1, tab(D, H)) + M * (H + N + mix + H) * 2,
            "flops": 2 * M * (H * N + D * H)}


def tolerance(case):
    """About four times what the same products show with their K split otherwise (another order of the fp32 sums)."""
    kind = case["kind"]
    if kind == "head":
        # fp32 sums over K of exact products (2e-7 off the 64-bit ones); the token may differ in a near tie
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.01}
    if kind in ("mlp", "mlp_i8"):
        # bf16 (and int8) roundings between the two products: one that moves by a place passes through the second product
        return {"rel": 2.3e-3, "max": 0.031}
    # one product: a bf16 rounding moves by one place (2^-8) now and then
    return {"rel": 2e-4, "max": 0.031}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------
def _decode(lin, n_lo, n_hi):
    """Columns [n_lo, n_hi) (multiples of 32) of the linear's weights as the format defines them: float64 [K][n]. A tile
    of 16 x 16 is a ring of 256 KB bits; position p's 16-bit state ends at bit KB (p + 1); the weight is one f16
    rounding of (1024 + the byte sum of state * 0x83DCD12D) * f16(0x1EEE) + f16(0xC931)."""
    K, KB = lin["K"], lin["KB"]
    KT, R = K // 16, 8 * KB
    w = lin["w"].view(lin["N"] // 32, KT, 2, R)[n_lo // 32:n_hi // 32].long() & 0xFFFFFFFF
    p = torch.arange(256, device="cuda")
    start = (KB * (p + 1) - 16) % (32 * R)
    i0, off = start // 32, start % 32
    two = (w[..., i0] << 32) | w[..., (i0 + 1) % R]       # stream bit 32 w is bit 31 of word w
    state = (two >> (48 - off)) & 0xFFFF
    h = (state * 0x83DCD12D) & 0xFFFFFFFF
    s = (h & 255) + ((h >> 8) & 255) + ((h >> 16) & 255) + (h >> 24)
    kinv = torch.tensor([0x1EEE], dtype=torch.int16).view(torch.float16).double().item()
    bias = torch.tensor([0xC931 - 0x10000], dtype=torch.int16).view(torch.float16).double().item()
    v = ((1024 + s).double() * kinv + bias).half().double()
    t, j = p // 8, p % 8
    c, m = t // 4, t % 4
    k = 2 * m + torch.tensor([0, 1, 8, 9], device="cuda")[j & 3]
    n = c + 8 * (j >> 2)
    out = torch.empty(v.shape[0], KT, 2, 256, dtype=F64, device="cuda")
    out[..., k * 16 + n] = v
    out = out.view(-1, KT, 2, 16, 16).permute(1, 3, 0, 2, 4)     # [kt][k][pair][tile][n]
    return out.reshape(K, n_hi - n_lo)


def _fwht(x):
    """Unnormalised Hadamard over each 128 of the last dimension."""
    h = torch.ones(1, 1, dtype=F64, device="cuda")
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ h).reshape(x.shape)


def _transform(x, suh):
    return _fwht(x * suh.double()) / math.sqrt(128.0)


def _finish(lin, sums):
    return _fwht(sums) * lin["svh"].double() * OUT_SCALE


def _exact_linear(lin, a, ends):
    """a[i]: float64 [M][K] of the columns [ends[i - 1], ends[i])."""
    outs, step = [], 2048
    for i, e in enumerate(ends):
        lo = ends[i - 1] if i else 0
        for n in range(lo, e, step):
            outs.append(a[i] @ _decode(lin, n, min(e, n + step)))
    return _finish(lin, torch.cat(outs, 1))


def _silu_mul(gu, inter):
    g, u = gu[:, :inter], gu[:, inter:]
    return g * torch.sigmoid(g) * u


def _quant(a, fine):
    """The int8 activation of a transformed input: f16 values, amax / 127 scales (fp32) per row or per row and 128."""
    v = a.half().float()
    v = v.view(v.shape[0], -1, 128) if fine else v.view(v.shape[0], 1, -1)
    m = v.abs().amax(-1, keepdim=True)
    s = torch.where(m > 0, m / 127.0, torch.ones_like(m))
    return torch.clamp(torch.round(v / s), -127, 127).double(), s.double()   # [M][blocks][k], [M][blocks][1]


def _exact_linear_i8(lin, a, ends, fine):
    outs, step = [], 2048
    for i, e in enumerate(ends):
        q, sa = _quant(a[i], fine)
        lo = ends[i - 1] if i else 0
        for n in range(lo, e, step):
            w = _decode(lin, n, min(e, n + step))
            w = w.view(-1, 128, w.shape[1]) if fine else w[None]             # [blocks][k][n]
            m = w.abs().amax(1, keepdim=True).float()
            s = torch.where(m > 0, m / 127.0, torch.ones_like(m))
            rs = torch.clamp((1.0 / s), max=60000.0).half()
            seff = (1.0 / rs.float()).double()
            wq = torch.round(w * rs.double())
            acc = torch.zeros(q.shape[0], w.shape[2], dtype=F64, device="cuda")
            for b in range(w.shape[0]):
                acc += (q[:, b] @ wq[b]) * sa[:, b] * seff[b]
            outs.append(acc)
    return _finish(lin, torch.cat(outs, 1))


def exact(case, seed):
    s, c, kind = _inputs(case, seed), case, case["kind"]
    if kind == "head":
        V, H, G = c["V"], c["H"], c["group"]
        a = s["a"].double()
        wq = s["wq"].view(V // 16, H // 64, 2, 16, 4)
        sz = s["wsz"].view(V // 16, H // G, 16)
        scale = (sz & 0xFFFF).to(torch.int16).view(torch.float16).double()
        zero = -(sz >> 16).to(torch.int16).view(torch.float16).double() - 1024.0
        nib = torch.tensor([0, 8, 1, 9, 2, 10, 3, 11], device="cuda")
        logits = torch.empty(c["M"], V, dtype=F64, device="cuda")
        step = 512                                              # 16-row tiles at a time
        for t in range(0, V // 16, step):
            w = wq[t:t + step]
            q = torch.empty(w.shape[0], H // 64, 16, 64, dtype=F64, device="cuda")
            for i in range(8):
                v = (((w >> (4 * i)) & 15) ^ 8).double()        # [tile][block][lh][row][s]
                for lh in range(2):
                    for ss in range(4):
                        q[..., 16 * ss + 4 * lh + int(nib[i])] = v[:, :, lh, :, ss]
            q = q.permute(0, 2, 1, 3).reshape(-1, 16, H // G, G)
            z = zero[t:t + step].permute(0, 2, 1)[..., None]
            f = scale[t:t + step].permute(0, 2, 1)[..., None]
            logits[:, 16 * t:16 * (t + w.shape[0])] = a @ ((q - z) * f).reshape(-1, H).T
        val, idx = logits.max(1)
        return [logits, idx.int(), val]
    x, l0 = s["x"].double(), s["l0"]
    a = [_transform(x, h) for h in l0["suh"]]
    if kind == "linear":
        return _exact_linear(l0, a, [l0["N"]])
    l1 = s["l1"]
    if kind == "mlp":
        gu = _exact_linear(l0, a, [c["I"], 2 * c["I"]])
        return _exact_linear(l1, [_transform(_silu_mul(gu, c["I"]), l1["suh"][0])], [c["H"]])
    if kind == "mlp_i8":   # the gate | up rows and the product are bf16 numbers before they are quantized
        gu = _exact_linear_i8(l0, a, [c["I"], 2 * c["I"]], not c["coarse"]).bfloat16().double()
        h = _silu_mul(gu, c["I"]).bfloat16().double()
        return _exact_linear_i8(l1, [_transform(h, l1["suh"][0])], [c["H"]], not c["coarse"])
    ends = [c["n0"], c["n0"] + c["n1"]] + ([c["n0"] + c["n1"] + c["n2"]] if c.get("n2") else [])
    mix = s["mix"].double()
    if kind == "gdn_i8":
        return [_exact_linear_i8(l0, a, ends, not c["coarse"]),
                _exact_linear_i8(l1, [_transform(mix, l1["suh"][0])], [c["H"]], not c["coarse"])]
    if kind == "attn":
        mix = mix * torch.sigmoid(s["gate"].double())
    return [_exact_linear(l0, a, ends), _exact_linear(l1, [_transform(mix, l1["suh"][0])], [c["H"]])]
