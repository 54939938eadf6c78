"""Writes this build's MI355X tuning rows in the reference engine's own C++ row formats, so the engine's planners
(`PickTuning` / `TrellisTuningFor` / `PlanTrellisM256` / `PlanTrellisI8`, src/model/linear.cpp:243-767) read them
unchanged in place of the RDNA4 tables:

* gemm_tuning_table_trellis.inc (+ _tp2): `{Layout::kTrellis, N, K, M, {WV, SK, MB, NPW, NT, SKG, U}, 0, KB}` rows
  (src/model/gemm_tuning_table_trellis.inc:30-40's format) inside `static const GemmTuningRow kGemmTuningTable[]`;
* gemm_tuning_table_trellis_i8.inc, _i8c.inc (+ _tp2): `{N, K, KB, skw, skg}` rows
  (src/model/gemm_tuning_table_trellis_i8c.inc:6-20's format) inside kTrellisI8Table / kTrellisI8cTable /
  kTrellisI8Tp2Table / kTrellisI8cTp2Table.

The rows come from the library's own planners (r4dx_amd/plan.py over r4d_mi355x_*_skg), which are the plan this
build measures:

* M = 1 (every M <= 16 chunk runs it, the row-identity rule of linear.cpp:33-53): SK = 4 (the 4-wave split order),
  SKG = r4d_mi355x_trellis_gemv_skg, NT = 1;
* M = 32 and M = 64 (prefill chunks): SK = 2 (the one-wave-per-pair order, which r4d_gemm_trellis_nt_m256 reproduces
  bit for bit) and the M = 256 plan's SKG, so PlanTrellisM256 (linear.cpp:696-722) reads a legal (SK, SKG) off the
  M = 64 row and finds skw = 2;
* WV = 4, NPW = 1 (a 128-column group per workgroup row, legal at every part boundary the loader accepts),
  MB = ceil(M / 16), U = 1: knobs this build accepts and ignores, chosen so every row passes the engine's
  TrellisRowFits (linear.cpp:243-255).

    python -m r4dx_amd.tuning_inc [out_dir]      (default: r4dx_amd/tables)
"""
import os
import sys

from . import plan

PKG = os.path.dirname(os.path.abspath(__file__))
TABLES = os.path.join(PKG, "tables")

# The engine's trellis linear classes of the 27B hybrid model (gemm_tuning_table_trellis.inc's comments), then the
# BASELINE config-1 shapes and the same-input merges this build launches as one linear: (N, K, name).
TP1_SHAPES = [
    (10240, 5120, "gdn.in_proj_qkv"),
    (6144, 5120, "gdn.in_proj_z, attn.q"),
    (5120, 6144, "gdn.out_proj, attn.o"),
    (12288, 5120, "attn.qg"),
    (1024, 5120, "attn.k, attn.v"),
    (34816, 5120, "mlp.gate_up"),
    (5120, 17408, "mlp.down"),
    (17408, 5120, "mlp.gate, mlp.up"),
    (16384, 5120, "gdn.in_proj_qkv | z (one launch)"),
    (8192, 5120, "attn.q | k | v (one launch)"),
]
# One TP = 2 rank's shapes (gemm_tuning_table_trellis_tp2.inc's classes).
TP2_SHAPES = [
    (5120, 5120, "gdn.in_proj_qkv"),
    (3072, 5120, "gdn.in_proj_z"),
    (5120, 3072, "gdn.out_proj, attn.o"),
    (6144, 5120, "attn.qg"),
    (512, 5120, "attn.k, attn.v"),
    (17408, 5120, "mlp.gate_up"),
    (5120, 8704, "mlp.down"),
]
RATES = (4, 5)
BANDS = (1, 32, 64)


def trellis_row(N, K, KB, M):
    """(WV, SK, MB, NPW, NT, SKG, U) of the M-band row, from plan.linear_tuning (which the kernels' _check accepts)."""
    p = plan.linear_tuning(N, K, KB, M)
    if not p.ok:
        raise ValueError(f"no plan for N={N} K={K} KB={KB} M={M}: {p.why}")
    return (4, p.SK, (M + 15) // 16, 1, 1 if M <= plan.DECODE_M else 0, p.SKG, 1)


def i8_row(N, K, KB, coarse):
    p = plan.plan_trellis_i8(N, K, KB, coarse=coarse)
    if not p.ok:
        raise ValueError(f"no int8 plan for N={N} K={K} KB={KB}: {p.why}")
    return (p.skw, p.SKG)


_HEAD = """// GENERATED by r4dx_amd/tuning_inc.py from libr4d_mi355x's planners (r4d_mi355x_trellis_gemv_skg,
// r4d_mi355x_trellis_m256_skg, r4d_mi355x_trellis_i8_skg via r4dx_amd/plan.py); do not edit by hand.
"""


def trellis_inc(shapes, tp2):
    lines = [_HEAD.rstrip(),
             "// MI355X (gfx950) trellis rows" + (" for one TP = 2 rank's shapes" if tp2 else "") + ", in the format of",
             "// src/model/gemm_tuning_table_trellis.inc:",
             "//   {Layout::kTrellis, N, K, M, {WV, SK, MB = MT, NPW = NP, NT, SKG, U}, group = 0, rate = KB}",
             "// M = 1 serves every chunk of M <= 16 (row identity): SK = 4 (the 4-wave split order) and the GEMV's SKG.",
             "// M = 32 / 64 serve prefill chunks: SK = 2 (the one-wave-per-pair order r4d_gemm_trellis_nt_m256 reproduces)",
             "// and the M = 256 plan's SKG, so PlanTrellisM256 reads a legal (SK, SKG) off the M = 64 row (skw = 2).",
             "// WV, MB, NPW, NT, U are accepted and ignored by this build; they are set so TrellisRowFits accepts",
             "// every row. Include it inside its own namespace, as the reference's table.",
             "static const GemmTuningRow kGemmTuningTable[] = {"]
    for KB in RATES:
        for N, K, name in shapes:
            for M in BANDS:
                t = trellis_row(N, K, KB, M)
                lines.append("    {Layout::kTrellis, %d, %d, %d, {%s}, 0, %d},  // %s" %
                             (N, K, M, ", ".join(str(v) for v in t), KB, name))
    lines.append("};")
    return "\n".join(lines) + "\n"


def i8_inc(shapes, coarse, tp2):
    name = "kTrellisI8" + ("c" if coarse else "") + ("Tp2" if tp2 else "") + "Table"
    lines = [_HEAD.rstrip(),
             "// MI355X (gfx950) " + ("coarse-scale " if coarse else "") + "int8 prefill rows" +
             (" for one TP = 2 rank's shapes" if tp2 else "") + " (r4d_gemm_trellis_nt_i8" + ("c" if coarse else "") +
             "), in the format of",
             "// src/model/gemm_tuning_table_trellis_i8" + ("c" if coarse else "") + ".inc: {N, K, KB, skw, skg}. skg is this "
             "build's K split; skw",
             "// (2, 4 or 8) is checked by the kernel's rule (K / 128) % (skw skg) == 0 and otherwise unused.",
             "const TrellisI8Row %s[] = {" % name]
    for N, K, nm in shapes:
        for KB in RATES:
            skw, skg = i8_row(N, K, KB, coarse)
            lines.append("    {%d, %d, %d, %d, %d},  // %s KB%d" % (N, K, KB, skw, skg, nm, KB))
    lines.append("};")
    return "\n".join(lines) + "\n"


def files():
    """{file name: text} of every table."""
    out = {
        "gemm_tuning_table_trellis.inc": trellis_inc(TP1_SHAPES, False),
        "gemm_tuning_table_trellis_tp2.inc": trellis_inc(TP2_SHAPES, True),
    }
    for coarse in (False, True):
        c = "c" if coarse else ""
        out[f"gemm_tuning_table_trellis_i8{c}.inc"] = i8_inc(TP1_SHAPES, coarse, False)
        out[f"gemm_tuning_table_trellis_i8{c}_tp2.inc"] = i8_inc(TP2_SHAPES, coarse, True)
    return out


def write(out_dir=TABLES):
    os.makedirs(out_dir, exist_ok=True)
    for name, text in files().items():
        with open(os.path.join(out_dir, name), "w") as f:
            f.write(text)
    return sorted(files())


if __name__ == "__main__":
    print("\n".join(write(sys.argv[1] if len(sys.argv) > 1 else TABLES)))
