"""Regenerate the pointwise-algebra include files.

    python -m sympygr_amd.codegen

writes
    oracle/gen/bssn_algebra.inc              (CPU restatement: the whole RHS algebra)
    sympygr_amd/csrc/gen/bssn_algebra_pw.inc (GPU pointwise kernel, advection in tails)
    oracle/gen/ccz4_algebra.inc, sympygr_amd/csrc/gen/ccz4_algebra_pw.inc (CCZ4)
    {oracle,sympygr_amd/csrc}/gen/bssn_constraints.inc
    {oracle,sympygr_amd/csrc}/gen/bssn_constraints_psi4.inc (with the Weyl scalar Psi4)
and prints the flop counts of the emitted algebra.
"""
from __future__ import annotations

import os
import sys

from .bssn_eqs import bssn_rhs_stages, constraint_stages
from .ccz4_eqns import ccz4_rhs_stages
from .emit import emit_stages

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

HEADER = """// Generated by `python -m sympygr_amd.codegen` from
// sympygr_amd/codegen/bssn_eqs.py -- do not edit.
// BSSN RHS pointwise algebra (standard gauge, constant eta): {flops} flops,
// {ntemps} named temporaries, {ninputs} inputs.
// Needs in scope: type R; R lambda0..3, lambda_f0..1, eta; macros
// BSSN_U(f), BSSN_D1(f,d), BSSN_D2(f,s), BSSN_ADV(f), BSSN_LAP(f), BSSN_GDB(j), BSSN_OUT(f,v),
// BSSN_OUT_ALT(f,v) (Rochester-gauge value of f), R xi1, xi2,
// BSSN_BARRIER() (may be empty).
"""


# Cheap first-derivative outputs first, then K and the Gamma-driver, then
# At (which needs the Ricci tensor): each group's temporaries die before the
# next group starts, which keeps the FP64 kernel free of scratch spills.
OUTPUT_ORDER = [0, 6, 7, 8, 1, 12, 13, 14, 15, 16, 17, 2, 3, 9, 4, 10, 5, 11, 18, 19, 20, 21, 22, 23]


def generate(write=True):
    S = bssn_rhs_stages()
    E = emit_stages(S, output_order=OUTPUT_ORDER, barrier=False)
    text = HEADER.format(flops=E.flops, ntemps=E.ntemps, ninputs=len(E.inputs)) + E.text
    if write:
        for rel in ("oracle/gen/bssn_algebra.inc",):
            path = os.path.join(ROOT, rel)
            os.makedirs(os.path.dirname(path), exist_ok=True)
            with open(path, "w") as f:
                f.write(text)
    return E


# Output order of the GPU pointwise kernel.  The outputs that need the
# Christoffel symbols, A^ij and D_i D_j alpha (At with the Ricci tensor, K,
# Gt, B) come first, the first-derivative equations (alpha, beta, chi, gt)
# last: their inputs are all read by the first part already, and in this
# order the one kernel needs no more registers than the first part alone
# (the other order holds the first part's inputs across it and spills).
# The advection of every output arrives in a per-output tail
# (bssn_eqs.TAIL_FIELDS), not through the algebra.
GROUPS = {
    "pw": [18, 19, 20, 21, 22, 23, 2, 3, 9, 4, 10, 5, 11,   # At, K, Gt, B
           0, 6, 7, 8, 1, 12, 13, 14, 15, 16, 17],          # alpha, beta, chi, gt
}

TAIL_NOTE = """// Advection is not part of this algebra: the caller adds each output's tail
// (c_f adv f + sigma KO f, c_f the advection coefficient of the equation; for
// B^i (1 - lambda3) adv Gt^i + lambda2 adv B^i + sigma KO B^i).
"""


def generate_groups(write=True):
    S = bssn_rhs_stages(tails=True)
    res = {}
    for g, order in GROUPS.items():
        E = emit_stages(S, output_order=order, barrier=False, alt_early=True)
        text = HEADER.format(flops=E.flops, ntemps=E.ntemps, ninputs=len(E.inputs)) + TAIL_NOTE + E.text
        if write:
            with open(os.path.join(ROOT, f"sympygr_amd/csrc/gen/bssn_algebra_{g}.inc"), "w") as f:
                f.write(text)
        res[g] = (E, text)
    return res


CONSTRAINT_HEADER = """// Generated by `python -m sympygr_amd.codegen` from
// sympygr_amd/codegen/bssn_eqs.py (constraint_stages) -- do not edit.
// Hamiltonian and momentum constraints: {flops} flops, {ninputs} inputs.
// Outputs BSSN_OUT(0, ham), BSSN_OUT(1..3, mom0..2).
"""


def generate_constraints(write=True):
    S = constraint_stages()
    E = emit_stages(S, output_order=[0, 1, 2, 3], barrier=False)
    text = CONSTRAINT_HEADER.format(flops=E.flops, ninputs=len(E.inputs)) + E.text
    if write:
        for rel in ("sympygr_amd/csrc/gen/bssn_constraints.inc", "oracle/gen/bssn_constraints.inc"):
            with open(os.path.join(ROOT, rel), "w") as f:
                f.write(text)
    return E, text


PSI4_HEADER = """// Generated by `python -m sympygr_amd.codegen` from
// sympygr_amd/codegen/bssn_eqs.py (constraint_stages(psi4=True)) -- do not edit.
// Hamiltonian and momentum constraints and the Weyl scalar Psi4
// (GR/constraints.py:46-173): {flops} flops, {ninputs} inputs.
// Needs in scope: type R; R px, py, pz (the point's coordinates).
// Outputs BSSN_OUT(0, ham), BSSN_OUT(1..3, mom0..2), BSSN_OUT(4, psi4_real),
// BSSN_OUT(5, psi4_img).
"""


def generate_constraints_psi4(write=True):
    S = constraint_stages(psi4=True)
    E = emit_stages(S, output_order=[0, 1, 2, 3, 4, 5], barrier=False)
    text = PSI4_HEADER.format(flops=E.flops, ninputs=len(E.inputs)) + E.text
    if write:
        for rel in ("sympygr_amd/csrc/gen/bssn_constraints_psi4.inc", "oracle/gen/bssn_constraints_psi4.inc"):
            with open(os.path.join(ROOT, rel), "w") as f:
                f.write(text)
    return E, text


CCZ4_HEADER = """// Generated by `python -m sympygr_amd.codegen` from
// sympygr_amd/codegen/ccz4_eqns.py -- do not edit.
// CCZ4 right-hand side pointwise algebra: {flops} flops, {ntemps} named
// temporaries, {ninputs} inputs; fields as BSSN plus Theta (24).
// Needs in scope: type R; R lambda0..3, lambda_f0..1, eta, kappa1..3; macros
// BSSN_U(f), BSSN_D1(f,d), BSSN_D2(f,s), BSSN_ADV(f), BSSN_LAP(f), BSSN_GDB(j), BSSN_OUT(f,v).
"""

# GPU output order of CCZ4: as BSSN's, Theta with the heavy part.
CCZ4_GROUPS = {
    "pw": [18, 19, 20, 21, 22, 23, 2, 24, 3, 9, 4, 10, 5, 11,
           0, 6, 7, 8, 1, 12, 13, 14, 15, 16, 17],
}


def generate_ccz4(write=True):
    """oracle/gen/ccz4_algebra.inc (whole algebra, with advection) and
    sympygr_amd/csrc/gen/ccz4_algebra_pw.inc (GPU kernel, tails)."""
    S = ccz4_rhs_stages()
    E = emit_stages(S, output_order=list(range(25)), barrier=False)
    texts = {"oracle/gen/ccz4_algebra.inc": CCZ4_HEADER.format(flops=E.flops, ntemps=E.ntemps,
                                                               ninputs=len(E.inputs)) + E.text}
    ST = ccz4_rhs_stages(tails=True)
    res = {"all": E}
    for g, order in CCZ4_GROUPS.items():
        EG = emit_stages(ST, output_order=order, barrier=False)
        texts[f"sympygr_amd/csrc/gen/ccz4_algebra_{g}.inc"] = CCZ4_HEADER.format(
            flops=EG.flops, ntemps=EG.ntemps, ninputs=len(EG.inputs)) + TAIL_NOTE + EG.text
        res[g] = EG
    if write:
        for rel, text in texts.items():
            with open(os.path.join(ROOT, rel), "w") as f:
                f.write(text)
    return res, texts


if __name__ == "__main__":
    E = generate(write="--dry-run" not in sys.argv)
    print(f"bssn algebra: {E.flops} flops, {E.ntemps} temporaries, {len(E.inputs)} inputs")
    for g, (EG, _) in generate_groups(write="--dry-run" not in sys.argv).items():
        print(f"bssn algebra group {g}: {EG.flops} flops, {len(EG.inputs)} inputs")
    EC, _ = generate_constraints(write="--dry-run" not in sys.argv)
    print(f"constraints: {EC.flops} flops, {len(EC.inputs)} inputs")
    EP, _ = generate_constraints_psi4(write="--dry-run" not in sys.argv)
    print(f"constraints with psi4: {EP.flops} flops, {len(EP.inputs)} inputs")
    R4, _ = generate_ccz4(write="--dry-run" not in sys.argv)
    for g, EG in R4.items():
        print(f"ccz4 algebra {g}: {EG.flops} flops, {len(EG.inputs)} inputs")
