"""Child process of tests/test_emu_chem.py: implicit chemistry with a wave per
cell (64 lanes) through the CPU emulation against the oracle, air (two cells, the
first block takes both) or the 30-species mechanism (one), one Rosenbrock step.
Prints "CASE <name> <max abs difference> <cells>"; exits non-zero on the first
mismatch (FP64: any difference; refined solves: ten times the step tolerance)."""
import os
import sys

sys.path[:0] = [os.path.dirname(os.path.abspath(__file__))]

import run_emu as R  # noqa: E402
import numpy as np  # noqa: E402
from hotpath import air_state  # noqa: E402
from htr_amd import cases  # noqa: E402

H, O = R.H, R.O


def main():
    H.init(0)
    air = sys.argv[1] == "air"
    n, ns = ((2, 1, 1), 5) if air else ((1, 1, 1), 30)
    st, meta = air_state(2, seed=0, composition="per-seed") if air else cases.chem30_box(2, seed=0)
    st = {k: np.ascontiguousarray(v[..., :n[2], :n[1], :n[0]]) for k, v in st.items()}
    st, om = R.complete_state(st, meta, n, sensors=False)
    H.chem_launch_config(64, 1)
    for precision in [int(a, 0) for a in sys.argv[2:]]:
        g, f = R.oracle_fields(st, ns, n)
        f["Conserved_t"] = 0.0
        O.chem_update(g, f, 1e-9, om, jacobian=O.JAC_ANALYTIC if precision & 0x10 else O.JAC_FD)
        fs = R.to_host_fs(st, ns, n, nsteps=True)
        fs["Conserved_t"] = 0.0
        H.update_chemistry(fs, 1e-9, R.gpu_mix(meta), precision=precision, diag=True)
        d = float(np.abs(fs["Conserved"].numpy() - f["Conserved"]).max())
        print("CASE %s_%#x %.3e %d" % (sys.argv[1], precision, d, n[0]), flush=True)
        if not d <= (1e-9 if precision & 1 else 0.0) or int(fs["nsteps"].min()) < 1:
            sys.exit(3)


if __name__ == "__main__":
    main()
