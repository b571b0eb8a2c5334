"""Child process of tests/test_emu_edges.py: the per-cell Kennedy-Gruber and
diffusion kernels through the CPU emulation of tests/emu/hip, against the
oracle, on the forms their indexing can go wrong on: extents of one to three
cells (the stencil wraps more than once around them), extents that are no
multiple of a block, strip or brick, a rect that starts inside the box, walls
with the staggered or collocated ghost cells in the rect (the minus face of a
line's first cell is then its own face), one and several directions.  Prints
"CASE <name> 0 <cells>"; exits
non-zero on the first mismatch."""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [HERE]

import run_emu as R  # noqa: E402
import numpy as np  # noqa: E402
from emu_edges_state import state  # noqa: E402

H, O = R.H, R.O


def report(name, got, ref, cells):
    """Bit for bit (and not a number in the same places)."""
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    same = np.array_equal(got, ref, equal_nan=True)
    print("CASE %s %s %d" % (name, "0" if same else "differs", cells), flush=True)
    if not same:
        sys.exit(3)


R.report = report


def main():
    H.init(0)
    which = sys.argv[1]
    for k, (n, lo, hi, walls) in enumerate([
            ((1, 2, 3), None, None, None), ((5, 3, 1), None, None, None), ((67, 3, 2), None, None, None),
            ((3, 35, 2), None, None, None), ((9, 7, 11), (1, 2, 3), (8, 5, 9), None),
            ((6, 10, 3), None, None, "staggered"), ((6, 9, 3), None, None, "collocated"),
            ((5, 12, 3), (0, 1, 0), (4, 10, 2), "staggered"), ((35, 6, 5), None, None, None)]):
        st, meta = state(n, 10 + k, walls)
        st, om = R.complete_state(st, meta, n)
        # the ghost cells' own faces have no TENO stencil: Kennedy-Gruber only
        schemes = ((O.SCHEME_KG, "kg"),) + (() if walls and not lo else ((O.SCHEME_HYBRID, "hybrid"),))
        lo, hi = lo or (0, 0, 0), hi or tuple(x - 1 for x in n)
        cells = int(np.prod(n))
        if which == "sweeps":
            for d in range(3):
                for scheme, label in schemes:
                    R.euler(st, meta, n, om, d, scheme, "%s_%d" % (label, k), lo=lo, hi=hi)
                g, f = R.oracle_fields(st, 5, n)
                f["Conserved_t"] = 0.0
                O.diffusion_flux(g.with_rect(lo, hi), f, d, om)
                fs = R.to_host_fs(st, 5, n)
                fs["Conserved_t"] = 0.0
                H.update_using_diffusion_flux(fs, d, R.gpu_mix(meta), grid=fs.grid(lo, hi))
                report("diffusion_%d_d%d" % (k, d), fs["Conserved_t"].numpy(), f["Conserved_t"], cells)
        else:
            for scheme, label in schemes:
                for layout in ("soa", "aos"):
                    g, f = R.oracle_fields(st, 5, n)
                    O.full_rhs(g.with_rect(lo, hi), f, scheme, 1.0, 0.0, 1e-4, 1, om)
                    fs = R.to_host_fs(st, 5, n, layout=layout)
                    H.full_rhs(fs, scheme, (1.0, 0.0), 1e-4, True, R.gpu_mix(meta), grid=fs.grid(lo, hi))
                    report("rhs_%s_%s_%d" % (label, layout, k), fs["Conserved_t"].numpy(), f["Conserved_t"], cells)


if __name__ == "__main__":
    main()
