"""Child process of tests/test_emu_lines.py: diffusion along one direction
through the CPU emulation, against the oracle, at the edges of the blocks' lines:
along x 254 cells of a line a block, along y and z 14 cells of 16 lines.  Prints
"CASE <name> 0 <cells>"; exits non-zero on the first mismatch."""
import os
import sys

sys.path[:0] = [os.path.dirname(os.path.abspath(__file__))]

import run_edges as E  # noqa: E402

R, H, O, state = E.R, E.H, E.O, E.state


def main():
    H.init(0)
    for d, n, lo, hi, walls in ((0, (252, 1, 1), None, None, None), (0, (253, 2, 1), None, None, None),
                                (0, (256, 1, 2), None, None, None), (0, (40, 17, 2), (2, 0, 0), (38, 16, 1), None),
                                (1, (5, 13, 3), None, None, None), (1, (8, 14, 2), None, None, None),
                                (1, (17, 15, 1), None, None, None), (1, (4, 30, 5), (1, 2, 0), (3, 28, 3), None),
                                (1, (6, 16, 3), (0, 1, 0), (5, 14, 2), "staggered"),
                                (1, (6, 17, 3), (0, 1, 0), (5, 15, 2), "collocated"),
                                (2, (3, 5, 12), None, None, None), (2, (16, 1, 14), None, None, None),
                                (2, (7, 5, 29), (0, 1, 1), (6, 3, 27), None)):
        for layout in ("soa", "aos"):
            st, meta = state(n, sum(n), walls)
            st, om = R.complete_state(st, meta, n)
            a, b = lo or (0, 0, 0), hi or tuple(x - 1 for x in n)
            g, f = R.oracle_fields(st, 5, n)
            f["Conserved_t"] = 0.25
            O.diffusion_flux(g.with_rect(a, b), f, d, om)
            fs = R.to_host_fs(st, 5, n, layout=layout)
            fs["Conserved_t"] = 0.25
            H.update_using_diffusion_flux(fs, d, R.gpu_mix(meta), grid=fs.grid(a, b))
            E.report("diffusion_%s_d%d_%dx%dx%d" % ((layout, d) + n), fs["Conserved_t"].numpy(), f["Conserved_t"],
                     n[0] * n[1] * n[2])


if __name__ == "__main__":
    main()
