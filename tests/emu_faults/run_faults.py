"""Child process of tests/test_emu_faults.py: library calls that fail on the
way (tests/emu_faults/hip), through the kernel source compiled for the CPU.
Prints "CASE <name> <figures>"; exits non-zero on the first that is wrong."""
import ctypes as C
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [os.path.join(os.path.dirname(HERE), "emu")]

import numpy as np  # noqa: E402
import run_emu as R  # noqa: E402
from hotpath import complete_state, gpu_mix, tgv_state  # noqa: E402

H = R.H
H.init(0)
LIB = H.lib()
for _name, _res, _arg in (("arm", None, C.c_long), ("calls", C.c_long, None), ("launches", C.c_long, None),
                          ("limit", None, C.c_size_t), ("unfollowed", C.c_int, C.c_void_p)):
    _f = getattr(LIB, "hipfault_" + _name)
    _f.restype, _f.argtypes = _res, [_arg] if _arg else []


def check(ok, name, *figures):
    print("CASE", name, *figures, flush=True)
    if not ok:
        sys.exit(3)


def small_vortex(n=(6, 5, 4)):
    st, meta = tgv_state(6)
    st = {k: v[..., :n[2], :n[1], :n[0]].copy() for k, v in st.items()}
    st, _ = complete_state(st, meta, n)
    for d in range(3):
        st["shockSensor%d" % d][:] = 0            # every face takes the TENO branch
    return R.to_host_fs(st, 1, n), gpu_mix(meta)


def side_streams():
    """Whatever call or launch of a right-hand side on side streams fails: the
    caller's stream follows all the work that was launched."""
    H.rhs_overlap(True)
    failed = 0
    for k in range(1, 200):
        fs, mix = small_vortex()
        LIB.hipfault_arm(k)
        try:
            H.full_rhs(fs, 0, (1.0, 0.0), 1e-3, False, mix)
            error = None
        except Exception as e:
            error = str(e)
        calls = LIB.hipfault_calls()
        LIB.hipfault_arm(0)
        left = LIB.hipfault_unfollowed(None)
        if left:
            check(False, "side_streams", k, "left", left, error)
        if calls < k:
            break
        failed += error is not None
    check(failed >= 20 and error is None, "side_streams", k, failed)


def air_box(n=(6, 5, 4)):
    from emu_edges_state import state
    st, meta = state(n, 2)
    st, _ = complete_state(st, meta, n)
    rng = np.random.default_rng(0)
    for d in range(3):
        st["shockSensor%d" % d] = (rng.random(n[::-1]) > 0.05).astype(np.uint8)
    return R.to_host_fs(st, 5, n), gpu_mix(meta)


def faces(n):
    """faces of the largest direction of a box"""
    return max(n[0] * n[1] * n[2] // n[d] * (n[d] + 1) for d in range(3))


def teno_memory():
    """A pure TENO sweep takes 22 doubles a face beside its fluxes (9 doubles a
    face) and nothing larger."""
    n = (15, 14, 15)               # (more than the fixed part of a workspace)
    fs, mix = air_box(n)
    LIB.hipfault_limit(22 * 8 * faces(n))
    try:
        H.update_using_teno_euler_flux(fs, 1, "TENO", (1.0, 0.0), 1e-4, mix)
        error = None
    except Exception as e:
        error = str(e)
    check(error is None, "teno_memory", error)


def rhs_memory():
    """A full right-hand side where there is memory for one direction's face
    fluxes (9 doubles a face) but not for three: the same result to the bit, and
    not a call more that is refused; the larger buffer is tried for again by a
    reservation alone."""
    n = (15, 14, 15)
    out = []
    for limit in (0, 22 * 8 * faces(n)):
        fs, mix = air_box(n)
        LIB.hipfault_limit(limit)
        if limit:
            # (a workspace that has grown keeps what it has: another stream's)
            R.A.stream_ptr = lambda stream=None: C.c_void_p(8)
        for call in range(2 if limit else 1):
            try:
                H.full_rhs(fs, 0, (1.0, 0.0), 1e-4, True, mix)
                H.workspace_reserve(fs, mix)
                error = None
            except Exception as e:
                error = str(e)
            check(error is None, "rhs_memory", limit, call, error)
            out.append(fs["Conserved_t"].numpy().copy())
    check(all((o == out[0]).all() for o in out), "rhs_memory equal")


def mixture_upload():
    """A finalize that fails after its allocation, then more reactions, then one
    that does not fail: the image has room for them all."""
    from htr_amd import cases, mechanism
    mech = mechanism.synthetic_30(0)
    few = dict(mech, reactions=mech["reactions"][:1])
    check_, codes = R.A.check, []
    for k in (2, 3):                               # the copy of the mixture, the copy of its rows
        R.A.check = codes.append
        LIB.hipfault_arm(k)
        mix = H.Mixture.from_mechanism(few)
        LIB.hipfault_arm(0)
        r = mech["reactions"][0]
        two = lambda key, t: ((C.c_int * 2)(*[e[0] for e in r[key]]), (t * 2)(*[e[1] for e in r[key]]))
        ei, en = two("educts", C.c_float)
        pi, pn = two("products", C.c_float)
        for _ in range(179):
            codes.append(LIB.htr_mix_add_reaction(mix.h, r["kind"], r["A"], r["n"], r["EovR"], 1, 2, ei, en, 2, pi, pn,
                                                  0, None, None))
        xr = (C.c_double * 30)(*mech["XiRef"])
        codes.append(LIB.htr_mix_finalize(mix.h, mech["PRef"], mech["TRef"], mech["LRef"], xr))
        R.A.check = check_
        failed = [c for c in codes if c]
        check(len(failed) == 1, "mixture_upload", k, failed)
        codes.clear()


if __name__ == "__main__":
    for which in sys.argv[1:]:
        globals()[which]()
