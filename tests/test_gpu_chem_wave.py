"""Implicit chemistry with a wave per cell (64 lanes) against the group kernel
(32 lanes), which forms the same operations in the same order: equal to the
bit.  Mechanisms at the edges of the wave kernel's rules: a last round of
reactions that is nearly empty or full, third bodies, irreversible reactions,
coefficients of 2, fractional coefficients (the general power), no reaction at
all, and mass fractions at their clip."""
import copy

import numpy as np
import pytest

from hotpath import complete_state, gpu_mix, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import htr_amd
    htr_amd.init(0)
    yield


def mechanism_of(kind, base):
    mech = copy.deepcopy(base)
    r = mech["reactions"]
    if kind == "none":
        r = []
    elif kind.startswith("n"):
        r = r[:int(kind[1:])]
    elif kind == "forms":
        for i, q in enumerate(r):
            if i % 5 == 0:
                q.update(kind=1, thirdb=[(i % 30, 2.5), ((i + 7) % 30, 0.5)] if i % 10 else [])
            if i % 7 == 0:
                q["has_backward"] = False
            if i % 9 == 0:
                # (reversible, its reverse rate would leave the range the solver integrates)
                q.update(educts=[(q["educts"][0][0], 2.0)], A=q["A"] * 1e-2, has_backward=False)
    elif kind == "fractional":
        for q in r[::11]:
            q["educts"] = [(q["educts"][0][0], 1.5)] + q["educts"][1:]
    mech["reactions"] = r
    return mech


@pytest.mark.parametrize("kind,precision", [("none", 0), ("n1", 0x10), ("n64", 0), ("n65", 0), ("forms", 0),
                                            ("forms", 0x10), ("fractional", 0), ("trace", 0), ("trace", 0x10)])
def test_wave_kernel_equals_group_kernel(kind, precision):
    import htr_amd as H
    from htr_amd import cases
    n = (3, 3, 3)
    st, meta = cases.chem30_box(3, seed=1)
    if kind == "trace":                  # most species at the clip of Y or below it
        X = np.full_like(st["MolarFracs"], 1e-60)
        X[:4] = st["MolarFracs"][:4]
        st["MolarFracs"] = X / X.sum(0)
    meta = dict(meta, mech=mechanism_of(kind, meta["mech"]))
    st, om = complete_state(st, meta, n, sensors=False)
    gm = gpu_mix(meta)
    out = []
    for lanes in (64, 32):
        H.chem_launch_config(lanes, 0)
        fs = to_gpu(st, 30, n, nsteps=True)
        fs["Conserved_t"] = 0.0
        if kind == "n65":
            fs["Conserved_t"][:30] = 1e-4 * fs["Conserved"][:30]
        H.update_chemistry(fs, 1e-8, gm, precision=precision, diag=True)
        torch.cuda.synchronize()
        out.append([fs[k].cpu().numpy().copy() for k in ("Conserved", "temperature", "nsteps")])
    H.chem_launch_config(0, 0)
    assert out[0][2].min() > 0 and np.all(np.isfinite(out[0][0]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
