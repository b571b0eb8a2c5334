"""Kernels at the edges of their dispatch rules and tiles, against the oracle
(the bounds of tests/test_gpu_parity.py: 1e-12 normalised per component)."""
import numpy as np
import pytest

from hotpath import TOL, air_state, complete_state, gpu_mix, norm_err, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import htr_amd
    htr_amd.init(0)
    yield


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("temps", [(800.0,), (6000.0007, 6000.0), (800.0, 3000.0), (900.0, 7000.0, 2500.0)])
def test_properties_across_polynomial_ranges(temps):
    """Waves whose lanes share one temperature range of the polynomials, and
    waves whose lanes alternate between ranges (or sit on a switch)."""
    import htr_amd as H
    st, meta = air_state(8, seed=2)
    n = (8, 8, 8)
    T = np.resize(np.asarray(temps) / meta["TRef"], 512).reshape(8, 8, 8)
    st = dict(st, temperature=T)
    ref, _ = complete_state(st, meta, n, sensors=False)
    fs = to_gpu({k: st[k] for k in ("pressure", "temperature", "MolarFracs", "velocity")}, 5, n)
    gm = gpu_mix(meta)
    H.update_properties_from_primitive(fs, gm)
    H.update_conserved_from_primitive(fs, gm)
    for k in ("rho", "mu", "lam", "Di", "SoS", "MassFracs", "Conserved"):
        assert max(norm_err(host(fs[k]), ref[k])) <= TOL, k


@pytest.mark.parametrize("layout", ["soa", "aos"])
@pytest.mark.parametrize("n,lo,hi", [((3, 2, 1), None, None), ((67, 5, 3), None, None), ((33, 17, 6), None, None),
                                     ((40, 37, 9), (1, 2, 3), (38, 36, 7)), ((96, 64, 40), None, None)])
def test_full_rhs_at_extent_edges(n, lo, hi, layout):
    """Extents below the stencil's reach, no multiple of a block, strip or
    brick, a rect inside the box, and one large enough for every kernel form."""
    import htr_amd as H
    from emu_edges_state import state
    from hotpath import oracle_fields
    from oracle import oracle as O
    st, meta = state(n, 3)
    st, om = complete_state(st, meta, n)
    lo, hi = lo or (0, 0, 0), hi or tuple(x - 1 for x in n)
    g, f = oracle_fields(st, 5, n)
    O.full_rhs(g.with_rect(lo, hi), f, O.SCHEME_HYBRID, 1.0, 0.0, 1e-4, 1, om)
    fs = to_gpu(st, 5, n, layout=layout)
    H.full_rhs(fs, O.SCHEME_HYBRID, (1.0, 0.0), 1e-4, True, gpu_mix(meta), grid=fs.grid(lo, hi))
    sl = (Ellipsis,) + tuple(slice(a, b + 1) for a, b in zip(lo[::-1], hi[::-1]))
    assert max(norm_err(host(fs["Conserved_t"])[sl], f["Conserved_t"][sl])) <= TOL
