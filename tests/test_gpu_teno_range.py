"""TENO-LAD where the ratio of the smoothness indicators overflows: its
cut-off takes that for the sharpest jump there is.  A jump of 1e295 beside a
collocated wall, where the flat stencil (whose ratio overflows) has no weight
and the two others straddle the jump: with the cut-off of a smooth flow both
would be dropped and the flux would not be a number."""
import numpy as np
import pytest

from hotpath import complete_state, gpu_mix, oracle_fields, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("first", [1.0, 1e295])
@pytest.mark.parametrize("at", [2, 12])
def test_tenolad_with_overflowing_ratio(first, at):
    import htr_amd as H
    from htr_amd import cases
    from oracle import oracle as O
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    H.init(0)
    n, lo, hi = (2, 14, 2), (0, 1, 0), (1, 12, 1)
    shape = n[::-1]
    p = np.full(shape, first)
    p[:, at:, :] = 1e295 if first == 1.0 else 1.0
    st = dict(pressure=p, temperature=p.copy(), MolarFracs=np.ones((1,) + shape), velocity=np.zeros((3,) + shape))
    cases.set_metrics(st, [cases.periodic_metrics(2), cases.wall_metrics(12, 1.0, 1.5, collocated=True)[:4],
                           cases.periodic_metrics(2)], n)
    meta = cases.tgv(4)[1]
    st, om = complete_state(st, meta, n, sensors=False)
    g, f = oracle_fields(st, 1, n)
    f["Conserved_t"] = 0.0
    O.euler_flux(g.with_rect(lo, hi), f, 1, O.SCHEME_TENOLAD, 1.0, 0.0, 1e-3, om, None)
    fs = to_gpu(st, 1, n)
    fs["Conserved_t"] = 0.0
    H.update_using_teno_euler_flux(fs, 1, "TENOLAD", (1.0, 0.0), 1e-3, gpu_mix(meta), grid=fs.grid(lo, hi))
    torch.cuda.synchronize()
    got, ref = fs["Conserved_t"].cpu().numpy(), f["Conserved_t"]
    assert np.isfinite(ref).any(axis=(1, 3)).any()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = np.isfinite(ref)
    assert np.allclose(got[ok], ref[ok], rtol=1e-12, atol=0.0)
