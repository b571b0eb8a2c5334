"""The list of TENO faces in each of the sizes its blocks take (256, 1024 and
4096 faces: below 2^18, below 2^20 and from 2^20 faces on), on boxes on both sides
of the lines, against the oracle: values (the bound of tests/test_gpu_parity.py)
and the decision of every face."""
import numpy as np
import pytest

from hotpath import TOL, complete_state, gpu_mix, norm_err, oracle_fields, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,faces", [((63, 65, 63), 1), ((64, 66, 65), 4), ((99, 103, 101), 4), ((101, 105, 103), 16)])
def test_listed_faces(n, faces):
    import htr_amd as H
    from emu_edges_state import state
    from oracle import oracle as O
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    H.init(0)
    st, meta = state(n, 11)
    st, om = complete_state(st, meta, n, sensors=False)
    rng = np.random.default_rng(0)
    for d in range(3):
        count = n[0] * n[1] * n[2] // n[d] * (n[d] + 1)
        assert faces == (16 if count >= 2 ** 20 else 4 if count >= 2 ** 18 else 1)
        # one cell in eight asks for TENO: neither every face nor none of a block
        st["shockSensor%d" % d] = (rng.random(n[::-1]) > 0.125).astype(np.uint8)
    gm = gpu_mix(meta)
    for d in range(3):
        g, f = oracle_fields(st, 5, n)
        f["Conserved_t"] = 0.0
        dec = np.zeros(f["rho"].shape, np.uint32)
        O.euler_flux(g, f, d, O.SCHEME_HYBRID, 1.0, 0.0, 1e-4, om, dec)
        fs = to_gpu(st, 5, n, decisions=True)
        fs["Conserved_t"] = 0.0
        H.update_using_hybrid_euler_flux(fs, d, (1.0, 0.0), 1e-4, gm, diag=True)
        torch.cuda.synchronize()
        got = fs["decisions%d" % d].cpu().numpy().astype(np.uint32)
        assert 0.1 < np.mean((dec & 1) == 0) < 0.9
        assert np.array_equal(got & 1, dec & 1)
        same = got == dec
        assert np.mean(~same) <= 1e-4
        prev = np.roll(same, 1, axis=2 - d)
        assert max(norm_err(fs["Conserved_t"].cpu().numpy(), f["Conserved_t"], mask=same & prev)) <= TOL
