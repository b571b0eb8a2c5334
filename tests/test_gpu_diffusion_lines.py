"""Diffusion along one direction (blocks of lines: along x 254 cells of a line,
along y and z 14 cells of 16 lines) at the edges of the blocks, against the oracle
(the bound of tests/test_gpu_parity.py)."""
import pytest

from hotpath import TOL, complete_state, gpu_mix, norm_err, oracle_fields, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import htr_amd
    htr_amd.init(0)
    yield


@pytest.mark.parametrize("layout", ["soa", "aos", "padded"])
@pytest.mark.parametrize("d,n,lo,hi,walls", [
    (0, (252, 17, 3), None, None, None), (0, (254, 5, 2), None, None, None), (0, (511, 3, 2), (1, 0, 0), (509, 2, 1), None),
    (0, (1, 40, 3), None, None, None), (1, (15, 14, 3), None, None, None), (1, (17, 29, 5), (2, 1, 0), (16, 27, 3), None),
    (1, (33, 30, 7), (0, 1, 0), (32, 28, 6), "staggered"), (1, (20, 31, 3), (0, 1, 0), (19, 29, 2), "collocated"),
    (2, (16, 3, 14), None, None, None), (2, (9, 7, 43), (0, 2, 3), (8, 6, 40), None)])
def test_one_direction_at_block_edges(d, n, lo, hi, walls, layout):
    import htr_amd as H
    from emu_edges_state import state
    from oracle import oracle as O
    st, meta = state(n, 7, walls)
    st, om = complete_state(st, meta, n, sensors=False)
    lo, hi = lo or (0, 0, 0), hi or tuple(x - 1 for x in n)
    g, f = oracle_fields(st, 5, n)
    f["Conserved_t"] = 0.0
    O.diffusion_flux(g.with_rect(lo, hi), f, d, om)
    fs = to_gpu(st, 5, n, layout=layout)
    fs["Conserved_t"].fill_(0.0)
    H.update_using_diffusion_flux(fs, d, gpu_mix(meta), grid=fs.grid(lo, hi))
    torch.cuda.synchronize()
    # cells outside the rect stay as they are
    assert max(norm_err(fs["Conserved_t"].cpu().numpy(), f["Conserved_t"])) <= TOL
