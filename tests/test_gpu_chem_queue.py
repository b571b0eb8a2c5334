"""Implicit chemistry with a wave per cell where a block integrates several cells
one after the other (fewer blocks than cells), where the FP32 factors are too
coarse for the refinement, and from a temperature that no cell has."""
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
    htr_amd.chem_launch_config(0, 0)


def update(st, n, gm, dt, precision, lanes, blocks_per_cu):
    import htr_amd as H
    H.chem_launch_config(lanes, blocks_per_cu)
    fs = to_gpu(st, 30, n, nsteps=True)
    fs["Conserved_t"] = 0.0
    H.update_chemistry(fs, dt, gm, precision=precision, diag=True)
    torch.cuda.synchronize()
    return [fs[k].cpu().numpy().copy() for k in ("Conserved", "temperature", "nsteps")]


@pytest.mark.parametrize("precision", [0, 0x10, 1, 0x11])
def test_blocks_take_several_cells(precision):
    """512 different cells on 256 blocks and on 512: nothing that a block keeps
    from one cell reaches the next.  FP64 also equals the group kernel."""
    from htr_amd import cases
    n = (8, 8, 8)
    st, meta = cases.chem30_box(8, seed=2)
    st, _ = complete_state(st, meta, n, sensors=False)
    gm = gpu_mix(meta)
    few = update(st, n, gm, 1e-7, precision, 64, 1)
    other = update(st, n, gm, 1e-7, precision, *((64, 8) if precision & 1 else (32, 0)))
    assert few[2].min() > 0 and few[2].max() > few[2].min()
    for a, b in zip(few, other):
        assert np.array_equal(a, b)


def _refined(A, b):
    """Sweeps of the FP32 solve with FP64 residuals until a correction is below
    1e-15 of the solution, negative where one is not half of the one before
    (chem_wave.hpp: equilibrate, refine)."""
    def pow2_inv(a):
        return 2.0 ** -(np.floor(np.log2(a)) + 1)
    rs = pow2_inv(np.abs(A).max(1))
    cs = pow2_inv(np.abs(rs[:, None] * A).max(0))
    M = (rs[:, None] * A * cs).astype(np.float32)
    n = len(M)
    perm, vv = np.arange(n), np.float32(1) / np.abs(M).max(1)
    for j in range(n):
        k = j + int(np.argmax(vv[j:] * np.abs(M[j:, j])))
        for a in (M, vv, perm):
            a[[j, k]] = a[[k, j]]
        M[j + 1:, j] /= M[j, j]
        M[j + 1:, j + 1:] -= np.outer(M[j + 1:, j], M[j, j + 1:])
    x, prev = np.zeros(n), 0.0
    for it in range(9):
        y = ((b - A @ x) * rs)[perm].astype(np.float32)
        for k in range(n):
            y[k + 1:] -= M[k + 1:, k] * y[k]
        for k in range(n - 1, -1, -1):
            y[k] /= M[k, k]
            y[:k] -= M[:k, k] * y[k]
        c = cs * y
        x = x + c
        nc, nx = np.abs(c).max(), np.abs(x).max()
        if it > 0 and not nc > 1e-15 * nx:
            return it
        if it > 0 and not nc < 0.5 * prev:
            return -it
        prev = nc
    return -9


@pytest.mark.parametrize("precision", [1, 0x11])
def test_refinement_gives_way_to_fp64_factors(precision):
    """Over 1e-3 s the matrix of a cell's first attempt (2/dt against rates of 1e9)
    is too ill-conditioned to refine: the step goes on with FP64 factors in the
    Jacobian's place, and the attempt after it forms the Jacobian again.  Held to
    the FP64 path as the parity tests hold both to the oracle (ten times the
    step tolerance)."""
    from htr_amd import cases
    from oracle import oracle as O
    dt, n = 1e-3, (5, 1, 1)
    box, meta = cases.chem30_box(3, seed=1)
    box, om = complete_state(box, meta, (3, 3, 3), sensors=False)
    pick = [0, 2, 6, 8, 20]
    st = {k: np.ascontiguousarray(v.reshape(v.shape[:-3] + (27,))[..., pick].reshape(v.shape[:-3] + (1, 1, 5)))
          for k, v in box.items()}
    for c in range(5):
        x = np.ascontiguousarray(st["Conserved"][:, 0, 0, c])
        J, _ = O.chem_jacobian(om, x, np.zeros(34), float(st["temperature"][0, 0, c]), O.JAC_ANALYTIC)
        assert _refined(2.0 / dt * np.eye(34) - J, J @ x) < 0
    gm = gpu_mix(meta)
    got = update(st, n, gm, dt, precision, 64, 0)
    ref = update(st, n, gm, dt, precision & ~1, 64, 0)
    assert got[2].min() > 1 and np.isfinite(ref[0]).all()
    assert np.abs(got[0][:30] - ref[0][:30]).max() <= 1e-9
    assert np.abs(got[0][33] - ref[0][33]).max() <= 1e-12 * np.abs(ref[0][33]).max()


def test_temperature_of_minus_one():
    """A guess of -1 is a temperature like another: not a number afterwards, as
    with the group kernel."""
    from htr_amd import cases
    st, meta = cases.chem30_box(2, seed=0)
    st, _ = complete_state(st, meta, (2, 2, 2), sensors=False)
    st["temperature"] = np.full_like(st["temperature"], -1.0)
    gm = gpu_mix(meta)
    a, b = (update(st, (2, 2, 2), gm, 1e-8, 0x10, lanes, 0) for lanes in (64, 32))
    assert np.isnan(b[1]).all()
    for u, v in zip(a, b):
        assert np.array_equal(u, v, equal_nan=True)
