"""States for the edge tests of the per-cell kernels."""
import numpy as np

from htr_amd import cases


def state(n, seed, walls=None):
    """Random 5-species air on n cells; walls: None, "staggered", "collocated"
    (along y, ghosts included in n)."""
    nx, ny, nz = n
    rng = np.random.default_rng(seed)
    shape = (nz, ny, nx)
    Y = rng.dirichlet([8.0, 2.0, 0.5, 0.5, 0.5], size=shape).transpose(3, 0, 1, 2)
    X = Y / cases.AIR_W[:, None, None, None]
    st = dict(pressure=0.1 * (1.0 + 0.2 * rng.random(shape)), temperature=6.0 + 4.0 * rng.random(shape),
              MolarFracs=X / X.sum(0), velocity=rng.standard_normal((3,) + shape))
    m = [cases.periodic_metrics(k, 0.1 * k) for k in n]
    if walls:
        m[1] = cases.wall_metrics(ny - 2, 0.1 * ny, 0.8, collocated=walls == "collocated")[:4]
    cases.set_metrics(st, m, n)
    meta = dict(kind="airmix", vorticityScale=1.0, **cases.AIR_REFS)
    return st, meta
