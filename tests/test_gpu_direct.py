"""The sampled direct sum at the edges of its blocks and parts: targets around
the 64 of a block and the 4,096 of a tile, sources around the 256 of a part
and of a staged tile, coincident points, the Laplace kernel, both signs of
the wavenumber and phases beyond the table's range; against numpy in long
double."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(src, q, trg, kappa):
    s, ld = src.astype(np.longdouble), np.longdouble
    out = np.zeros(len(trg), dtype=np.clongdouble)
    size = np.zeros(len(trg))  # sum of the terms' magnitudes
    for i, t in enumerate(trg):
        d = s - t.astype(ld)
        r2 = (d * d).sum(1)
        ok = r2 >= ld(1e-16)
        r = np.sqrt(r2[ok])
        k = 1 / (4 * ld("3.14159265358979323846264338327950288") * r)
        e = np.cos(ld(kappa) * r) + 1j * np.sin(ld(kappa) * r)
        out[i] = (k * e * q[ok].astype(np.clongdouble)).sum()
        size[i] = float((k * np.abs(q[ok])).sum())
    return out, size


@pytest.mark.parametrize("kappa", [0.0, 7.0, -7.0, 3.0e6])
@pytest.mark.parametrize("n,m", [(1, 1), (255, 3), (257, 33), (1000, 64), (1000, 65),
                                 (16385, 10), (300, 4099)])
def test_direct_sum_edges(n, m, kappa):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = wl.sphere(n, seed=3)
    trg = wl.sphere(m, seed=17)
    trg[0] = src[0]  # a coincident pair is left out
    q = wl.charges(n, seed=5)
    print(f"case: {n} sources, {m} targets, kappa {kappa}", flush=True)
    p = dm.direct(src, q, trg, kappa)
    pick = np.unique(np.concatenate([np.arange(min(m, 40)), np.arange(max(0, m - 8), m)]))
    ref, size = _reference(src, q, trg[pick], kappa)
    # a term's relative error: 8 roundings of its value, and the phase's
    # |kappa r| (r <= 2) times 4 roundings of r
    tol = size * (8 + 4 * 2 * abs(kappa)) * 2.0 ** -53
    err = np.abs(p[pick] - ref)
    assert (err <= tol + 1e-300).all(), (err / (tol + 1e-300)).max()
