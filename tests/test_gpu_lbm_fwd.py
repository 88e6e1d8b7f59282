"""Collide-stream and forward x-transform, and the inverse one of the step
before, in one launch (small contexts of narrow rows): the coupled step against the same step in a context that one
wide channel more keeps on the separate launches, and on both sides of the
size limit.  The same bits."""
import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "ux", "uy", "cpos", "cneg", "psi")


def start(sizes, precision, **kw):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, kappa_h=min(4.0, 0.15 * ny)) for nx, ny in sizes],
                     precision=precision, **kw)
    for ch, (nx, ny) in enumerate(sizes):
        rng = np.random.default_rng(100 * nx + ny)
        zw = -1 + 0.3 * rng.standard_normal(nx)
        s.set_wall_profile(ch, psi_lo=zw, psi_hi=zw[::-1].copy())
        g = rng.standard_normal((5, ny, nx))
        s.set_fields(ch, 1 + 1e-3 * g[0], 1e-3 * g[1], 1e-3 * g[2], 1 + 0.1 * g[3], 1 + 0.1 * g[4])
    s.init_equilibrium()
    return s


def state(s, ch):
    out = {f: s.get_field(ch, f) for f in FIELDS}
    return out | {sp: s.get_populations(ch, sp) for sp in ("f", "h", "g")}


def same(a, b, what):
    for k in a:
        assert np.array_equal(a[k], b[k]), (what, k, np.abs(a[k] - b[k]).max())


# rows per tile from 1 to 128, last tiles with rows past the channel's end;
# direct sums below 24 nodes, every power of two; k_lbm, the row kernel, both
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("sizes", [
    [(2, 9), (3, 40), (4, 130), (5, 7), (10, 101), (14, 37), (22, 25), (23, 30)],
    [(8, 33), (16, 20), (32, 64), (32, 5)],
    [(64, 128), (128, 21), (256, 9)],
    [(64, 31), (4, 70), (32, 17), (256, 6), (8, 50)],
    [(10, 101)],
    [(64, 128)],
])
def test_step_equals_the_separate_launches(sizes, precision):
    a, b = start(sizes, precision), start(sizes + [(320, 8)], precision)
    for n in (5, 4):  # over a re-centring; steps that write no macroscopic fields among them
        a.step(n)
        b.step(n)
    for ch in range(len(sizes)):
        same(state(a, ch), state(b, ch), sizes[ch])
    assert np.array_equal(a.reductions(), b.reductions()[:-1])


def test_replayed_and_enqueued_steps_are_the_same():
    sizes = [(64, 40), (10, 33), (32, 20)]
    a, b = start(sizes, "fp32"), start(sizes, "fp32", use_graph=False)
    for n in (7, 1, 2, 70):  # the spectrum's two buffers in every order
        a.step(n)
        b.step(n)
    for ch in range(len(sizes)):
        same(state(a, ch), state(b, ch), sizes[ch])


# one tile per row: at and just past the limits of a card with 256 CUs, of the
# forward transforms in the launch and of the inverse ones
@pytest.mark.parametrize("nx,ny,precision,copies", [(256, 6, "fp32", (256, 257)), (256, 6, "fp64", (256, 257)),
                                                    (4, 64, "fp32", (3072, 3073)), (256, 6, "fp64", (128, 129))])
def test_both_sides_of_the_limit(nx, ny, precision, copies):
    got = []
    for n in copies:
        s = start([(nx, ny)] * n, precision)
        s.step(9)
        got.append((state(s, 0), state(s, n - 1)))
        s.close()
    same(got[0][0], got[1][0], "first")
    same(got[0][1], got[1][1], "last")
    same(got[0][0], got[0][1], "copies")
