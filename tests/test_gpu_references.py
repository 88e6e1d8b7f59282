"""Storage references (FP32 storage) as a checkpoint holds them, against numpy:
the means of rho, c+, c- over each row, the rows' fluxes of them (none on
wall rows) and the means over each 64-node block, for rows of one wave and
wider, from the initial fields, after a step's re-centring and after a restart
of one channel."""
import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu

WIDTHS = (4, 10, 64, 65, 130, 255, 256, 257, 320, 1000)
EPS = 2.0 ** -53


def references(path, sizes):
    """per channel: rows [ny][8] FP64, blocks [ny][nb][4] FP32"""
    raw = open(path, "rb").read()
    off = 8 + 16 + 32 + 8 * len(sizes)
    out = []
    for nx, ny in sizes:
        nn, nb = nx * ny, (nx + 63) // 64
        off += 27 * nn * 4
        rows = np.frombuffer(raw, np.float64, 8 * ny, off).reshape(ny, 8)
        off += rows.nbytes
        blocks = np.frombuffer(raw, np.float32, 4 * nb * ny, off).reshape(ny, nb, 4)
        off += blocks.nbytes + 8 * (6 * nn + 6 * nx + nn)
        out.append((rows, blocks))
    assert off == len(raw)
    return out


def check(rows, blocks, rho, ux, cpos, cneg, what):
    ny, nx = rho.shape
    X = np.stack([rho, cpos, cneg], axis=-1)  # [ny][nx][3]
    # FP64 sums of nx terms in any order, and the division: (nx + 2) roundings of the sum of magnitudes
    tol = (nx + 2) * EPS * np.abs(X).mean(axis=1)
    assert np.all(np.abs(rows[:, :3] - X.mean(axis=1)) <= tol), what
    J = X * ux[:, :, None]
    tol = (nx + 3) * EPS * np.abs(J).mean(axis=1)
    want = J.mean(axis=1)
    want[[0, -1]] = 0.0
    assert np.all(np.abs(rows[:, 3:6] - want) <= tol), what
    assert not rows[[0, -1], 3:].any() and not rows[:, 6:].any() and not blocks[:, :, 3].any(), what
    for k in range(blocks.shape[1]):
        b = X[:, 64 * k:64 * k + 64]
        want = b.mean(axis=1)
        # rounded to FP32 once
        assert np.all(np.abs(blocks[:, k, :3] - want) <= 2.0 ** -24 * np.abs(want) + 66 * EPS * np.abs(b).mean(axis=1)), what


def test_references_are_the_means(tmp_path):
    sizes = [(nx, 5 + i) for i, nx in enumerate(WIDTHS)]
    sizes = sizes[5:] + sizes[:5]  # narrow rows behind wide ones
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, kappa_h=0.6) for nx, ny in sizes], precision="fp32")
    given = []
    for ch, (nx, ny) in enumerate(sizes):
        g = np.random.default_rng(nx).standard_normal((5, ny, nx))
        given.append((1 + 1e-2 * g[0], 1e-2 * g[1], 1e-2 * g[2], 1 + 0.3 * g[3], 1 + 0.3 * g[4]))
        s.set_fields(ch, *given[-1])
    s.init_equilibrium()
    path = str(tmp_path / "c.ckpt")
    s.save_checkpoint(path)
    for size, f, (rows, blocks) in zip(sizes, given, references(path, sizes)):
        check(rows, blocks, f[0], f[1], f[3], f[4], (size, "initial"))

    def now(what):
        s.rebase()
        s.save_checkpoint(path)
        for ch, (rows, blocks) in enumerate(references(path, sizes)):
            f = [s.get_field(ch, n) for n in ("rho", "ux", "cpos", "cneg")]
            check(rows, blocks, *f, (sizes[ch], what))

    s.step(20)
    now("stepped")
    for ch in (1, 5, 7):
        s.restart_channel(ch, ekpnp.COLD_NOISE, 3)
        s.save_checkpoint(path)
        f = [s.get_field(ch, n) for n in ("rho", "ux", "cpos", "cneg")]
        check(*references(path, sizes)[ch], *f, (sizes[ch], "restarted"))
    s.step(3)
    now("restarted and stepped")
