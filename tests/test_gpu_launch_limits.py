"""The coupled step on both sides of the limits of the one-launch
collide-stream for rows of 6, 8 and 16 nodes: the same bits."""
import pytest

from test_gpu_lbm_fwd import same, start, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,copies", [(16, 60, (384, 385)), (6, 150, (384, 385)), (8, 192, (384, 385))])
def test_both_sides_of_the_narrow_limits(nx, ny, copies):
    got = []
    for n in copies:
        s = start([(nx, ny)] * n, "fp32")
        s.step(9)
        got.append((state(s, 0), state(s, n - 1)))
        s.close()
    same(got[0][0], got[1][0], "first")
    same(got[0][1], got[1][1], "last")
    same(got[0][0], got[0][1], "copies")
