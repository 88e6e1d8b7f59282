"""Which kernels a context of given channels launches (CPU only: the library on a
HIP runtime without a device)."""
import pytest

import fake_hip


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


def fused(steps):
    """(collide-stream and forward transforms in one launch, the inverse ones too)"""
    k = [n for n in steps if n.startswith("k_lbm_fwd<")]
    return bool(k), any(n.endswith(", true>") for n in k)


def test_one_launch_limits_follow_the_compute_units(so):
    # 64x128: 32 work-groups; limits of 6 (in FP64 storage 3 with the inverse
    # transforms) a compute unit
    contexts = [([(64, 128)] * n, p, {}) for p in ("fp32", "fp64") for n in (3, 6, 12, 13)]
    got = {cus: [fused(s) for s in fake_hip.launches(so, contexts, cus)] for cus in (256, 64, 32)}
    assert got[256] == [(True, True)] * 8
    assert got[64] == [(True, True)] * 3 + [(False, False)] + [(True, True)] * 2 + [(True, False), (False, False)]
    assert got[32] == ([(True, True)] * 2 + [(False, False)] * 2 + [(True, True), (True, False)] + [(False, False)] * 2)


# work-groups of a channel, its copies on either side of a limit of a card with
# 256 CUs (1536, 2304 or 3072 work-groups), the launches there
@pytest.mark.parametrize("sizes,copies,want", [
    ([(16, 60)], (384, 385), [(True, True), (False, False)]),
    ([(16, 128)], (192, 193), [(True, True), (False, False)]),
    ([(8, 160), (16, 96)], (139, 140), [(True, True), (False, False)]),
    ([(32, 64)], (192, 193), [(True, True), (False, False)]),
    ([(6, 150)], (384, 385, 768, 769), [(True, True), (True, False), (True, False), (False, False)]),
    ([(7, 110)], (384, 385, 768, 769), [(True, True), (True, False), (True, False), (False, False)]),
    ([(10, 101)], (307, 308, 614, 615), [(True, True), (True, False), (True, False), (False, False)]),
    ([(18, 100), (12, 40)], (153, 154, 307, 308), [(True, True), (True, False), (True, False), (False, False)]),
    ([(8, 192)], (384, 385, 512, 513), [(True, True), (True, False), (True, False), (False, False)]),
    ([(2, 128)], (1537, 3072, 3073), [(True, True), (True, True), (False, False)]),
    ([(4, 64)], (1537, 3072, 3073), [(True, True), (True, True), (False, False)]),
    ([(12, 84)], (385, 768, 769), [(True, True), (True, True), (False, False)]),
    ([(12, 21), (20, 12)], (769, 1536, 1537), [(True, True), (True, True), (False, False)]),
])
def test_narrow_rows_leave_the_launch_where_it_loses(so, sizes, copies, want):
    got = fake_hip.launches(so, [(sizes * n, "fp32", {}) for n in copies])
    assert [fused(s) for s in got] == want
