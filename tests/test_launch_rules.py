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
