"""Which kernels a context of given channels launches (CPU only: the library on a
HIP runtime without a device)."""
import json
import os

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


def cached(steps):
    """population planes that the collide-stream's last launch takes through the caches"""
    k = [n for n in steps if n.startswith(("k_lbm<", "k_lbm_rows<false"))]
    return int(k[-1].rstrip(">").split(", ")[-1])


# both lattices of a context in MB beside each
@pytest.mark.parametrize("sizes,precision,options,want", [
    ([(1024, 800)], "fp64", {}, 13),           # 354
    ([(1024, 1000)], "fp64", {}, 9),           # 442
    ([(1024, 1300)], "fp64", {}, 9),           # 575
    ([(1024, 2000)], "fp64", {}, 6),           # 885
    ([(2048, 1024)], "fp64", {}, 4),           # 906
    ([(4096, 640)], "fp64", {}, 4),            # 1132
    ([(1024, 514)], "fp64", {}, 27),           # 227
    ([(512, 256)], "fp64", {}, 0),             # 57
    ([(256, 256)] * 14, "fp64", {}, 13),       # 396
    ([(255, 256)] * 14, "fp64", {}, 9),        # 395: narrow channels keep to the smaller limit
    ([(4, 200)] * 700, "fp64", {}, 13),        # 242
    # the batches of test_gpu_lbm_cache.py, and the last narrow one below its limit
    *[([(1024, 64)] * n, "fp32", {}, w) for n, w in ((5, 0), (6, 27), (11, 27), (12, 18), (16, 18), (20, 13), (30, 9),
                                                     (45, 6), (70, 4), (100, 2), (160, 0))],
    *[([(1000, 64)] * n, "fp32", {}, w) for n, w in ((16, 27), (17, 18), (24, 13), (45, 6), (90, 2))],
    *[([(32, 256)] * n, "fp32", {}, w) for n, w in ((129, 27), (130, 0), (131, 0))],
    *[([(1000, 64)] * n, "fp32", {"compute_fp64": False}, w) for n, w in ((16, 27), (17, 18))],
    *[([(1024, 64)] * n, "fp64", {}, w) for n, w in ((2, 0), (3, 27), (8, 27), (9, 18), (12, 13), (35, 4))],
])
def test_cached_planes(so, sizes, precision, options, want):
    assert cached(fake_hip.launches(so, [(sizes, precision, options)])[0]) == want


@pytest.mark.parametrize("config,size", [("c1", (4096, 1024)), ("c4", (8192, 2048))])
def test_traffic_summaries_are_of_the_kernel_that_runs(so, config, size):
    with open(os.path.join(fake_hip.ROOT, "profiles", f"k_lbm_{config}_fp32_traffic.json")) as f:
        d = json.load(f)
    runs = {n for n in fake_hip.launches(so, [([size], "fp32", {})])[0] if n.startswith("k_lbm_rows<")}
    named = {k.split("ekpnp::", 1)[1].split("(")[0] for k in [d["kernel"], *d["kernel_by_tile_rows"].values()]}
    assert set(d["kernel_by_tile_rows"]) == set(d["bytes_per_launch_by_tile_rows"]) == {"0", "2", "4"}
    assert named == runs
