"""The kernel that bench.py's roofline names is the one that the density pass
launches first, on each side of the rules that pick it."""
import pytest


@pytest.mark.parametrize("n,over,name", [
    (1000000, {}, "k_density_lists<8, 0, false, 8>"),
    (20000, {}, "k_density_lists<16, 0, false, 4>"),
    (100000, {}, "k_density_lists<8, 0, false, 8>"),
    (1000000, {"density_stop": 1}, "k_density_lists<8, 1, false, 8>"),
    (100000, {"density_stop": 1}, "k_density_lists<8, 4, false, 8>"),
    (20000, {"density_stop": 1}, "k_density_lists<16, 2, false, 4>"),
    (20000, {"density_stop": 1, "small_n_lanes": 0}, "k_density_lists<8, 1, false, 8>"),
    (1000000, {"activity_rule": 1}, "k_density_lists<8, 0, true, 8>"),
    (20000, {"activity_rule": 1, "density_stop": 1}, "k_density_lists<8, 2, true, 8>"),
    (1000000, {"resolution_eta": 1.6}, "k_density_group<8, 0, 0, false, false>"),
    (1000000, {"density_lanes": 0}, "k_density"),
    (100000, {"density_flat": 1}, "k_density_group<32, 0, 1, false, false>"),
    (1000000, {"density_lanes": 16, "lane_split": 1}, "k_density_group<16, 1, 0, false, false>"),
])
def test_density_kernel_name(sph, n, over, name):
    import bench
    assert sph.SPH_ACTIVE_README == 1
    assert bench.density_kernel(sph, sph.default_params(**over), n) == name
