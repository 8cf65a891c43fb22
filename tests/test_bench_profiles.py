"""Which committed profile bench.py quotes, without a GPU: only one taken on the kernels that the sources hold, under the
configuration that ran, with the kernel variants named that 0 stands for."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


CONFIG = dict(tile_w=8, xcd_remap=1, packet=1, pair_limit=64, persistent=1, lane_min_triangles=300, sort_rays=1, render_blocks=0,
              rgb_blocks=0, ray_blocks=0, backward_blocks=0, rgb_two_pass=1)


def test_a_profile_of_other_kernels_is_not_this_ones(bench):
    built = bench._built(CONFIG, 130, 2000, 64)
    entry = dict(trace_config=dict(built), hbm_bytes_per_launch=5, kernels={"render_kernel_sq": {"valu_busy": 0.9}})
    summary = dict(trace_config=dict(built, render_blocks=7), hbm_bytes_per_launch=4, variants=[entry],
                   kernel_digest=bench.kernel_digest())
    assert bench._profiled(summary, "render", built) == (5, True, entry)
    assert bench._profiled(summary, "render", dict(built, render_blocks=7))[:2] == (4, True)
    assert bench._profiled(summary, "render", dict(built, render_blocks=5))[:2] == (4, False)
    for digest in ("0" * 16, None):
        assert bench._profiled(dict(summary, kernel_digest=digest), "render", built)[:2] == (5, False)


def test_the_digest_is_of_the_code(bench):
    code = "int f(int a) { return a / 2; }  // halves\n"
    assert bench._code_digest(code) == bench._code_digest("/* of\n two lines */\nint f(int a)\n{ return a/2; }")
    assert bench._code_digest(code) != bench._code_digest(code.replace("2", "3"))
    assert bench.kernel_digest() == bench.kernel_digest() and len(bench.kernel_digest()) == 16


def test_the_variants_that_zero_stands_for(bench):
    named = bench._built(CONFIG, 130, 2000, 64)
    assert (named["render_blocks"], named["rgb_blocks"], named["backward_blocks"]) == (8, 6, 6)
    assert bench._built(CONFIG, 8, 2000, 80)["rgb_blocks"] == 5 and bench._built(CONFIG, 8, 2000, 80)["backward_blocks"] == 5
    assert bench._built(dict(CONFIG, persistent=0), 130, 2000, 64)["render_blocks"] == 7
    assert bench._built(dict(CONFIG, lane_min_triangles=1 << 30), 130, 2000, 64)["render_blocks"] == 7
    asked = dict(CONFIG, render_blocks=5, rgb_blocks=7, backward_blocks=4)
    assert bench._built(asked, 130, 2000, 64) == asked


def test_committed_profiles_say_which_kernels_they_are_of(bench):
    for name in os.listdir(os.path.join(ROOT, "profiles")):
        if name.endswith("_traffic.json"):
            assert len(bench._profile_summary(name).get("kernel_digest", "")) == 16, name
