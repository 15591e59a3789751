"""What the library asks the HIP runtime for (launch shapes, per-device set-up),
checked on the CPU: a program whose own stand-ins for the runtime's entry points
take the place of the real ones links the built library."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    from cuot_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    exe = str(tmp_path_factory.mktemp("launch") / "check")
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-o", exe, os.path.join(HERE, "launch_host_check.cpp"),
                    f"-L{libdir}", "-lcuot_amd", f"-Wl,-rpath,{libdir}", "-Wl,--allow-shlib-undefined"], check=True)

    def run(what, *args):
        r = subprocess.run([exe, what, *map(str, args)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 and f"{what} ok" in r.stdout, r.stdout + r.stderr
        return r.stdout

    return run


def test_every_device_is_set_up(check):
    check("devices")


def test_ggm_knob_without_a_split_is_the_rule(check):
    check("ggm_dfs")


def test_lpn_slices_need_rows(check):
    check("lpn_slices")


def test_sparse_product_of_many_words(check):
    check("sparse")


def test_tuner_can_choose_the_ggm_rule():
    from cuot_amd import tune

    for h in range(1, 17):
        space = [k["ggm_dfs"] for k in tune.ggm_space(h)]
        assert space[0] == 0
        assert space[1:] == [L for L in range(1, 7) if h - 10 <= L <= h - 8], h


# the tuner times no launch sequence twice, and its picture of the passes is the launches'
@pytest.mark.parametrize("n, settings", [(16384, 1), (40000, 1), (65537, 2), (200000, 3), (300001, 4), (1 << 24, 4),
                                         ((1 << 24) + 1, 16)])
def test_tuner_qc_space(check, n, settings):
    from cuot_amd import tune

    space = tune.qc_space(n)
    assert len(space) == settings
    assert dict(space[-1], qc_cols=0) == dict(qc_radix=7, qc_cols=0) or n > 1 << 24
    if n > 1 << 24:
        return
    plans = [tune.qc_passes(n, k["qc_radix"]) for k in space]
    assert len(set(plans)) == len(plans)
    for k, p in zip(space, plans):
        assert f"passes {2 * len(p) + 1}" in check("passes", n, k["qc_radix"])
