"""What the zero fields of a tuning stand for (swpathtracer_amd/csrc/spt_tuning.h,
compiled here for the host): a call that asks for no number of wavefronts runs
one, is reported as three, and still runs one after the report is set again."""
import ctypes as C
import os
import subprocess

import pytest

import swpathtracer_amd._lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "spt_tuning.h"
extern "C" {
void t_reported(const spt_tuning* t, spt_tuning* r) { *r = spt::resolve_tuning(*t); }
void t_running(const spt_tuning* t, spt_tuning* r) { *r = spt::running_tuning(*t); }
void t_returned(const spt_tuning* t, spt_tuning* r) { *r = spt::returned_tuning(*t); }
}
"""


@pytest.fixture(scope="module")
def tuning(tmp_path_factory):
    d = tmp_path_factory.mktemp("tuning")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "swpathtracer_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    lib = C.CDLL(str(d / "t.so"))

    def call(name, fields):
        t, r = L.Tuning(), L.Tuning()
        for k, v in fields.items():
            setattr(t, k, v)
        getattr(lib, name)(C.byref(t), C.byref(r))
        return {f: getattr(r, f) for f, _ in L.Tuning._fields_}
    return call


def _shape(t):
    return t["wavefronts"], t["shade_blocks_per_cu"], t["refill_lanes"]


def test_a_default_call_runs_one_wavefront(tuning):
    assert _shape(tuning("t_running", {})) == (1, 128, 48)
    assert _shape(tuning("t_reported", {})) == (3, 64, 20)
    assert _shape(tuning("t_running", {"shade_blocks_per_cu": 16, "refill_lanes": 8})) == (1, 16, 8)


@pytest.mark.parametrize("k, shade, refill", [(1, 128, 48), (2, 64, 20), (3, 64, 20), (4, 64, 20)])
def test_asked_for_wavefronts_run(tuning, k, shade, refill):
    assert _shape(tuning("t_running", {"wavefronts": k})) == (k, shade, refill)
    assert tuning("t_running", {"wavefronts": k}) == tuning("t_reported", {"wavefronts": k})


@pytest.mark.parametrize("change", [{}, {"path_capacity": 1 << 20}, {"use_graph": 1}, {"extend_blocks_per_cu": 4},
                                    {"check_every": 8}, {"tile_pixels": 1024, "tile_samples": 4}])
def test_a_report_set_again_runs_what_ran(tuning, change):
    back = tuning("t_returned", {**tuning("t_reported", {}), **change})
    want = {**tuning("t_running", {}), **change}
    assert tuning("t_running", back) == want
    assert tuning("t_reported", back) == {**tuning("t_reported", {}), **change}


@pytest.mark.parametrize("t", [{"wavefronts": 3}, {"wavefronts": 3, "shade_blocks_per_cu": 64, "refill_lanes": 20},
                               {"wavefronts": 1}, {}])
def test_other_tunings_are_kept(tuning, t):
    whole = {f: t.get(f, 0) for f, _ in L.Tuning._fields_}
    assert tuning("t_returned", t) == whole
    changed = {**tuning("t_reported", {}), "wavefronts": 2}
    assert tuning("t_returned", changed) == changed
    changed = {**tuning("t_reported", {}), "shade_blocks_per_cu": 32}
    assert tuning("t_returned", changed) == changed
