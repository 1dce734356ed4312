"""bench.py's roofline block names the kernel that the library launches for a family, knows
only families that the library profiles, and quotes stored counters only for launches of as
many work items as they were taken on."""
import glob
import json
import os
import re

import pytest

import bench

CSRC = os.path.join(bench.ROOT, "isothermal_mhd_amd", "csrc")


def sources():
    return {os.path.basename(p): open(p).read() for p in glob.glob(os.path.join(CSRC, "*"))}


@pytest.mark.parametrize("family,esz,recon,kernel", [
    ("stage_pred", 4, "plm", "k_vl_stage"), ("stage_pred", 8, "plm", "k_vl_near"), ("stage_pred", 8, "ppm_char", "k_vl_near"),
    ("stage_corr_cfl", 4, "plm", "k_vl_stage"), ("stage_corr", 8, "plm", "k_vl_near"),
    ("stage_corr", 8, "ppm_prim", "k_vl_stage"), ("stage_corr_cfl", 4, "ppm_char", "k_vl_char"),
    ("stage_corr", 8, "ppm_char", "k_vl_char"), ("corner_corr", 8, "plm", "k_corner_z"), ("fill_ghosts", 4, "plm", "k_fill_ghost_band")])
def test_symbol_is_the_launched_kernel(family, esz, recon, kernel):
    assert bench.kernel_symbol(family, esz, recon) == kernel
    assert any(re.search(r"__global__[^;{]*\b" + kernel + r"\(", t) for t in sources().values())


def test_roe_plm_corrector_in_fp64():
    assert bench.kernel_symbol("stage_corr", 8, "plm", "roe") == "k_vl_stage"
    assert bench.kernel_symbol("stage_pred", 8, "plm", "roe") == "k_vl_near"


def test_families_are_profiled_by_the_library():
    api = sources()["imhd_api.cpp"]
    for family in list(bench.FAMILY_SYMBOL) + ["stage_pred", "stage_corr", "stage_corr_cfl"]:
        assert f'"{family}"' in api or f'"{family}_x"' in api, family


def test_stored_counters_need_the_same_launch(tmp_path, monkeypatch):
    os.makedirs(tmp_path / "profiles")
    for name, value in (("pmc_traffic.json", 8.0e9), ("sq_valu.json", {"valu_wave_instr": 1.0e9})):
        with open(tmp_path / "profiles" / name, "w") as f:
            json.dump({"_workload": "w", "_items": {"stage_corr": 1000}, "stage_corr": value}, f)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    same = bench.roofline({"stage_corr": (20.0, 2, 2000)}, 4, 900, 0, 12.0, "w")
    assert same["traffic"] == 8.0e9 and "measured" in same and "valu_issue" in same
    for other in (bench.roofline({"stage_corr": (20.0, 2, 1998)}, 4, 900, 0, 12.0, "w"),
                  bench.roofline({"stage_corr": (20.0, 2, 2000)}, 4, 900, 0, 12.0, "v")):
        assert other["traffic"] is None and "measured" not in other and "valu_issue" not in other
