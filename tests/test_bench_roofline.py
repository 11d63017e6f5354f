"""The bench's roofline record: kernels named by what their sizes select, and
counter traffic only where the counters ran the same launch."""
import json
import os
import re

import pytest

import bench
from tests.conftest import ROOT


def _table():
    with open(os.path.join(ROOT, "profiles", "hbm_traffic.json")) as fh:
        return json.load(fh)


def _prof(kind, nbytes, launches=4, ms=1.0):
    return {kind: dict(ms=ms, launches=launches, bytes=nbytes * launches, GBps=nbytes * launches / (ms * 1e-3) / 1e9)}


@pytest.mark.parametrize("kind,kernel", [("residual", "k_cell_residual"), ("spmv", "k_spmv")])
def test_traffic_is_of_the_same_launch(kind, kernel):
    ref = _table()[kernel]
    same = bench.roofline(_prof(kind, ref["algorithmic_bytes"]))
    assert same["kernel"] == kernel and same["traffic"] == ref["bytes_per_launch"]
    for factor in (0.02, 0.7, 1.5):   # another mesh, another layout
        r = bench.roofline(_prof(kind, factor * ref["algorithmic_bytes"]))
        assert r["traffic"] is None and r["traffic_source"] is None


def test_traffic_table_names_kernels_of_the_bench():
    names = set(bench.KERNEL_NAMES.values()) | {n for f in bench.FORM_KERNEL_NAMES.values() for n in f.values()}
    with open(os.path.join(ROOT, "profiles", "hbm_traffic_pmc.md")) as fh:
        source = fh.read()
    for kernel, row in _table().items():
        assert kernel in names
        assert f"| `{kernel}` | {row['what']} |" in source, kernel


def test_small_meshes_name_their_kernels():
    p = _prof("residual", 1e6)
    assert bench.roofline(p, bench.form_names(2, 40000))["kernel"] == "k_residual_faces"
    assert bench.roofline(p, bench.form_names(3, 2_000_000))["kernel"] == "k_cell_residual"
    assert bench.roofline(p, bench.form_names(3, 31104, 64))["kernel"] == "k_cell_residual"
    assert bench.form_names(3, 83000)["spmv"] == "k_spmv_slots"
    assert bench.form_names(3, 83000)["krylov"] == "k_mdot+k_orth_slots"
    assert "spmv" not in bench.form_names(3, 2_000_000)


def test_size_lines_are_the_library_s():
    def source(name):
        with open(os.path.join(ROOT, "bes_amd", "csrc", name)) as fh:
            return fh.read()

    m = re.search(r"line = c->common \? \(c->nd == 2 \? (\d+) : (\d+)\)", source("explicit.hip"))
    assert bench.SPLIT_PASS == {2: int(m[1]), 3: int(m[2])}
    imp = source("implicit.hip")
    m = re.search(r"slot_split\(const bes_ctx \*c\) \{ return [^}]*c->B == 1 \? 1u << (\d+)", imp)
    assert bench.SLOT_SPLIT == 1 << int(m[1])
    assert bench.ORTH_SLOTS == 64 * int(re.search(r"kSlotUnits = (\d+);", imp)[1])
