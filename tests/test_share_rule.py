"""The share of a staging fill that crosses the link with its gather or scatter
launch: where the fill is cut, on the CPU (tests/native/share_rule.cpp), and that the
GPU tests of it reach the cuts and launches that they name."""

import os
import shutil
import subprocess

import pytest

import bench
from pegaflow_amd.transfer import plan_staged_fills
from tests.test_gpu_blocks import LARGE_SHARES, PAGE_SHARES, SHARE_SLOT, SHARES

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_cut_of_a_fill_leaves_its_tail(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = tmp_path / "share_rule"
    proc = subprocess.run(["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-Werror",
                           os.path.join(NATIVE, "share_rule.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "all ok\n", out.stdout


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = tmp_path_factory.mktemp("share_cases") / "share_cases"
    subprocess.run(["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-Werror",
                    os.path.join(NATIVE, "share_cases.cpp"), "-o", str(exe)], check=True)
    return lambda *args: subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, check=True).stdout


def _fills(planner, layers, slot):
    """What the planner makes of each fill of these layers, their host images laid end to end."""
    eligible, at = [], 0
    for n, frag, segments in layers:
        eligible.append(int(frag % 16 == 0 and at % 16 == 0))
        at += n * frag * segments
    units, n_fills = plan_staged_fills([n for n, _, _ in layers], [f * s for _, f, s in layers], slot)
    return [planner("fill", *(f"{u.count}:{layers[u.layer][1]}:{layers[u.layer][2]}:{eligible[u.layer]}"
                              for u in units if u.fill == fill)).strip() for fill in range(n_fills)]


CUTS = {
    "tail_of_v": "staged 1 launches 1 cut unit 0 segment 1",
    "tail_of_k_and_v": "staged 2 launches 1 cut unit 1 segment 0",
    "one_segment": "staged 1 launches 1 cut unit 0 segment 0",
    "whole_layers": "staged 1 launches 1 cut unit 0 segment 1",
    "whole_layer_to_the_fragment": "staged 1 launches 1 cut unit 0 segment 0",
    "whole_layer_alone": "staged 1 launches 1 cut units",
    "short_tiles": "staged 2 launches 1 cut unit 1 segment 1",
    "fragments_of_1k": "staged 1 launches 1 cut unit 0 segment 0",
    "fragment_larger_than_the_share": "staged 1 launches 1 cut none",
    "last_layer_off_the_grid": "staged 2 launches 1 cut none",
    "off_the_grid_before": "staged 2 launches 1 cut unit 1 segment 1",
    "units_inner": "staged 12 launches 1 cut unit 11 segment 1",
    "unlike_lengths_in_runs": "staged 12 launches 2 cut unit 11 segment 1",
    "rows_folded": "staged 2 launches 1 cut unit 1 segment 0",
    "most_rows_of_one_unit": "staged 1 launches 1 cut unit 0 segment 0",
    "too_many_rows": "staged 1 launches 1 cut unit 0 segment 0",  # the launch's grid has no planes left for it
}


@pytest.mark.parametrize("name", sorted(SHARES))
def test_cases_are_cut_as_they_are_named(planner, name):
    fills = _fills(planner, SHARES[name], 0)
    assert len(fills) == 1 and fills[0].split(" ", 2)[2] == CUTS[name]


def test_large_cases_share_in_the_fills_that_they_name(planner):
    fills = {name: _fills(planner, layers, SHARE_SLOT) for name, layers in LARGE_SHARES.items()}
    assert {k: [not f.endswith("none") for f in v] for k, v in fills.items()} == {
        "every_fill_shares": [True, True], "one_fill_cannot_share": [True, False], "runs_in_the_second_fill": [True, True]}
    assert " launches 2 " in fills["runs_in_the_second_fill"][1]
    # The stream of the copies is a question from 64 MiB a fill on.
    for name in ("every_fill_shares", "one_fill_cannot_share"):
        assert sum(n * f * s for n, f, s in LARGE_SHARES[name]) >= 2 * (64 << 20)


def test_page_cases_share_in_the_chunks_that_they_name(planner):
    pages = {}
    for name, (sizes, chunks) in PAGE_SHARES.items():
        page = sum(sizes)
        assert all(c == SHARE_SLOT // page for c in chunks[:-1]) and chunks[-1] <= SHARE_SLOT // page
        pages[name] = [planner("pages", c, page).strip() for c in chunks]
        if len(chunks) > 1:
            assert sum(chunks) * page >= len(chunks) * (64 << 20)
    assert pages == {"unlike_slices": ["pages 2"], "every_chunk_shares": ["pages 1"] * 2,
                     "last_chunk_cannot_share": ["pages 1", "pages 1", "pages 0"]}


def test_bytes_that_the_bench_charges_to_its_launches(planner):
    """bench.py leaves the share out of what a launch moves through HBM: the same shares
    as the planner's, for every fill of its workloads."""
    for name, w in bench.WORKLOADS.items():
        fills = bench.staging_fills(w, w["layers"], 512 << 20, 0)
        segments = 2 if w["split"] else 1
        assert sum(fills) == w["layers"] * w["n"] * segments * w["seg"]
        if w["page_first"]:
            page = w["layers"] * w["seg"]
            want = [int(planner("pages", b // page, page).split()[1]) * page for b in fills]
            shares = [bench.link_share(b, page) for b in fills]
        else:
            want = [int(planner("fill", f"{b // (segments * w['seg'])}:{w['seg']}:{segments}:1").split()[1]) for b in fills]
            shares = [bench.link_share(b, w["seg"]) for b in fills]
        assert shares == want, name
        assert bench.link_shares(fills, 1, 1) == [0] * len(fills)
    # The last chunk of 25 pages cannot share one: with the stream left to the call none does.
    w = bench.WORKLOADS["dsv3_mla"]
    page = w["layers"] * w["seg"]
    fills = bench.staging_fills(w, w["layers"], 512 << 20, 0)
    assert bench.link_share(fills[0], page) == 2 * page and fills[-1] == 25 * page
    assert bench.link_shares(fills, page, 0) == [0] * 18 and sum(bench.link_shares(fills, page, 2)) == 17 * 2 * page
