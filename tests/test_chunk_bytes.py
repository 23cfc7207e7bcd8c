"""Chunks of square-root jobs stay within their byte budget (a served group's is what
it was admitted with), whatever the graphs weigh: packed edge lists take only the
room that 4-byte entries leave free, and a graph that runs in 64 bits is not packed."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "comm-avoiding-cuts-cc_amd"


@pytest.fixture(scope="module")
def chunks(tmp_path_factory):
    exe = tmp_path_factory.mktemp("chunk") / "chunk_bytes"
    subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O1", "--offload-arch=gfx950", f"-I{ROOT / 'include'}",
                    f"-I{PKG / 'csrc'}", str(ROOT / "tests" / "chunk_bytes.cpp"), "-o", str(exe), f"-L{PKG / 'lib'}",
                    "-lcac", f"-Wl,-rpath,{PKG / 'lib'}"], check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout
    return [(k, *map(int, r)) for k, *r in (line.split() for line in out.splitlines())]


@pytest.mark.parametrize("kind", ["light", "heavy", "unknown", "mixed"])
def test_chunks_hold_at_most_their_budget(chunks, kind):
    rows = [r[1:] for r in chunks if r[0] == kind]
    assert rows
    for shape, share, jobs, held, budget, packed in rows:
        # one job always runs, unpacked where the budget is short of it
        assert held <= budget or (jobs == 1 and packed == 0), (shape, share, jobs, held, budget, packed)


def test_heavy_graphs_are_not_packed(chunks):
    assert all(r[-1] == 0 for r in chunks if r[0] == "heavy")


@pytest.mark.parametrize("shape,jobs", [(0, 2), (1, 15), (2, 6), (3, 3), (4, 42), (5, 8)])
def test_admitted_groups_run_in_one_chunk(chunks, shape, jobs):
    """The packed lists of simple graphs fit beside 4-byte entries, so a served group
    keeps its trials together."""
    assert [r[3] for r in chunks if r[:3] == ("light", shape, 1)] == [jobs]
    assert [r[3] for r in chunks if r[:3] == ("heavy", shape, 1)] == [jobs]
    if shape != 5:  # of 70000 vertices: too large to pack
        assert all(r[-1] > 0 for r in chunks if r[:3] == ("light", shape, 1))
