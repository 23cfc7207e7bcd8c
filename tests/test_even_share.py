"""Chunks of large square-root trials take their even share of the room: no more
chunks than the full room would give, none of them far above the mean."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "comm-avoiding-cuts-cc_amd"


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    exe = tmp_path_factory.mktemp("share") / "even_share"
    subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O1", "--offload-arch=gfx950", f"-I{ROOT / 'include'}",
                    f"-I{PKG / 'csrc'}", str(ROOT / "tests" / "even_share.cpp"), "-o", str(exe), f"-L{PKG / 'lib'}",
                    "-lcac", f"-Wl,-rpath,{PKG / 'lib'}"], check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_no_more_chunks_than_the_full_room_gives(rows, kind):
    mine = [r for r in rows if r[1] == kind]
    assert mine
    for count, _, room, chunks, largest, greedy, mean, most in mine:
        assert chunks <= greedy, (count, room, chunks, greedy)
        assert largest <= max(room, most), (count, room, largest)
        if room >= most:
            assert largest <= mean + most, (count, room, largest, mean, most)


def test_sixteen_trials_run_as_eight_and_eight(rows):
    assert [r[3:5] for r in rows if r[:3] == (16, 0, 14000)] == [(2, 8000)]
