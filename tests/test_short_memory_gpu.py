"""The approximate cut runs in the memory of its edges and one level's forests: several
levels side by side are taken only where there is room for them."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent
LIB = ROOT / "comm-avoiding-cuts-cc_amd" / "lib"


def test_approx_cut_in_little_memory(orc, tmp_path):
    exe = tmp_path / "short_memory"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "short_memory.cpp"), "-o",
                    str(exe), f"-L{LIB}", "-lcac", "-ldl", f"-Wl,-rpath,{LIB}"], check=True, timeout=120)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=100).stdout
    print(out, flush=True)
    need, approx, trials = map(int, out.split())
    n = 100000
    e = np.stack([np.arange(n - 1), np.arange(1, n), np.full(n - 1, 64)], axis=1).astype(np.int64)
    assert (approx, trials) == orc.approx_cut(n, e, 0.95, 7)
    forest = 4 * n * orc.approx_trials(0.95)
    assert need <= 16 * n + forest * 9 // 8 + (1 << 18)  # a buffer is grown by an eighth
