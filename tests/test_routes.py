"""Host rules of the dispatch (mirrorofmapgraph_amd/csrc/routes.h), compiled by the host
compiler and run without a GPU."""
import shutil
import subprocess

import pytest

from conftest import ROOT

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def run(tmp_path, body):
    """Compiles `body` as the main of a program over routes.h and returns what it prints."""
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text('#include <cstdio>\n#include "routes.h"\nusing namespace mg;\nint main() {\n' + body + "\n}\n")
    cmd = ["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", str(ROOT / "mirrorofmapgraph_amd" / "csrc"), str(src),
           "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return r.stdout


def test_pushed_and_pulled_batches_never_share_steps(tmp_path):
    # every width of a bucket around the number of every batch size, and the unbucketed one
    out = run(tmp_path, """
    long same = 0;
    for (int k = 1; k <= MG_BATCH_MAX; ++k) {
        const StepKey p = batch_pull_steps(k);
        for (long long d = 1; d < 40000; ++d) {
            const StepKey s = batch_sssp_steps(d);
            same += s.kind == p.kind && s.key == p.key;
        }
        const StepKey s = batch_sssp_steps(INT64_MAX / 4);
        same += s.kind == p.kind && s.key == p.key;
    }
    printf("%ld", same);
    """)
    assert out == "0"
