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


def test_teams_grow_only_where_a_whole_team_was_outgrown(tmp_path):
    out = run(tmp_path, """
    {   // short of workgroups: one more try, and nothing to remember, however often it happens
        TeamsRule r;
        for (int call = 0; call < 100; ++call)
            if (!r.wanted() || !r.retry(TEAMS_SHORT, 16, 16, false) || r.retry(TEAMS_SHORT, 16, 16, true)) return 1;
        if (r.wgs || r.skip || r.wait) return 2;
    }
    {   // a vertex no team takes: no larger teams
        TeamsRule r;
        if (!r.wanted() || r.retry(TEAMS_HUB, 2, 16, false) || r.wgs) return 3;
    }
    {   // outgrown: doubled up to the largest, then the general route
        TeamsRule r;
        int wgs = 2, tries = 0;
        while (r.retry(TEAMS_OUTGROWN, wgs, 16, false)) wgs = r.wgs, ++tries;
        if (wgs != 16 || tries != 3 || r.wanted()) return 4;
    }
    // tries of a graph whose calls all fail, and the calls until one that would not fail is tried
    TeamsRule r;
    int tries = 0;
    for (int call = 0; call < 100000; ++call)
        if (r.wanted()) {
            ++tries;
            r.retry(TEAMS_HUB, 16, 16, false);
        }
    TeamsRule s;
    s.retry(TEAMS_HUB, 16, 16, false);
    int until = 1;
    while (!s.wanted()) ++until;
    s.succeeded();
    printf("%d %d %d", tries, until, s.wanted());
    """)
    assert out == "7 33 1"  # 32 + 128 + 512 + ... calls between them


def test_a_team_that_soon_hands_back_is_asked_for_less_often(tmp_path):
    # pauses of searches of 100,000 narrow levels whose teams run a given number of levels each: the
    # graph's first search, a later one, and one whose teams run long again after them
    out = run(tmp_path, """
    for (int levels : {0, 4, 31, 32, 1000}) {
        int start = TEAM_AFTER;
        auto search = [&](int levels) {
            long at = 0, pauses = 0;
            int after = start;
            for (; (at += after) < 100000; at += levels) {
                ++pauses;
                after = team_after_next(after, levels);
            }
            start = team_after_start(after);
            return pauses;
        };
        printf("%ld ", search(levels));
        printf("%ld ", search(levels));
        for (int i = 0; i < 10; ++i) search(1000);
        printf("%ld ", search(1000));
    }
    """)
    rows = [tuple(map(int, out.split()[3 * i: 3 * i + 3])) for i in range(5)]
    assert all(r[0] <= 7 and r[1] <= 2 for r in rows[:3])
    assert rows[3][:2] == (2500, 2500) and rows[4][0] <= 100
    assert all(r[2] == rows[4][0] for r in rows)


def test_pulled_batches_of_one_row_width_share_their_steps(tmp_path):
    out = run(tmp_path, """
    int changes = 0;
    for (int k = 1; k <= MG_BATCH_MAX; ++k) {
        const StepKey a = batch_pull_steps(k), b = batch_pull_steps(k > 1 ? k - 1 : 1);
        if (4 * pull_lanes(k) < k || 64 % pull_lanes(k) || a.kind >= NKINDS || a.kind < KIND_BATCH_PULL) return 1;
        changes += a.kind != b.kind;
        if (a.key != b.key || (a.kind != b.kind) != (pull_lanes(k) != pull_lanes(k > 1 ? k - 1 : 1))) return 2;
    }
    printf("%d", changes);
    """)
    assert out == "3"  # one slot a width, so calls of several widths do not capture in turn either


def test_a_lightly_loaded_server_does_not_hold_pagerank_queries_back(tmp_path):
    out = run(tmp_path, """
    for (long others : {0, 1, 10, 63, 64, 1000}) {
        const PprGate d = ppr_gate(0, 0, others), own = ppr_gate(5, 3, others);
        if (own.us != 5 || own.batch != 3) return 1;
        printf("%d/%d ", d.us, d.batch);
    }
    """)
    assert out.split() == 4 * ["20000/8"] + 2 * ["70000/16"]
