"""The rules that choose launches from sizes (wsclean_amd/csrc/hws_rules.h),
compiled for the host."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wsclean_amd",
                    "csrc")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")

    def evaluate(expressions):
        src = d / "rules.cpp"
        lines = "".join(f'  std::printf("%d\\n", int({e}));\n' for e in expressions)
        src.write_text('#include <cstdio>\n#include "hws_rules.h"\nint main() {\n'
                       f'  using namespace hws;\n{lines}}}\n')
        subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(d / "rules"), str(src)],
                       check=True)
        out = subprocess.run([str(d / "rules")], check=True, capture_output=True, text=True)
        return [int(x) for x in out.stdout.split()]

    return evaluate


def test_degridding_launches_whole_rounds_of_resident_workgroups(rule):
    residents = list(range(0, 17))
    for r, per in zip(residents, rule([f"wholeRounds({r})" for r in residents])):
        assert per % max(r, 1) == 0 and per >= 5 and per - max(r, 1) < 5


def test_runtime_radix_transforms_run_fused_where_they_fill_the_chip(rule):
    sizes = [60, 300, 600, 840, 1260, 1500, 1600, 1680, 1920, 3072, 6144]
    want = [int(n >= 1600) for n in sizes]
    assert rule([f"fusedModelRows({n}, 300)" for n in sizes]) == [int(n >= 1400) for n in sizes]
    assert rule(["fusedModelRows(300, 1800)", "fusedModelRows(480, 3000)"]) == [0, 1]
    assert rule([f"fusedColumns({n}, 1)" for n in sizes]) == want
    assert rule(["fusedColumns(480, 3)", "fusedColumns(960, 3)", "fusedColumns(512, 6)",
                 "fusedColumns(1200, 2)"]) == [0, 1, 1, 0]
