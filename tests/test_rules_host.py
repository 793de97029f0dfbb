"""The choices between kernels by sizes (csrc/qob_rules.h), compiled with the
host compiler: what each rule answers on both sides of its line."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "rules_check"
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", str(ROOT / "tests" / "rules_check.cpp"),
                        "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def f(*questions):
        text = "".join(" ".join(map(str, q)) + "\n" for q in questions)
        r = subprocess.run([str(exe)], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return [int(x) for x in r.stdout.split()]
    return f


def test_matrix_vector_in_one_launch_only_while_both_sides_are_short(ask):
    sizes = [(1, 1), (16, 1536), (1536, 1536), (1537, 16), (1536, 1537), (1, 1 << 20), (64, 65536), (1 << 20, 1)]
    assert ask(*(("zgemv_in_one", m, n) for m, n in sizes)) == [1, 1, 1, 0, 0, 0, 0, 0]
