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


def test_transposed_matrix_vector_loads(ask):
    """10 * loads in flight + elements per load."""
    c64 = [(16, 65536), (2048, 2048), (3200, 3200), (3300, 3300), (65536, 4), (1 << 20, 16)]
    assert ask(*(("zgemv_t_form", 1, k, m) for k, m in c64)) == [41, 41, 41, 11, 41, 41]
    c32 = [(3, 1 << 20), (16, 65536), (127, 10), (128, 10), (255, 10), (256, 10), (2048, 2048), (3300, 3300)]
    assert ask(*(("zgemv_t_form", 0, k, m) for k, m in c32)) == [11, 11, 11, 12, 12, 42, 42, 12]


def test_tile_of_states_by_their_number(ask):
    c64 = [(10, 1), (18, 1), (21, 1), (12, 256), (12, 8192), (11, 1 << 20), (16, 255), (16, 256), (18, 31), (18, 32), (22, 1), (25, 1)]
    assert ask(*(("qubit_state_tbits", n, 1, c, 0) for n, c in c64)) == [10, 10, 10, 10, 12, 10, 10, 12, 10, 12, 10, 12]
    assert ask(*(("qubit_state_tbits", n, 1, c, 1) for n, c in [(22, 4), (22, 8), (24, 1), (24, 2)])) == [10, 12, 10, 12]
    c32 = [(3, 1), (10, 4096), (11, 1023), (11, 1024), (18, 4), (18, 8), (20, 1), (21, 1)]
    assert ask(*(("qubit_state_tbits", n, 0, c, 0) for n, c in c32)) == [10, 10, 10, 11, 10, 11, 10, 11]


def test_rows_of_a_site_group_tile(ask):
    """Long runs only while every one of 256 CUs has a tile, short ones only while
    the tiles stay one round."""
    c64 = [(16, 50, 1), (64, 90, 1), (2048, 4, 1), (4096, 4, 1), (16000, 16, 1), (1 << 20, 16, 1), (1 << 20, 2000, 1)]
    assert ask(*(("any_rows", 1, n1, P, n3, 256) for n1, P, n3 in c64)) == [2, 2, 8, 16, 32, 128, 8]
    c32 = [(16, 50, 1), (1000, 121, 4), (4096, 16, 1), (16000, 16, 1), (1 << 20, 16, 1), (40, 24, 508)]
    assert ask(*(("any_rows", 0, n1, P, n3, 256) for n1, P, n3 in c32)) == [2, 16, 16, 32, 256, 64]


def test_one_factor_by_a_mode_kernel(ask):
    q = [(1, 1 << 24, 1, 16), (1, 1 << 15, 1, 17), (1, 1 << 15, 5, 17), (1, 1 << 20, 1, 25), (1, (1 << 20) - 1, 1, 25), (1, 1 << 19, 2, 24), (1, 1 << 18, 5, 33),
         (1, (1 << 18) - 1, 5, 33), (0, 1 << 24, 1, 28), (0, 1 << 20, 1, 22), (0, 1 << 21, 1, 22), (0, 1 << 17, 5, 22),
         (0, 1 << 18, 5, 22), (0, 1 << 19, 2, 33), (1, 1 << 17, 16, 17), (1, 1 << 17, 26, 17), (0, 1 << 17, 26, 17),
         (1, 1 << 20, 40, 24), (1, 1 << 20, 64, 24), (0, 1 << 20, 64, 24), (0, 1 << 21, 64, 24), (1, 1 << 24, 600, 25)]
    assert ask(*(("one_factor_by_mode",) + x for x in q)) == [1, 1, 0, 0, 1, 0, 0, 1, 1, 1, 0, 0, 1, 0, 1, 0, 1, 1, 0, 1, 0, 1]


def test_groups_over_few_rows(ask):
    q = [(0, 54, 2, 2400, 3), (0, 54, 2, 1024, 3), (0, 54, 4, 2400, 3), (0, 1, 1, 2400, 3), (1, 54, 2, 2400, 3),
         (1, 54, 2, 2400, 2), (1, 54, 2, 1024, 2), (1, 1, 1, 2400, 2)]
    assert ask(*(("group_too_thin",) + x for x in q)) == [1, 0, 0, 0, 0, 1, 0, 0]
