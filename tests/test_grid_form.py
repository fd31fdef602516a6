"""The blocks of a large mover's search meet and part (grid_form.hpp) so that the
one that ends last changes nothing another still reads, however late a block
without work is."""
import pathlib
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("grid") / "grid_form_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-o", str(exe), str(HERE / "grid_form_check.cpp")], check=True)
    return exe


@pytest.mark.parametrize("blocks,working", [(1, 0), (2, 1), (4, 1), (8, 8), (8, 0)])
@pytest.mark.parametrize("at_barrier", [0, 1])
def test_late_block_reads_the_search_it_belongs_to(check, blocks, working, at_barrier):
    out = subprocess.run([str(check), str(blocks), str(working), str(at_barrier)], capture_output=True, text=True,
                         check=True, timeout=60).stdout.split()
    gave_up, other_plan, ended = map(int, out)
    assert (gave_up, other_plan, ended) == (0, 0, 3)
