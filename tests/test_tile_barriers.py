"""Waves of a workgroup may run different instances of the register tiles' step loops
and meet at barriers inside them, which tile_barrier (tile_kernel.hpp) allows on two
conditions.  Both are looked up in the sources: the choice of an instance depends on
nothing that differs between the lanes of a wave, and the loops' barriers are
tile_barrier, whose number follows from the number of steps alone."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "trotter-suzuki-mpi_amd", "csrc")
PER_LANE = {"threadIdx", "lane", "xl", "xs"}


def source(name):
    return re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())


def words(text):
    return set(re.findall(r"[A-Za-z_]\w*", text))


def body(text, head):
    """The braces that follow `head`."""
    i = text.index("{", text.index(head))
    depth = 0
    for j in range(i, len(text)):
        depth += {"{": 1, "}": -1}.get(text[j], 0)
        if depth == 0:
            return text[i:j + 1]
    raise AssertionError(head)


@pytest.mark.parametrize("name,flags", [("tile_kernel.hpp", {"eh", "ev"}), ("pair_tile_kernel.hpp", {"edge"}),
                                        ("adjoint_tile_kernel.hpp", {"edge"})])
def test_the_choice_is_uniform_in_a_wave(name, flags):
    text = source(name)
    assert "const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);" in text
    found = set()
    for flag, value in re.findall(r"const bool (eh|ev|edge) = ([^;]*);", text):
        found.add(flag)
        assert not PER_LANE & words(value), (flag, value)
    assert found == flags
    for var, value in re.findall(r"const int (X0|y_tile|y0|strip|seg|A) = ([^;]*);", text):
        assert not PER_LANE & words(value), (var, value)
    for cond in re.findall(r"if \(([^\n]*)\) \{?\s*\w*tile_steps<", text):
        assert not PER_LANE & words(cond), cond


@pytest.mark.parametrize("name,loop,calls", [("tile_kernel.hpp", "__device__ __forceinline__ void tile_steps(", 6),
                                             ("pair_tile_kernel.hpp", "void two_field_steps(", 4)])
def test_the_loops_meet_at_tile_barrier(name, loop, calls):
    steps = body(source(name), loop)
    assert "__syncthreads" not in steps and "s_barrier" not in steps
    assert steps.count("tile_barrier()") == 1                       # the vertical pass's
    passes = body(steps, "auto vpass = ")
    assert "tile_barrier()" in passes
    assert len(re.findall(r"\bvpass\(", steps.replace(passes, ""))) == calls
    # no pass under a condition on the instance's edges
    assert not {"EH", "EV"} & words(steps[steps.rindex("for (int st = 0"):])
