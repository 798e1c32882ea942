"""What a layered decoder's steps ask of the device, with the device calls stubbed (tests/layered_steps_check.cpp): launches, recordings and replays."""
import json
import os
import subprocess

import pytest

import fomunex_common
import gulidra_common
import natatar_common
import pimosun_common
from pimosun_common import layer, mixer

HERE = os.path.dirname(os.path.abspath(__file__))

# Pimosun so wide that products of one row and of 70 are cut into different numbers of parts
WIDE = dict(pimosun_common.config_even(), width=2048, layers=[layer(mixer(4, 64, 32, 64, 256, 128), 4096)])
DESIGNS = dict(pimosun=WIDE, gulidra=gulidra_common.config_even(), natatar=natatar_common.config_wide(),     # these two end with a mixer, whose product the head adds
               fomunex=fomunex_common.config_wide())
MANY_WORDS = dict(pimosun_common.config_one(), vocab=1 << 18)         # a row of logits is a megabyte


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    at = tmp_path_factory.mktemp("steps")
    exe = str(at / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "layered_steps_check.cpp"), "-o", exe, "-lpthread"],
                   check=True)

    def call(design, mode, steps, max_sequences=4, max_rows=256, errors=False):
        """steps: lists of (sequence, tokens, copies of the last place wanted), or a word of the driver"""
        path = at / (design + ".json")
        path.write_text(json.dumps(MANY_WORDS if design == "many_words" else DESIGNS[design]))
        words = ["steps", path, mode, max_sequences, max_rows]
        for s in steps:
            words += [s] if isinstance(s, str) else ["s", len(s), *(w for e in s for w in e)]
        out = subprocess.run([exe], input=" ".join(str(w) for w in words) + "\n", capture_output=True, text=True, check=True, timeout=60).stdout
        got = json.loads(out)
        assert errors or "error" not in got, got
        return got
    return call


@pytest.mark.parametrize("design", list(DESIGNS))
@pytest.mark.parametrize("singles", [[(0, 1, 300)], [(i, 1, 1) for i in range(300)]], ids=["places wanted more than once", "many sequences"])
def test_more_logits_than_one_head_takes(run, design, singles):
    """The head of rows past the first 256 reads the planes and streams of its own pass, whatever ran before."""
    steps = [[(300, 70, 1)]] + [singles] * 5 + [[(301, 70, 1)]] + [singles] * 2      # a prompt first, so that the second one replaces no buffer
    want, got = (run(design, mode, steps, 302, 320)["steps"] for mode in (0, 2))
    for w, g in zip(want, got):
        assert g["head"] == w["head"][-len(g["head"]):]


@pytest.mark.parametrize("design", list(DESIGNS))
def test_steps_are_recorded_beside_the_contexts_stream(run, design):
    """What another thread enqueues on the context's stream while a step is recorded has to run, so nothing of a recording goes there."""
    got = run(design, 2, [[(0, 1, 1), (1, 1, 1)]] * 6)
    assert not got["captured_shared"] and not any(s["recorders"] for s in got["steps"])      # that stream is made with the model: 3 ms in a process's first
    assert sum(s["recordings"] for s in got["steps"]) == 1 and sum(s["replays"] for s in got["steps"]) >= 3
    for s in got["steps"]:
        assert ("BRE" in s["order"]) == (s["recordings"] == 1) and s["order"].count("R") == s["recordings"], s["order"]


@pytest.mark.parametrize("design", list(DESIGNS))
def test_a_step_is_recorded_behind_its_launches(run, design):
    """The step that is recorded runs from its own launches, which come first, so that nothing waits for the recording; the next one is the first replay."""
    orders = [s["order"] for s in run(design, 2, [[(0, 1, 1)]] * 6)["steps"]]
    assert orders == ["L", "L", "LBRE", "G", "G", "G"]


@pytest.mark.parametrize("design", list(DESIGNS))
def test_a_step_whose_recording_fails_is_a_launched_one(run, design):
    orders = [s["order"] for s in run(design, 2, ["f"] + [[(0, 1, 1)]] * 5)["steps"]]
    assert orders == ["L", "L", "LBRX", "L", "L"]


def test_rows_that_fit_come_through_pinned_memory(run):
    """16 megabytes of logits have a place in host memory that kernels write, whatever rows all sequences together would take."""
    steps = [[(i, 1, 1) for i in range(n)] for n in (1, 16, 17, 1)]
    assert [s["blocking_copies"] for s in run("many_words", 2, steps, 40, 64)["steps"]] == [0, 0, 1, 0]


@pytest.mark.parametrize("mode", [0, 2])
def test_logits_without_a_place_are_an_error(run, mode):
    assert run("pimosun", mode, ["n", [(0, 3, 0)]])["steps"]
    assert "place" in run("pimosun", mode, ["n", [(0, 3, 0)], [(0, 1, 0), (1, 1, 1)]], errors=True)["error"]
