"""The meeting of a resident solve's blocks (vfd_amd/csrc/resident.h), run on the host with a thread for each wave."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "vfd_amd", "csrc")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("resident") / "model")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I", CSRC,
                           os.path.join(HERE, "resident_model.cpp"), "-o", exe])

    def run(*args):
        p = subprocess.run([exe] + [str(a) for a in args], stdout=subprocess.PIPE, text=True, timeout=100)
        assert p.stdout.strip() == "ok", p.stdout
    return run


@pytest.mark.parametrize("blocks", [1, 2, 64, 65, 100])  # one polled word up to 64 blocks, a word per chunk beyond
def test_every_block_passes_every_barrier(model, blocks):
    model("all_pass", blocks)


@pytest.mark.parametrize("blocks", [2, 64, 65, 100])
def test_blocks_that_may_not_wait_all_leave(model, blocks):
    model("no_time", blocks)


@pytest.mark.parametrize("blocks", [3, 70])
def test_a_block_that_starts_after_the_others_gave_up_leaves_as_a_whole(model, blocks):
    model("late", blocks)


@pytest.mark.parametrize("blocks", [3, 64, 100])
def test_barriers_hold_past_the_arrivals_32_bits(model, blocks):
    model("wrap", blocks)


def test_a_store_that_nobody_waits_for_lands_before_the_words_are_cleared(model):
    model("slow_store")


@pytest.mark.parametrize("tiles,scenes,cus,group", [
    (0, 1, 256, 0), (1, 1, 256, 1), (256, 1, 256, 1), (257, 1, 256, 2), (512, 1, 256, 2), (513, 1, 256, 4),
    (1024, 1, 256, 4), (1025, 1, 256, 0), (1024, 1, 304, 4), (1025, 1, 304, 0), (64, 1, 64, 1), (257, 1, 64, 0),
    # a wave decides for at most twelve scenes, a solve for at most 64
    (48, 48, 256, 1), (49, 49, 256, 0), (128, 128, 256, 0), (256, 256, 256, 0), (300, 64, 256, 2), (300, 65, 256, 0),
    (1000, 64, 256, 4), (1000, 250, 256, 0)])
def test_which_simulations_have_resident_solves(model, tiles, scenes, cus, group):
    model("rule", tiles, scenes, cus, group)


def test_simulations_that_abort_each_other_lose_little_time(model):
    model("pause")


def test_groups_of_recorded_steps_fit_the_chip(model):
    model("recorded")
