"""Host code of the library on a recording HIP runtime (tests/cpp/
recording_hip.hpp): launches, copies and waits in the order the calls make
them, and calls that fail.  Runs without a GPU; no kernel runs."""
import os
import subprocess

import pytest

from tests.cpp import build as cppbuild

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "raja_amd", "libraja_cdna4.so")


@pytest.fixture(scope="module")
def exe():
    return cppbuild.build_host_paths()


def run(exe, name, tmp_path):
    r = subprocess.run([exe, LIB, name], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, RAJA_CDNA4_TUNE_DIR=str(tmp_path)))
    print(r.stdout + r.stderr)
    assert r.returncode == 0, r.stdout + r.stderr


def test_plan_after_a_failed_upload(exe, tmp_path):
    """A batched call whose table upload fails reports it and leaves the plan
    as it was; the next call uploads the whole table."""
    run(exe, "failed_upload", tmp_path)


def test_lookback_gate_is_not_held_across_host_waits(exe, tmp_path):
    """While a sort waits for its decision, scans on other threads and streams
    go through; the gate's event covers the scatters, not the block sorts."""
    run(exe, "gate_across_waits", tmp_path)


def test_batched_sort_grows_its_scratch_first(exe, tmp_path):
    """A batched sort takes all its scratch before its first launch; one of
    short segments takes none, so a capture needs no growth."""
    run(exe, "batched_sort_scratch", tmp_path)


def test_allocation_free_scans_of_two_streams_are_ordered(exe, tmp_path):
    """They share one descriptor array, whatever their length."""
    run(exe, "noalloc_order", tmp_path)


def test_tuner_measures_and_takes_the_shapes_it_names(exe, tmp_path):
    """Each candidate runs its own tile (digit passes for sorts, whatever the
    keys), and a recorded full tile is the full tile."""
    run(exe, "tuner_shapes", tmp_path)


def test_refused_spans_count_their_digits_once(exe, tmp_path):
    """A span that the partition's sample refuses goes from the sample to one
    digit histogram and the passes, with no copy back to the host."""
    run(exe, "refused_spans", tmp_path)


def test_small_batch_of_short_sorts_is_one_launch(exe, tmp_path):
    run(exe, "batched_sort_launches", tmp_path)


def test_batched_sorts_of_two_threads_on_one_stream(exe, tmp_path):
    run(exe, "batched_sorts_of_two_threads", tmp_path)


def test_answers_that_come_late(exe, tmp_path):
    """A sort behind a long queue polls its answers and asks the stream now and
    then: "not ready" is no error, a missing answer is."""
    run(exe, "late_answers", tmp_path)
