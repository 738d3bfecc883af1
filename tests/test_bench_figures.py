"""The bench line's rates are those of what ran: a batch whose states stay on the chip is held against the FP64 units,
which it cannot exceed, and not against a memory that it does not use."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_states_on_the_chip_are_held_against_the_fp64_units(bench):
    # 4e11 points and steps a second: more than the memory could carry
    r = bench.propagation_rate(4e11, 1.0, True)
    assert r["bound"] == "fp64" and r["unit"] == "TFLOP/s"
    assert r["frac"] == pytest.approx(4e11 * bench.FLOP_PER_PT_STEP / 1e12 / bench.FP64_PEAK_TFLOPS) and r["frac"] < 1


def test_streamed_states_are_held_against_the_memory(bench):
    r = bench.propagation_rate(1.7e11, 1.0, False)
    assert r["bound"] == "hbm" and r["achieved"] == pytest.approx(1.7e11 * 32 / 1e9) and r["frac"] < 1
