"""Dispatches whose blocks' sums the host adds (at most 512 blocks) against the
finishing kernel's sums of the same paths, bit for bit: a one-set
nt_exec_replay_many, which always runs that kernel. Path counts around a
block, around 128 blocks and around the 512-block limit, and around the limit
of 4,608 words of rows (384 blocks of a Heston tape's 12, 124 of a basket's
37); lanes left to the exception kernel; the reverse sweep; two outputs; more
channels than a wave has lanes; inputs bound before every call, once for
several, and changed between calls of both kinds."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import MERTON
from conftest import equity_tape, merton_call_tape, two_output_tape
from nablatensor_amd import workloads

pytestmark = pytest.mark.gpu

COUNTS = [1, 63, 64, 65, 255, 256, 257, 10_000, 127 * 256, 128 * 256, 128 * 256 + 1, 511 * 256 + 3, 512 * 256,
          512 * 256 + 1, 600 * 256]


@pytest.fixture(scope="module")
def rocm():
    from nablatensor_amd import rocm as r
    assert r.probe() > 0, "no gfx950 device"
    return r


def wide_tape(nt, n=70):
    """One step on each of n inputs: 72 channels."""
    def body(rec):
        x = [rec.input(f"x{i}", 1.0 + 0.01 * i) for i in range(n)]
        total = rec.constant(0.0)
        for v in x:
            total = total.add(v.mul(rec.randn()))
        rec.output(total.mul(total))
    return nt.AadRecorder.record(body).flat()


def tape_of(nt, name):
    if name == "merton":
        return merton_call_tape(nt, MERTON, steps=32).flat()
    if name == "two":
        return two_output_tape(nt).flat()
    if name == "wide":
        return wide_tape(nt)
    if name == "heston":
        return nt.record(nt.HestonModel.asian(nt.OptionTypeEnum.CALL, 1.0, 16), nt.HestonMarket.create(
            spot=100, strike=100, rate=0.03, v0=0.04, kappa=2.0, theta=0.04, xi=0.5, rho=-0.7)).flat()
    if name == "basket":
        fx = workloads.worst_of_inputs()
        return nt.record(nt.WorstOfBasket.call(fx["corr"], 100.0, 1.0, 16),
                         nt.WorstOfBasket.market([100.0] * 16, fx["sigma"], 0.03)).flat()
    steps = 1 if name == "european" else 16
    return equity_tape(nt, nt.Products.europeanCall() if steps == 1 else nt.Products.asianCall(),
                       nt.EquityMarket.atmOneYear(), steps).flat()


@pytest.mark.parametrize("name,precision,mode", [("european", "fp64", 0), ("asian", "fp64", 2), ("asian", "fp64", 1),
                                                 ("asian", "fp32", 0), ("two", "fp64", 0), ("wide", "fp64", 0)])
def test_small_dispatch_sums_equal_the_finishing_kernels(nt, rocm, name, precision, mode):
    flat = tape_of(nt, name)
    x0 = np.array(flat["recorded_inputs"])
    with rocm.Executable(flat, rocm.options(precision, mode=mode)) as x:
        for k, paths in enumerate(COUNTS):
            inputs = x0 * (1.0 + 0.01 * (k % 5))
            print(f"case {name} {precision} mode={mode} paths={paths} grid={x.grid(paths)}", flush=True)
            many, _ = x.replay_many(inputs[None, :], paths, 17, 5)
            x.set_inputs(inputs)
            for again in range(3):  # inputs read from host memory, then uploaded, then resident
                sums, tm = x.replay(paths, 17, 5)
                assert np.array_equal(sums, many[0]), (paths, again)
                assert 0.0 < tm["replay_ms"] <= tm["kernel_ms"] <= tm["wall_ms"]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name,blocks", [("heston", [128, 383, 384, 385]), ("basket", [123, 124, 125])])
def test_small_dispatches_around_the_limit_in_words(nt, rocm, name, blocks, precision):
    flat = tape_of(nt, name)
    x0 = np.array(flat["recorded_inputs"])
    with rocm.Executable(flat, rocm.options(precision)) as x:
        x.set_inputs(x0)
        for b in blocks:
            print(f"case {name} {precision} blocks={b}", flush=True)
            many, _ = x.replay_many(x0[None, :], b * 256 - 3, 17, 5)
            assert np.array_equal(x.replay(b * 256 - 3, 17, 5)[0], many[0]), b


def test_small_dispatch_with_exception_lanes(nt, rocm):
    """The Merton tape's saturated indicators flag paths: the rows say so and
    the exception kernel's sums are added as in the three-kernel dispatch."""
    flat = tape_of(nt, "merton")
    x0 = np.array(flat["recorded_inputs"])
    with rocm.Executable(flat, rocm.options("fp64")) as x:
        for paths in (257, 5_000, 40_000):
            print(f"case merton paths={paths} grid={x.grid(paths)}", flush=True)
            many, _ = x.replay_many(x0[None, :], paths, 3, 42)
            x.set_inputs(x0)
            for _ in range(2):
                sums, _ = x.replay(paths, 3, 42)
                assert np.isfinite(sums).all() and np.array_equal(sums, many[0]), paths


def test_inputs_changed_between_small_and_large_dispatches(nt, rocm):
    flat = tape_of(nt, "asian")
    x0 = np.array(flat["recorded_inputs"])
    sets = np.stack([x0, x0 * 1.05, x0 * 0.9])
    with rocm.Executable(flat, rocm.options("fp64")) as x:
        want = {n: x.replay_many(sets, n, 0, 9)[0] for n in (1_000, 400_000)}
        for m, n in [(0, 1_000), (1, 400_000), (2, 1_000), (2, 400_000), (0, 400_000), (1, 1_000), (1, 1_000)]:
            x.set_inputs(sets[m])
            assert np.array_equal(x.replay(n, 0, 9)[0], want[n][m]), (m, n)
            assert np.array_equal(x.replay(1_000, 0, 9)[0], want[1_000][m]), (m, n)


def test_small_dispatches_are_drained(nt, rocm):
    """A small dispatch returns without waiting for the stream, at most 255 times
    running; any other dispatch waits for it."""
    import ctypes as C
    undrained = rocm.lib().nt_testing_undrained
    undrained.argtypes, undrained.restype = [C.c_void_p], C.c_int32
    with rocm.Executable(tape_of(nt, "european"), rocm.options("fp64")) as x:
        seen = []
        print("case 600 small dispatches", flush=True)
        for k in range(600):
            x.replay(1_000, k * 1_000, 5)
            seen.append(undrained(x._h))
        # one more each time, zero after 255 or where the sums took longer than the host watches
        assert all(b == (a + 1 if a < 255 else 0) or b == 0 for a, b in zip(seen, seen[1:])) and max(seen) <= 255
        x.replay(600 * 256, 0, 5)  # the finishing kernel adds these
        assert undrained(x._h) == 0
