"""A step's linear map of its draws, taken once on the draws' sums after the
loop: baskets of GBM spots read only by the payoff, whose step exponents take
correlated normals (rows of a literal matrix), compiled for the host and on the
device, held to the oracle per path. Cases: three to five assets (three is the smallest
basket that takes it), an odd number of draws per step (Box-Muller pairs split
over two steps), step counts around the fp32 sums' 16 steps, rows written as
differences, a draw that the step also reads by
itself, a row that another value of the step reads, uniforms among the draws,
and several markets."""
from __future__ import annotations

import re
import time

import numpy as np
import pytest

import emu
import oracle
from conftest import check_per_path, rel_err, tape_slots

OFFSET = 0x100000003


def basket(nt, assets, draws, steps, form):
    """max(sum of the spots - K, 0); asset i's normal is row i of a literal
    matrix times the step's draws, in the shape `form` names."""
    dt = 1.0 / steps
    g = np.random.Generator(np.random.PCG64(assets * 100 + draws))
    a = g.uniform(-0.6, 0.6, (assets, draws))

    def body(rec):
        spots = [rec.input(f"S{i}", 90.0 + 5.0 * i) for i in range(assets)]
        vols = [rec.input(f"v{i}", 0.15 + 0.05 * i) for i in range(assets)]
        rate = rec.input("r", 0.03)
        p = [rate.sub(v.mul(v).mul(0.5)).mul(dt) for v in vols]
        r = [v.mul(dt ** 0.5) for v in vols]
        state = list(spots)
        extra = rec.constant(0.0)
        for _ in range(steps):
            z = [rec.randu() if form == "uniform" and d == 0 else rec.randn() for d in range(draws)]
            if form.startswith("deep"):
                # the first draw through a chain of sums that read one value twice
                for _ in range(int(form[4:])):
                    z[0] = z[0].add(z[0]).mul(0.5)
            rows = []
            for i in range(assets):
                w = rec.constant(0.0)
                for d in range(draws):
                    if form == "signed" and d % 2:
                        w = w.sub(z[d].mul(-a[i, d]))
                    else:
                        w = w.add(z[d].mul(a[i, d]))
                rows.append(w)
            if form == "draw_read":
                extra = extra.add(z[0].mul(rate))
            if form == "row_read":
                extra = extra.add(rows[1].mul(rate))
            for i in range(assets):
                state[i] = state[i].mul(p[i].add(r[i].mul(rows[i])).exp())
        total = extra
        for s in state:
            total = total.add(s)
        rec.output(total.sub(90.0 * assets).max(rec.constant(0.0)))
    return nt.AadRecorder.record(body).flat()


CASES = [(3, 3, 16, "rows"), (3, 4, 17, "rows"), (4, 4, 15, "signed"), (5, 3, 40, "signed"), (4, 4, 33, "draw_read"),
         (4, 4, 20, "row_read"), (4, 3, 31, "uniform"), (5, 5, 48, "rows"), (4, 4, 18, "deep9")]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("assets,draws,steps,form", CASES)
def test_draw_sums_match_the_oracle(nt, assets, draws, steps, form, precision):
    from nablatensor_amd import rocm
    flat = basket(nt, assets, draws, steps, form)
    src = rocm.lower(flat, rocm.options(precision, mode=2))
    fast = src[:src.index("nt_replay_slow")]
    assert "real ds" in fast and "real ds" not in src[len(fast):]
    k = emu.EmulatedKernel(src, len(flat["input_node"]), tape_slots(src))
    _, v, g = k.run(flat["recorded_inputs"], 150, OFFSET, 42, grid=2, block=64)
    if precision == "fp64":
        check_per_path(v, g, flat, 150, OFFSET, 42, min_strict=0.9)
    else:
        # fp32 rounding of the draws (2^-24 |z| each) through 48 steps at most, on spots of about 100
        ov, og = oracle.replay_paths(flat, 150, OFFSET, 42, f32=True, threads=1)
        assert rel_err(v, ov) < 2e-4 and rel_err(g, og) < 2e-3


@pytest.mark.parametrize("basis", [1, 2])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("assets,draws,steps,form", CASES[1::2])
def test_values_after_the_loop_emitted_on_first_use(nt, assets, draws, steps, form, precision, basis):
    """Kernels asked for two waves compute each set-up and final value after the
    loop where it is first read (over inputs and over parameters): the values
    of the kernels that compute them all at once, bit for bit."""
    from nablatensor_amd import rocm
    flat = basket(nt, assets, draws, steps, form)
    n = len(flat["input_node"])
    rows = []
    for waves in (0, 2):
        src = rocm.lower(flat, rocm.options(precision, mode=2, basis=basis, waves=waves))
        _, v, g = emu.EmulatedKernel(src, n, tape_slots(src)).run(flat["recorded_inputs"], 150, OFFSET, 42, grid=2, block=64)
        rows.append((src, v, g))
    assert rows[0][0] != rows[1][0]
    assert np.array_equal(rows[0][1], rows[1][1]) and np.array_equal(rows[0][2], rows[1][2])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_only_the_forms_are_evaluated_on_the_sums(nt, precision):
    """After the loop the step's form is taken on the draws' sums; the exponent and
    the exponential it fed belong to one step and are not emitted on them."""
    from nablatensor_amd import rocm
    src = rocm.lower(basket(nt, 3, 3, 16, "rows"), rocm.options(precision, mode=2))
    fast = src[:src.index("nt_replay_slow")]
    after = fast[fast.index("real r0_", fast.index("}", fast.index("nt_normal_pair_sum"))):]
    on_sums = [line for line in after.splitlines() if line.strip().startswith("const real r0_")]
    assert len(on_sums) >= 6  # three sums, three rows or more
    assert not [line for line in on_sums if "exp" in line or "in0" in line or re.search(r"\bv\d", line)], on_sums


def test_a_deep_form_lowers_at_once(nt):
    """Sums that read one value twice, 44 deep: each position of the step is
    looked at once, where a walk along every way to the draw would take 2^44."""
    from nablatensor_amd import rocm
    for depth in (12, 22, 44):
        flat = basket(nt, 5, 5, 16, f"deep{depth}")
        started = time.monotonic()
        src = rocm.lower(flat, rocm.options("fp64"))
        assert time.monotonic() - started < 0.5, depth
        assert "real ds" in src[:src.index("nt_replay_slow")]


def test_draw_sums_shared_by_the_markets(nt):
    """Several markets share the sums of the draws and keep the single kernel's bits."""
    from nablatensor_amd import rocm
    flat = basket(nt, 4, 4, 20, "rows")
    x0 = np.array(flat["recorded_inputs"])
    sets = np.stack([x0, x0 * 1.02, x0 * 0.97])
    src = rocm.lower(flat, rocm.options("fp64", markets=3))
    assert src[:src.index("nt_replay_slow")].count("real ds0 =") == 1
    sums, v, g = emu.EmulatedKernel(src, len(x0), 0).run(sets, 120, OFFSET, 7, grid=2, block=64, markets=3)
    one = rocm.lower(flat, rocm.options("fp64", mode=2))
    for m in range(3):
        s1, v1, g1 = emu.EmulatedKernel(one, len(x0), 0).run(sets[m], 120, OFFSET, 7, grid=2, block=64)
        assert np.array_equal(v[m], v1) and np.array_equal(g[m], g1) and np.array_equal(sums[m], s1)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("assets,draws,steps,form", CASES + [(12, 12, 17, "rows"), (7, 6, 16, "signed")])
def test_draw_sums_on_the_device(nt, assets, draws, steps, form, precision):
    from nablatensor_amd import rocm
    flat = basket(nt, assets, draws, steps, form)
    print(f"case {form} assets={assets} draws={draws} steps={steps} {precision}", flush=True)
    with rocm.Executable(flat, rocm.options(precision, mode=2)) as x:
        assert "real ds" in x.source()
        for paths in (1, 257, 3_000):
            v, g = x.replay_paths(paths, OFFSET, 42)
            sums, _ = x.replay(paths, OFFSET, 42)
            if precision == "fp64":
                check_per_path(v, g, flat, paths, OFFSET, 42, min_strict=0.0 if paths == 1 else 0.9)
            else:  # the emulator test's bounds, on the same tapes
                ov, og = oracle.replay_paths(flat, paths, OFFSET, 42, f32=True, threads=1)
                assert rel_err(v, ov) < 2e-4 and rel_err(g, og) < 2e-3
            rows = np.concatenate([v.reshape(-1, 1), v.reshape(-1, 1) ** 2, g.reshape(paths, -1)], axis=1)
            # the sums of the same rows in another order: 3,000 roundings at most, 1.1e-16 each
            assert np.all(np.abs(sums - rows.sum(0)) <= 1e-12 * np.maximum(np.abs(rows).sum(0), 1e-300))
