"""Reverse sweeps of rolled loops with the skeleton's own math: products and
sums of the body contract to fma, divisions are products with nt_recip, and a
body value's first adjoint contribution is stored instead of added to zero.
Against the oracle, on the CPU (the emulated kernel rounds products and sums
separately: the rules alone) and on the GPU (with the contraction), over steps
that use every operation, an operand used twice by one node and by several,
odd and even iteration counts and every checkpoint policy."""
from __future__ import annotations

import numpy as np
import pytest

import emu
import oracle
from conftest import check_per_path, rel_err, tape_slots

OFFSET = 0x100000003


def horner_tape(nt, coefficients, steps):
    """A step whose volatility is a clamped polynomial in the log spot."""
    def body(rec):
        spot = rec.input("spot", 100.0)
        theta = [rec.input(f"c{i}", 0.2 / (i + 1) ** 2 * (-1) ** i) for i in range(coefficients)]
        s, log0 = spot, spot.log()
        for _ in range(steps):
            level = s.log().sub(log0).max(-1.0).min(1.0)
            sigma = theta[-1]
            for c in reversed(theta[:-1]):
                sigma = sigma.mul(level).add(c)
            sigma = sigma.max(0.01)
            s = s.mul(sigma.mul(rec.randn()).mul(0.1).sub(sigma.mul(sigma).mul(0.005)).exp())
        rec.output(s.sub(95.0).max(0.0))
    return nt.AadRecorder.record(body).flat()


def every_op_tape(nt, steps):
    def body(rec):
        a, b, c = rec.input("a", 1.3), rec.input("b", 0.7), rec.input("c", 2.1)
        x, y = a, b
        for _ in range(steps):
            z = rec.randn()
            u = x.mul(x).add(c.mul(c)).add(1.0)      # one operand twice, an invariant's square
            w = y.div(u).add(u.log()).sub(z.mul(0.1).mul(b))
            h = w.neg().abs().max(y).min(c)
            x = x.mul(0.9).add(h.add(h).mul(0.05))   # a node added to itself
            y = c.div(w.mul(w).add(2.0)).sub(x.mul(0.1).neg().exp().mul(0.2))
        rec.output(x.mul(y).add(x))
    return nt.AadRecorder.record(body).flat()


CASES = [("horner", 2, 17, 1), ("horner", 3, 16, 2), ("horner", 24, 12, 1), ("horner", 5, 33, 3), ("every", 0, 13, 1),
         ("every", 0, 16, 2), ("every", 0, 21, 3)]


def tape_of(nt, kind, size, steps):
    return horner_tape(nt, size, steps) if kind == "horner" else every_op_tape(nt, steps)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind,size,steps,ckpt", CASES)
def test_reverse_rules_match_the_oracle(nt, kind, size, steps, ckpt, precision):
    from nablatensor_amd import rocm
    flat = tape_of(nt, kind, size, steps)
    src = rocm.lower(flat, rocm.options(precision, mode=1, checkpoint=ckpt))
    fast = src[:src.index("nt_replay_slow")]
    assert ("contract(fast)\n      const nt_u32 it0" in fast) == (precision == "fp64")
    assert "contract(fast)\n      const nt_u32 it0" not in src[len(fast):]
    k = emu.EmulatedKernel(src, len(flat["input_node"]), tape_slots(src))
    _, v, g = k.run(flat["recorded_inputs"], 150, OFFSET, 42, grid=2, block=64)
    if precision == "fp64":
        check_per_path(v, g, flat, 150, OFFSET, 42, min_strict=0.9)
    else:
        # fp32 rounding (2^-24 per operation) through 33 steps of at most 50 operations
        ov, og = oracle.replay_paths(flat, 150, OFFSET, 42, f32=True, threads=1)
        assert rel_err(v, ov) < 2e-4 and rel_err(g, og) < 2e-3


def test_quotients_of_far_apart_sizes(nt):
    """A divisor's adjoint where adjoint / divisor (1e-313) is subnormal and
    adjoint * quotient / divisor (1e-36) is not."""
    from nablatensor_amd import rocm

    def body(rec):
        x, s = rec.input("a", 1e23), rec.constant(0.0)
        for _ in range(16):
            s = s.add(rec.constant(1e300).div(x).mul(1e-290).mul(rec.randn()))
            x = x.mul(1.001)
        rec.output(s)

    flat = nt.AadRecorder.record(body).flat()
    src = rocm.lower(flat, rocm.options("fp64", mode=1))
    assert "nt_recip" in src
    _, v, g = emu.EmulatedKernel(src, 1, tape_slots(src)).run(flat["recorded_inputs"], 50, 0, 42, grid=1, block=64)
    ov, og = oracle.replay_paths(flat, 50, 0, 42, threads=1)
    # 16 steps of four roundings each, whose sum may cancel a few digits
    assert np.abs(v / ov - 1.0).max() < 1e-13 and np.abs(g / og - 1.0).max() < 1e-13


def test_variance_roots_keep_their_rounding(nt, tapes):
    """A tape with the square root of an active drawn value is not contracted."""
    from nablatensor_amd import rocm
    src = rocm.lower(tapes["C4"], rocm.options("fp64", mode=1))
    assert "contract(fast)" not in src


@pytest.mark.gpu
@pytest.mark.parametrize("kind,size,steps,ckpt", CASES)
def test_contracted_reverse_loops_match_the_oracle(nt, kind, size, steps, ckpt):
    from nablatensor_amd import rocm
    flat = tape_of(nt, kind, size, steps)
    print(f"case {kind} size={size} steps={steps} checkpoint={ckpt}", flush=True)
    with rocm.Executable(flat, rocm.options("fp64", mode=1, checkpoint=ckpt)) as x:
        for paths in (1, 257, 3_000):
            v, g = x.replay_paths(paths, OFFSET, 42)
            check_per_path(v, g, flat, paths, OFFSET, 42, min_strict=0.0 if paths == 1 else 0.9)
            sums, _ = x.replay(paths, OFFSET, 42)
            # the sums of the same per-path rows: 3,000 roundings at most, 1e-16 each
            assert abs(sums[0] - v.sum()) <= 1e-12 * max(1.0, np.abs(v).sum())
            assert np.all(np.abs(sums[2:] - g.reshape(paths, -1).sum(0)) <= 1e-12 * np.maximum(1.0, np.abs(g.reshape(paths, -1)).sum(0)))
