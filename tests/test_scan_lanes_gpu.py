"""The scan with time across the lanes (csrc/scan_lanes.hip): chunk, lane and state edges, each
way of sharing the states among waves, time split into segments, growing states -- against the
fp64 oracle at test_scan_gpu's bars, and against the general path on the same values."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_close, config0_inputs, features_inputs
from test_scan_gpu import TOL, check, gpu_scan, oracle_scan

pytestmark = pytest.mark.gpu

# (batch, dim, dstate, seqlen): one vector of steps; ends inside a chunk, a lane and a vector; one
# whole chunk; a few elements past one; several state groups, the last one partial
EDGES = [(1, 8, 16, 8), (1, 1, 1, 9), (2, 13, 5, 511), (1, 24, 16, 512), (3, 40, 16, 513),
         (1, 16, 24, 1025), (2, 8, 64, 700), (1, 7, 33, 1543)]
# states shared by 4, 2 and 1 waves; two launches (segments), the first and last of one chunk or two
SHAPES = EDGES + [(1, 1100, 16, 530), (1, 2048, 16, 601), (2, 2100, 16, 520), (1, 16, 16, 9001),
                  (1, 256, 16, 2100), (1, 64, 16, 32769), (1, 512, 32, 1030)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_time_contiguous(oracle_lib, dev, shape, dtype):
    check(oracle_lib, dev, config0_inputs(*shape, seed=sum(shape)), f"lanes {shape}", dtype=dtype, softplus=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[1] % 8 == 0 and s[2] % 8 == 0], ids=str)
def test_channel_contiguous(oracle_lib, dev, shape, dtype):
    check(oracle_lib, dev, config0_inputs(*shape, seed=sum(shape)), f"lanes {shape}", dtype=dtype, softplus=True,
          layout="bld")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,first", [(8, 9), (1800, 513), (4104, 505)], ids=str)
def test_every_end_of_a_vector(oracle_lib, dev, dim, first, dtype):
    """Sequences that end after 1 .. 7 steps of a vector of 8, in one wave per channel and in two and
    four: the vector with the end in it is read 8 (or a lane's) steps before the end and moved."""
    for L in range(first, first + 7):
        check(oracle_lib, dev, config0_inputs(1, dim, 16 if L % 2 else 5, L, seed=L), f"end {dim} {L}", dtype=dtype,
              softplus=True)


@pytest.mark.parametrize("shape", [(1, 1024, 16, 520), (1, 1032, 16, 520), (1, 2056, 8, 513), (3, 1000, 24, 40)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_channel_contiguous_wave_counts(oracle_lib, dev, shape, dtype):
    """Either side of the channel counts up to which two waves share a channel of 16-bit rows (1024) and
    its states go in pairs (2048), more channels in fp32 (two waves always), one to three state groups."""
    check(oracle_lib, dev, config0_inputs(*shape, seed=sum(shape)), f"lanes {shape}", dtype=dtype, softplus=True,
          layout="bld")


@pytest.mark.parametrize("shape", [(1, 16, 16, 700), (1, 1032, 16, 700)], ids=str)
def test_channel_contiguous_slow_growth(oracle_lib, dev, shape):
    """A > 0 in 16 bits: chunks whose decays may not be multiplied up leave the pairs (states grow by
    e^(0.01 x 70) at most)."""
    inp = config0_inputs(*shape, seed=8)
    inp["delta"][:] = 0.1
    inp["A"] = np.broadcast_to(np.linspace(-20.0, 0.01, shape[2], dtype=np.float32), inp["A"].shape).copy()
    check(oracle_lib, dev, inp, f"lanes growth {shape}", dtype=torch.float16, layout="bld")


@pytest.mark.parametrize("use_D,use_z,softplus", [(False, False, False), (True, False, True), (False, True, False)])
@pytest.mark.parametrize("layout", ["bdl", "bld"])
def test_options(oracle_lib, dev, use_D, use_z, softplus, layout):
    inp = features_inputs(2, 24, 16, 1100, seed=3)
    if not softplus:
        inp["delta"] = np.abs(inp["delta"]) * 0.1
    check(oracle_lib, dev, inp, f"lanes D={use_D} z={use_z}", softplus=softplus, use_D=use_D, use_z=use_z, layout=layout)


def _general_path(inp, dev, dtype):
    """The same values through scan.hip: tensors of no unit stride take its element-wise loads."""
    return gpu_scan(inp, dev, dtype, softplus=True, layout="gather")


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(2, 40, 16, 777), (1, 2048, 8, 300), (1, 32, 16, 5000)], ids=str)
def test_matches_general_path(dev, shape, dtype, layout):
    inp = config0_inputs(*shape, seed=4)
    y, h = gpu_scan(inp, dev, dtype, softplus=True, layout=layout)
    yg, hg = _general_path(inp, dev, dtype)
    rt, at = TOL[dtype]
    assert_close(y, yg, rt, at, "y")
    assert_close(h, hg, 1e-5, 1e-5, "state")  # fp32 state either way


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("shape,quiet", [((1, 16, 16, 600), 400), ((1, 16, 16, 2000), 1850)], ids=str)
def test_growing_states(oracle_lib, dev, layout, shape, quiet):
    """A > 0: the product of decays over a chunk overflows fp32 (exp(0.3 x 600) and more) while the
    states, zero for the first `quiet` steps, stay finite (they grow for 200 steps at most)."""
    inp = config0_inputs(*shape, seed=6)
    inp["delta"][:] = 1.0
    inp["A"] = np.broadcast_to(np.linspace(-0.5, 0.3, shape[2], dtype=np.float32), inp["A"].shape).copy()
    inp["u"][..., :quiet] = 0.0
    y, h = gpu_scan(inp, dev, layout=layout)
    yo, ho = oracle_scan(oracle_lib, inp)
    # |y| reaches e^60 (relative bar 1e-4: ~200 fp32 steps at 2^-24 each, growing with the state)
    assert np.isfinite(y).all()
    assert_close(y, yo, 1e-4, 1e-5 * np.abs(yo).max(axis=(0, 1)).clip(1.0), "y")
    assert_close(h, ho, 1e-4, 1e-5 * np.abs(ho).max(), "state")


def test_nan_stays_behind(dev):
    """A NaN input reaches no earlier step and no other channel."""
    inp = config0_inputs(1, 16, 16, 1500, seed=7)
    ref, _ = gpu_scan(inp, dev, softplus=True)
    inp["u"][0, 3, 700] = np.nan
    for layout in ("bdl", "bld"):
        y, _ = gpu_scan(inp, dev, softplus=True, layout=layout)
        assert np.isnan(y[0, 3, 700:]).all()
        keep = np.ones_like(y, bool)
        keep[0, 3, 700:] = False
        assert np.isfinite(y[keep]).all()
        assert_close(y[keep], ref[keep], 1e-5, 1e-5, layout)


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(1, 16, 16, 500), (1, 1032, 16, 700), (1, 16, 16, 4096), (2, 2048, 16, 1500)], ids=str)
def test_infinite_input(oracle_lib, dev, shape, dtype, layout):
    """An infinite input makes every later state infinite, not NaN, however small the decays' products
    over many steps get (B and C positive, so no two infinities cancel)."""
    inp = config0_inputs(*shape, seed=9)
    for k in ("B", "C", "z"):
        inp[k] = np.abs(inp[k])
    inp["u"][0, 3, 20] = np.inf
    y, h = gpu_scan(inp, dev, dtype, softplus=True, layout=layout)
    sub = {k: v[:1, 3:4] if v.ndim == 3 and k in ("u", "delta", "z") else v[:1] if v.ndim == 3 else v[3:4]
           for k, v in inp.items()}
    yo, ho = oracle_scan(oracle_lib, sub, dtype, softplus=True)
    assert np.isinf(yo[0, 0, 20:]).all() and np.isinf(ho).all()
    assert np.array_equal(y[0, 3] == np.inf, yo[0, 0] == np.inf) and np.array_equal(h[0, 3], ho[0, 0])
    keep = np.ones(y.shape, bool)
    keep[0, 3] = False
    assert np.isfinite(y[keep]).all() and np.isfinite(y[0, 3, :20]).all()


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(1, 16, 16, 500), (1, 1032, 16, 700), (1, 16, 16, 4095)], ids=str)
def test_infinite_decay(oracle_lib, dev, shape, dtype, layout):
    """A = -inf: a state of its last input alone, also where the sequence ends inside a chunk and from
    segment to segment."""
    inp = config0_inputs(*shape, seed=10)
    inp["A"][:, 7] = inp["A"][:, 15] = -np.inf
    check(oracle_lib, dev, inp, f"A = -inf {shape}", dtype=dtype, softplus=True, layout=layout)
