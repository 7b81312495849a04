"""The scan with time across the lanes (csrc/scan_lanes.hip): chunk, lane and state edges, each
way of sharing the states among waves, time split into segments, growing states -- against the
fp64 oracle at test_scan_gpu's bars, and against the general path on the same values."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_close, config0_inputs, features_inputs, scan_route
from test_scan_gpu import TOL, check, gpu_scan, oracle_scan

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def on_lanes(layout, dtype, shape, waves=None, segments=None):
    """The call runs on the lane scan, as many waves per channel and segments as the case is there for."""
    w, s = scan_route(layout, dtype, *shape)
    assert w > 0 and waves in (None, w) and segments in (None, s), (layout, dtype, shape, w, s)


# (batch, dim, dstate, seqlen), waves per channel, segments: one vector of steps; ends inside a chunk, a
# lane and a vector; one whole chunk; a few elements past one; several state groups, the last one
# partial; the states of a channel on 4, 2 and 1 waves, partial workgroups
EDGES = [((1, 8, 16, 8), 4, 1), ((1, 1, 1, 9), 4, 1), ((2, 13, 5, 511), 4, 1), ((1, 24, 16, 512), 4, 1),
         ((3, 40, 16, 513), 4, 1), ((1, 16, 24, 1025), 4, 1), ((2, 8, 64, 700), 4, 1), ((1, 7, 33, 1543), 4, 1),
         ((1, 512, 32, 1030), 4, 1), ((1, 1100, 16, 530), 4, 1), ((1, 2047, 16, 601), 2, 1), ((4, 1530, 16, 505), 1, 1),
         ((1, 2100, 24, 900), 2, 1), ((1, 5001, 33, 513), 1, 1)]
# two launches: segments of one chunk, the last one whole or not, on 4, 2 and 1 waves; of two and three chunks
SPLIT = [((1, 16, 16, 9001), 4, 18), ((1, 256, 16, 2000), 4, 4), ((1, 64, 16, 32700), 1, 64), ((1, 190, 16, 4096), 2, 8),
         ((1, 128, 16, 16384), 1, 32), ((1, 16, 16, 40000), 4, 40), ((1, 8, 5, 70000), 4, 46)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,waves,segments", EDGES + SPLIT, ids=str)
def test_time_contiguous(oracle_lib, dev, shape, waves, segments, dtype):
    on_lanes("bdl", dtype, shape, waves, segments)
    check(oracle_lib, dev, config0_inputs(*shape, seed=sum(shape)), f"lanes {shape}", dtype=dtype, softplus=True)


# By rows (multiples of 8): one and two waves per channel (16 bits; fp32 unsplit always two), states in
# pairs (16 bits, up to 256 workgroups) or not, one to eight state groups, segments of one to three chunks
ROWS = [((1, 8, 16, 8), 2, 1), ((1, 24, 16, 512), 2, 1), ((1, 16, 8, 300), 2, 1), ((1, 16, 24, 1025), 2, 1), ((2, 8, 64, 700), 2, 1),
        ((1, 512, 32, 1030), 2, 1), ((1, 1024, 16, 520), 2, 1), ((1, 1032, 16, 520), 1, 1), ((1, 2048, 16, 601), 1, 1),
        ((1, 2056, 8, 500), 1, 1), ((3, 1000, 24, 200), 1, 1), ((2, 2024, 16, 1000), 1, 1)]
ROWS_SPLIT = [((1, 16, 16, 9001), 2, 18), ((1, 256, 16, 2000), 2, 4), ((1, 64, 16, 32700), 1, 64), ((1, 128, 16, 16384), 1, 32),
              ((1, 16, 16, 40000), 2, 40), ((1, 8, 8, 70000), 2, 46)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,waves,segments", ROWS + ROWS_SPLIT, ids=str)
def test_channel_contiguous(oracle_lib, dev, shape, waves, segments, dtype):
    on_lanes("bld", dtype, shape, 2 if dtype == torch.float32 and segments == 1 else waves, segments)
    check(oracle_lib, dev, config0_inputs(*shape, seed=sum(shape)), f"lanes {shape}", dtype=dtype, softplus=True,
          layout="bld")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,dim,first", [(1, 8, 9), (1, 1800, 513), (4, 1530, 505)], ids=str)
def test_every_end_of_a_vector(oracle_lib, dev, batch, dim, first, dtype):
    """Sequences that end after 1 .. 7 steps of a vector of 8, in one wave per channel and in two and
    four: the vector with the end in it is read 8 (or a lane's) steps before the end and moved."""
    for L in range(first, first + 7):
        shape = (batch, dim, 16 if L % 2 else 5, L)
        on_lanes("bdl", dtype, shape)
        check(oracle_lib, dev, config0_inputs(*shape, seed=L), f"end {shape}", dtype=dtype, softplus=True)


@pytest.mark.parametrize("shape", [(1, 16, 16, 500), (1, 1032, 16, 700)], ids=str)
def test_channel_contiguous_slow_growth(oracle_lib, dev, shape):
    """A > 0 in 16 bits: chunks whose decays may not be multiplied up leave the pairs (states grow by
    e^(0.01 x 70) at most)."""
    on_lanes("bld", torch.float16, shape)
    inp = config0_inputs(*shape, seed=8)
    inp["delta"][:] = 0.1
    inp["A"] = np.broadcast_to(np.linspace(-20.0, 0.01, shape[2], dtype=np.float32), inp["A"].shape).copy()
    check(oracle_lib, dev, inp, f"lanes growth {shape}", dtype=torch.float16, layout="bld")


@pytest.mark.parametrize("use_D,use_z,softplus", [(False, False, False), (True, False, True), (False, True, False)])
@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("shape", [(2, 24, 16, 500), (2, 24, 16, 2100), (1, 1100, 24, 700), (1, 1104, 16, 700)], ids=str)
def test_options(oracle_lib, dev, use_D, use_z, softplus, layout, shape):
    if layout == "bld" and shape[1] % 8:
        shape = (shape[0], shape[1] // 8 * 8, *shape[2:])
    on_lanes(layout, torch.float32, shape)
    inp = features_inputs(*shape, seed=3)
    if not softplus:
        inp["delta"] = np.abs(inp["delta"]) * 0.1
    # y sums dstate terms of magnitude 2 to 4 that may cancel: the bar of an fp32 evaluation, as in
    # test_dstate_many_chains
    y, h = gpu_scan(inp, dev, torch.float32, softplus=softplus, use_D=use_D, use_z=use_z, layout=layout)
    yo, ho = oracle_scan(oracle_lib, inp, softplus=softplus, use_D=use_D, use_z=use_z)
    y32, _ = oracle_scan(oracle_lib, inp, softplus=softplus, use_D=use_D, use_z=use_z, precision="f32")
    assert_close(y, yo, 1e-5, max(1e-5, 2 * float(np.abs(y32.astype(np.float64) - yo).max())), "y")
    assert_close(h, ho, 1e-5, 1e-5, "state")


def _general_path(inp, dev, dtype):
    """The same values through scan.hip: tensors of no unit stride take its element-wise loads."""
    return gpu_scan(inp, dev, dtype, softplus=True, layout="gather")


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(2, 40, 16, 500), (1, 2048, 8, 300), (1, 32, 16, 5000), (1, 520, 32, 1500)], ids=str)
def test_matches_general_path(dev, shape, dtype, layout):
    on_lanes(layout, dtype, shape)
    inp = config0_inputs(*shape, seed=4)
    y, h = gpu_scan(inp, dev, dtype, softplus=True, layout=layout)
    yg, hg = _general_path(inp, dev, dtype)
    rt, at = TOL[dtype]
    assert_close(y, yg, rt, at, "y")
    assert_close(h, hg, 1e-5, 1e-5, "state")  # fp32 state either way


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("shape,quiet", [((1, 16, 16, 500), 300), ((1, 16, 16, 2000), 1850)], ids=str)
def test_growing_states(oracle_lib, dev, layout, shape, quiet):
    """A > 0: the product of decays over a chunk overflows fp32 (exp(0.3 x 500) and more) while the
    states, zero for the first `quiet` steps, stay finite (they grow for 200 steps at most)."""
    on_lanes(layout, torch.float32, shape)
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


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("kind", ["a rate above zero", "steps below zero", "both"])
@pytest.mark.parametrize("shape", [(1, 16, 16, 500), (1, 1032, 16, 700), (1, 16, 16, 4100)], ids=str)
def test_states_that_grow_a_little(oracle_lib, dev, layout, kind, shape):
    """Growth far below the products' range, beside decays far beyond it: rates of up to 0.002 (over 4100
    steps of 0.05, a factor of 1.5) and a few steps of about -0.01 (growth by e^(16 x 0.01) at most each)."""
    on_lanes(layout, torch.float32, shape)
    inp = config0_inputs(*shape, seed=11)
    rng = np.random.default_rng(11)
    inp["delta"][:] = rng.normal(0.05, 0.02, inp["delta"].shape) if kind != "a rate above zero" else 0.05
    if kind != "steps below zero":
        inp["A"] = np.broadcast_to(np.linspace(-16.0, 0.002, shape[2], dtype=np.float32), inp["A"].shape).copy()
    y, h = gpu_scan(inp, dev, layout=layout)
    yo, ho = oracle_scan(oracle_lib, inp)
    # y sums 16 terms that may cancel: the bar of an fp32 evaluation, as in test_dstate_many_chains
    y32, h32 = oracle_scan(oracle_lib, inp, precision="f32")
    e = lambda a, b: float(np.abs(a.astype(np.float64) - b).max())
    assert_close(y, yo, 1e-5, max(1e-5, 2 * e(y32, yo)), "y")
    assert_close(h, ho, 1e-5, max(1e-5, 2 * e(h32, ho)), "state")


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("L,t", [(500, 130), (2000, 700), (2000, 1999)])
def test_nan_stays_behind(dev, layout, L, t):
    """A NaN input reaches no earlier step and no other channel."""
    on_lanes(layout, torch.float32, (1, 16, 16, L))
    inp = config0_inputs(1, 16, 16, L, seed=7)
    ref, _ = gpu_scan(inp, dev, softplus=True, layout="bdl")
    inp["u"][0, 3, t] = np.nan
    y, _ = gpu_scan(inp, dev, softplus=True, layout=layout)
    assert np.isnan(y[0, 3, t:]).all()
    keep = np.ones_like(y, bool)
    keep[0, 3, t:] = False
    assert np.isfinite(y[keep]).all()
    assert_close(y[keep], ref[keep], 1e-5, 1e-5, layout)


@pytest.mark.parametrize("layout", ["bdl", "bld"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(1, 16, 16, 500), (1, 1032, 16, 700), (1, 16, 16, 4096), (2, 2048, 16, 1500)], ids=str)
def test_infinite_input(oracle_lib, dev, shape, dtype, layout):
    """An infinite input makes every later state infinite, not NaN, however small the decays' products
    over many steps get (B and C positive, so no two infinities cancel)."""
    on_lanes(layout, dtype, shape)
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
    on_lanes(layout, dtype, shape)
    inp = config0_inputs(*shape, seed=10)
    inp["A"][:, 7] = inp["A"][:, 15] = -np.inf
    check(oracle_lib, dev, inp, f"A = -inf {shape}", dtype=dtype, softplus=True, layout=layout)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout,shape", [("bld", (2, 64, 16, 500)), ("bld", (1, 1032, 16, 513)), ("bld", (2, 16, 16, 2050)),
                                          ("bdl", (2, 13, 16, 500)), ("bdl", (2, 16, 16, 2050)), ("bdl", (4, 1530, 16, 505))],
                         ids=str)
def test_views(dev, layout, shape, dtype):
    """Tensors at odd offsets and strides (no vector of theirs is aligned), B and C as columns of one
    buffer behind an odd count of others, B shared by the batch (stride 0): the bits of contiguous ones."""
    from mamba_metal_amd.selective_scan import selective_scan_into

    on_lanes(layout, dtype, shape)
    b, d, n, L = shape
    g = torch.Generator(device=dev)
    g.manual_seed(L)
    rows = layout == "bld"

    def wide(k, lead):  # k channels (or states) and what lies around them
        big = torch.full((b, L + 2, k + lead + 2) if rows else (b, k + lead + 2, L + 3), float("nan"), device=dev, dtype=dtype)
        return (big[:, 1:1 + L, lead:lead + k].transpose(1, 2) if rows else big[:, lead:lead + k, 1:1 + L])

    def fill(k, lead, std=1.0, mean=0.0):
        t = wide(k, lead)
        t.copy_((torch.randn((b, k, L), generator=g, device=dev) * std + mean).to(dtype))
        return t

    u, z, delta, C = fill(d, 1), fill(d, 3), fill(d, 5, 0.5, -1.0), fill(n, 63 + n)
    B = fill(n, 63)[:1].expand(b, n, L)
    A = -torch.rand((d, n), generator=g, device=dev) * 2 - 0.01
    D = torch.randn(d, generator=g, device=dev)

    def run(conv):
        y = wide(d, 7) if conv is None else conv(wide(d, 7))
        state = torch.full((b, d, n), float("nan"), device=dev)
        t = (lambda x: x) if conv is None else conv
        selective_scan_into(t(u), t(delta), A, t(B), t(C), y, D=D, z=t(z), delta_softplus=True, state_out=state)
        return y, state

    y, h = run(None)
    ref, href = run((lambda x: x.transpose(1, 2).contiguous().transpose(1, 2)) if rows else (lambda x: x.contiguous()))
    assert torch.isfinite(ref.float()).all() and torch.equal(y, ref) and torch.equal(h, href)
