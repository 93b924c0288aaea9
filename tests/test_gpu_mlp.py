"""GPU tests of the fused decode MLP (qnn_mlp.hip).

TrySwiGLUVector followed by the Int4Linear that reads its output runs as one
launch.  The work items, their order and the slice order are those
of the two per-op launches, so h and y must be bit-identical to the per-op path
(QNN_FUSE_MLP=0), and within 1e-3 normwise of the reference CPU path
(QwenHybrid.CPU.pas:238-248).  A recorded SwiGLU that is not followed by its
down projection is launched on its own by the next call.
"""
import numpy as np
import pytest

import oracle
from tests.conftest import normwise_rel_err, rand_int4

pytestmark = pytest.mark.gpu


def mlp(ctx, hip, layers, x0, hidden, inter):
    x = ctx.UploadRaw(x0)
    h = ctx.NewTensor(inter)
    ys = [ctx.NewTensor(hidden), ctx.NewTensor(hidden)]
    hs, outs, src = [], [], x
    for i, (g, u, d) in enumerate(layers):
        assert ctx.TrySwiGLUVector(h, src, g, u, hidden, inter)
        y = ys[i & 1]
        ctx.Int4Linear(y, h, d, 1, inter, hidden)
        hs.append(ctx.Download(h))
        outs.append(ctx.Download(y))
        src = y
    for t in [x, h] + ys:
        ctx.Recycle(t)
    return hs, outs


# inter 2048 and 1024: down K-ranges of 64 and 32 steps, which the per-op
# one-token matvec runs as 16- and 8-wave workgroups while the fused kernel
# keeps its four-wave slices.
@pytest.mark.parametrize("hidden,inter,nl", [(2560, 9728, 3), (1024, 3072, 2), (2048, 768, 2), (512, 1536, 1),
                                             (1024, 2048, 2), (768, 1024, 1), (1024, 1000, 1), (768, 996, 1)])
def test_fused_equals_per_op(ctx, rng, tune, hidden, inter, nl):
    from quicknn_amd import hip

    layers = [(hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)),
               hip.MemoryBlock.int4(rand_int4(rng, hidden, inter))) for _ in range(nl)]
    x0 = rng.standard_normal(hidden).astype(np.float32)
    before = ctx.status().mlp_fused
    h_f, y_f = mlp(ctx, hip, layers, x0, hidden, inter)
    fused = ctx.status().mlp_fused - before
    tune("QNN_FUSE_MLP", "0")
    h_p, y_p = mlp(ctx, hip, layers, x0, hidden, inter)
    assert ctx.status().mlp_fused - before == fused  # nothing fused with the switch off
    for i in range(nl):
        assert np.array_equal(h_f[i], h_p[i]), ("h", i)
        assert np.array_equal(y_f[i], y_p[i]), ("y", i)
    g, u, d = layers[0]
    want = oracle.cpu_mlp(g.data, u.data, d.data, oracle.ENC_INT4, x0, hidden, inter)[0]
    assert normwise_rel_err(y_f[0], want) < 1e-3
    if (hidden, inter) in ((2560, 9728), (1024, 2048), (768, 1024)):
        assert fused == nl  # the benchmark shape and the short down K-ranges run fused
    if (hidden, inter) in ((1024, 1000), (768, 996)):
        assert fused == nl  # h rows that end inside a down group


def test_recorded_swiglu_settles_on_other_calls(ctx, rng):
    """The recorded SwiGLU is launched before any other call: Download of h,
    an Int4Linear on another input, a second SwiGLU, events."""
    from quicknn_amd import hip

    hidden, inter = 1024, 3072
    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    d = hip.MemoryBlock.int4(rand_int4(rng, hidden, inter))
    x0 = rng.standard_normal(hidden).astype(np.float32)
    x, h, y = ctx.UploadRaw(x0), ctx.NewTensor(inter), ctx.NewTensor(hidden)
    other = ctx.UploadRaw(rng.standard_normal(inter).astype(np.float32))
    ref_h = None
    for case in ("download", "other_input", "second_swiglu", "event"):
        ctx.Kernel(hip.GO_FILL, inter, h, None, None, None, [0])
        assert ctx.TrySwiGLUVector(h, x, g, u, hidden, inter)
        if case == "download":
            ref_h = ctx.Download(h)
            got = ref_h
        elif case == "other_input":
            ctx.Int4Linear(y, other, d, 1, inter, hidden)  # not h: no fusion
            got = ctx.Download(h)
            yo = ctx.Download(y)
            want_o = oracle.cpu_linear(d.data, oracle.ENC_INT4, ctx.Download(other), inter, hidden)
            assert normwise_rel_err(yo, want_o) < 1e-3
        elif case == "second_swiglu":
            h2 = ctx.NewTensor(inter)
            assert ctx.TrySwiGLUVector(h2, x, g, u, hidden, inter)
            got = ctx.Download(h)
            assert np.array_equal(ctx.Download(h2), ref_h)
            ctx.Recycle(h2)
        else:
            ctx.EventRecord(20)
            ctx.EventRecord(21)
            ctx.EventElapsedMs(20, 21)
            got = ctx.Download(h)
        assert np.array_equal(got, ref_h), case
    gg = oracle.int4_dequant(g.data, hidden).astype(np.float64) @ x0.astype(np.float64)
    uu = oracle.int4_dequant(u.data, hidden).astype(np.float64) @ x0.astype(np.float64)
    from scipy.special import expit
    assert normwise_rel_err(ref_h, gg * expit(gg) * uu) < 1e-3
    for t in (x, h, y, other):
        ctx.Recycle(t)


def test_fused_error_in_down_still_runs_swiglu(ctx, rng):
    """A failing Int4Linear (bad weight shape) raises, and the recorded SwiGLU still runs."""
    from quicknn_amd import hip

    hidden, inter = 512, 1536
    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    bad = hip.MemoryBlock.int4(rand_int4(rng, hidden, inter + 32))  # wrong row width
    x, h, y = ctx.UploadRaw(rng.standard_normal(hidden).astype(np.float32)), ctx.NewTensor(inter), ctx.NewTensor(hidden)
    ctx.Kernel(hip.GO_FILL, inter, h, None, None, None, [0])
    assert ctx.TrySwiGLUVector(h, x, g, u, hidden, inter)
    with pytest.raises(hip.EArgumentException):
        ctx.Int4Linear(y, h, bad, 1, inter, hidden)
    assert np.any(ctx.Download(h) != 0)
    for t in (x, h, y):
        ctx.Recycle(t)


def batch_mlp(ctx, hip, g, u, d, x0, rows, hidden, inter):
    """The engine's multi-row MLP: Int4Linear gate and up, GO_SWIGLU, Int4Linear down."""
    x = ctx.UploadRaw(x0)
    g8, u8, hh, y = ctx.NewTensor(rows * inter), ctx.NewTensor(rows * inter), ctx.NewTensor(rows * inter), ctx.NewTensor(rows * hidden)
    ctx.Int4Linear(g8, x, g, rows, hidden, inter)
    ctx.Int4Linear(u8, x, u, rows, hidden, inter)
    ctx.Kernel(hip.GO_SWIGLU, rows * inter, hh, g8, u8, None, [inter, 0])
    ctx.Int4Linear(y, hh, d, rows, inter, hidden)
    out = [ctx.Download(t).view(np.uint32).copy() for t in (g8, u8, hh, y)]
    for t in (x, g8, u8, hh, y):
        ctx.Recycle(t)
    return out


@pytest.mark.parametrize("rows,hidden,inter", [(8, 2560, 9728), (3, 1024, 3072), (20, 512, 1536), (5, 2048, 768)])
def test_multi_row_gate_up_glu_one_launch(ctx, rng, tune, rows, hidden, inter):
    """Int4Linear gate + up on the same rows followed by GO_SWIGLU of their outputs run as one
    gate/up SwiGLU launch (qnn_status.glu_fused) that still writes both outputs; every output is
    bit-identical to the three separate operations (QNN_FUSE_MLP=0)."""
    from quicknn_amd import hip

    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    d = hip.MemoryBlock.int4(rand_int4(rng, hidden, inter))
    x0 = (rng.standard_normal((rows, hidden)) * 0.5).astype(np.float32)
    n0 = ctx.status().glu_fused
    fused = batch_mlp(ctx, hip, g, u, d, x0, rows, hidden, inter)
    n1 = ctx.status().glu_fused
    tune("QNN_FUSE_MLP", "0")
    sep = batch_mlp(ctx, hip, g, u, d, x0, rows, hidden, inter)
    assert ctx.status().glu_fused == n1
    for a, b, nm in zip(fused, sep, ("gate", "up", "glu", "down")):
        assert np.array_equal(a, b), nm
    # the pair runs fused where the gate/up and single-matrix plans agree (they do at the
    # benchmark shape); elsewhere the three run separately
    if (rows, hidden, inter) == (8, 2560, 9728):
        assert n1 - n0 == 1
    for r in range(rows):
        gw = oracle.cpu_linear(g.data, oracle.ENC_INT4, x0[r], hidden, inter)
        assert normwise_rel_err(fused[0].view(np.float32).reshape(rows, inter)[r], gw) < 1e-3, r


def test_multi_row_pair_settles_on_other_calls(ctx, rng):
    """A recorded multi-row Int4Linear (or pair) that no GO_SWIGLU completes is launched by the
    next call: a read of its output, a GLU over other inputs, or another projection."""
    from quicknn_amd import hip

    rows, hidden, inter = 4, 1024, 3072
    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    x0 = rng.standard_normal((rows, hidden)).astype(np.float32)
    want_g = np.stack([oracle.cpu_linear(g.data, oracle.ENC_INT4, x0[r], hidden, inter) for r in range(rows)])
    want_u = np.stack([oracle.cpu_linear(u.data, oracle.ENC_INT4, x0[r], hidden, inter) for r in range(rows)])
    x = ctx.UploadRaw(x0)
    g8, u8, hh = ctx.NewTensor(rows * inter), ctx.NewTensor(rows * inter), ctx.NewTensor(rows * inter)
    n0 = ctx.status().glu_fused
    ctx.Int4Linear(g8, x, g, rows, hidden, inter)  # recorded, then read
    assert normwise_rel_err(ctx.Download(g8).reshape(rows, inter), want_g) < 1e-3
    ctx.Int4Linear(g8, x, g, rows, hidden, inter)
    ctx.Int4Linear(u8, x, u, rows, hidden, inter)  # a pair, then a GLU with the inputs swapped
    ctx.Kernel(hip.GO_SWIGLU, rows * inter, hh, u8, g8, None, [inter, 0])
    silu = np.vectorize(oracle.silu, otypes=[np.float32])
    assert normwise_rel_err(ctx.Download(hh).reshape(rows, inter), silu(want_u) * want_g) < 1e-3
    ctx.Int4Linear(g8, x, g, rows, hidden, inter)
    ctx.Int4Linear(u8, x, u, rows, hidden, inter)  # a pair, then another projection
    ctx.Int4Linear(hh, x, g, rows, hidden, inter)
    ctx.Flush()
    assert normwise_rel_err(ctx.Download(u8).reshape(rows, inter), want_u) < 1e-3
    assert normwise_rel_err(ctx.Download(hh).reshape(rows, inter), want_g) < 1e-3
    assert ctx.status().glu_fused == n0
    for t in (x, g8, u8, hh):
        ctx.Recycle(t)


def test_multi_row_triple_under_graph_capture(ctx, rng):
    """Captured, the multi-row gate + up + GO_SWIGLU run as three launches (nothing is recorded
    during capture); every replay is bit-identical to the eager, fused run."""
    from quicknn_amd import hip

    rows, hidden, inter = 8, 1024, 3072
    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    x = ctx.UploadRaw(rng.standard_normal((rows, hidden)).astype(np.float32))
    g8, u8, hh = ctx.NewTensor(rows * inter), ctx.NewTensor(rows * inter), ctx.NewTensor(rows * inter)

    def triple():
        ctx.Int4Linear(g8, x, g, rows, hidden, inter)
        ctx.Int4Linear(u8, x, u, rows, hidden, inter)
        ctx.Kernel(hip.GO_SWIGLU, rows * inter, hh, g8, u8, None, [inter, 0])

    triple()  # eager (fused where the plans agree); also sizes the workspace
    want = [ctx.Download(t).view(np.uint32).copy() for t in (g8, u8, hh)]
    ctx.GraphBegin()
    triple()
    gid = ctx.GraphEnd()
    for rep in range(3):
        for t in (g8, u8, hh):
            ctx.Kernel(hip.GO_FILL, rows * inter, t, None, None, None, [0])
        ctx.GraphLaunch(gid)
        got = [ctx.Download(t).view(np.uint32) for t in (g8, u8, hh)]
        for a, b, nm in zip(got, want, ("gate", "up", "glu")):
            assert np.array_equal(a, b), (rep, nm)
    for t in (x, g8, u8, hh):
        ctx.Recycle(t)


@pytest.mark.parametrize("rows,hidden,inter,into", [(25, 512, 1536, "new"), (128, 2560, 9728, "new"), (100, 330, 321, "gate"),
                                                    (70, 256, 96, "up"), (65, 1000, 64, "new")])
def test_many_rows_pair_equals_separate(ctx, rng, tune, rows, hidden, inter, into):
    """From 25 rows gate, up and GO_SWIGLU run as one GEMM pair: both outputs and the GLU (also written over the
    gate or the up sums) are bit-identical to the three separate operations."""
    from quicknn_amd import hip

    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    x = ctx.UploadRaw(rng.standard_normal((rows, hidden)).astype(np.float32))
    got = {}
    for fuse in ("1", "0"):
        tune("QNN_FUSE_MLP", fuse)
        gt, ut, ht = (ctx.NewTensor(rows * inter) for _ in range(3))
        dst = {"new": ht, "gate": gt, "up": ut}[into]
        n0 = ctx.status().glu_fused
        ctx.Int4Linear(gt, x, g, rows, hidden, inter)
        ctx.Int4Linear(ut, x, u, rows, hidden, inter)
        ctx.Kernel(hip.GO_SWIGLU, rows * inter, dst, gt, ut, None, [inter, 0])
        assert ctx.status().glu_fused - n0 == int(fuse)
        got[fuse] = [ctx.Download(t).view(np.uint32).copy() for t in (gt, ut, dst)]
        for t in (gt, ut, ht):
            ctx.Recycle(t)
    for a, b in zip(got["1"], got["0"]):
        assert np.array_equal(a, b)
    ctx.Recycle(x)


@pytest.mark.parametrize("down", [True, False])
def test_one_row_swiglu_with_the_gemm_from_one_row(ctx, rng, tune, down):
    """QNN_I4_GEMM_ROWS=1 sends one-row Int4Linear calls to the GEMM.  A gate/up SwiGLU has no tensors for the two sums
    that the GEMM writes, so launched on its own (the next call is not its down projection) or fused, it is what it is
    with the default, to the bit."""
    from quicknn_amd import hip

    hidden, inter = 512, 1536
    g, u = hip.MemoryBlock.int4(rand_int4(rng, inter, hidden)), hip.MemoryBlock.int4(rand_int4(rng, inter, hidden))
    d = hip.MemoryBlock.int4(rand_int4(rng, hidden, inter))
    x = ctx.UploadRaw(rng.standard_normal(hidden).astype(np.float32))
    h, y = ctx.NewTensor(inter), ctx.NewTensor(hidden)
    got = {}
    for rows in ("25", "1"):
        tune("QNN_I4_GEMM_ROWS", rows)
        assert ctx.TrySwiGLUVector(h, x, g, u, hidden, inter)
        if down:
            ctx.Int4Linear(y, h, d, 1, inter, hidden)
        got[rows] = ctx.Download(h).view(np.uint32).copy()
    assert np.array_equal(got["25"], got["1"])
    for t in (x, h, y):
        ctx.Recycle(t)
