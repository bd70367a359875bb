"""Edge sizes of the dense kernels' tiles, loops and dispatch rules on the GPU,
against the CPU oracle."""
import numpy as np
import pytest

import m1moe_amd as m
from m1moe_amd.decoder import DenseOps
from oracle import oracle as orc

from cases import rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops_ctx():
    ctx = m.HIPContext(m.make_shape(128, 8, 2, 64, 64))
    yield ctx, DenseOps(ctx)
    ctx.close()


def bf16(a):
    from m1moe_amd.synth import f32_to_bf16
    return f32_to_bf16(np.asarray(a, np.float32))


@pytest.mark.parametrize("n", [2, 3, 5, 4095, 4097, 32768, 32769, 65539])
@pytest.mark.parametrize("where", ["first", "last", "tie", "nan0"])
def test_argmax_edges(ops_ctx, n, where):
    """The largest value in the first or last element (a group of four or the
    tail after it), tied across the passes, and the NaN rule; exact."""
    ctx, ops = ops_ctx
    x = np.random.default_rng(n).normal(0, 1, n).astype(np.float32)
    if where == "tie":
        x[[n // 2, n - 1]] = 20.0
    else:
        x[0 if where == "first" else n - 1] = 20.0
    if where == "nan0":
        x[0] = np.nan
    dx, di = ctx.to_device(x), ctx.alloc(16)
    say(f"argmax n={n} {where}")
    ops.argmax(dx, n, di)
    ctx.sync()
    assert int(di.download(np.int32, 1)[0]) == orc.argmax(x)
    dx.free()
    di.free()


@pytest.mark.parametrize("n", [4, 64, 4092, 4096, 4100, 8192, 8196])
def test_rmsnorm_edges(ops_ctx, n):
    """Both sides of the register form's limits (8192 elements, multiples of
    four): f32 sums of at most 8196 squares, well inside 1e-6."""
    ctx, ops = ops_ctx
    rng = np.random.default_rng(n)
    x, w = rng.normal(0, 2, n).astype(np.float32), bf16(rng.normal(1, 0.1, n))
    dx, dw, dout = ctx.to_device(x), ctx.to_device(w), ctx.alloc(4 * n)
    say(f"rmsnorm n={n}")
    ops.rmsnorm(dx, dw, dout, n, 1e-5)
    ctx.sync()
    assert rel_l2(dout.download(np.float32), orc.rmsnorm(x, w, 1e-5)) < 1e-6
    for b in (dx, dw, dout):
        b.free()
