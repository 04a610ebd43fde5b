"""The axis passes of small 2-D and 3-D C2C transforms, which one kernel takes by
default: with VKFX_FIELD=0 the shapes of the N-D parity and strided-group lists
run on rows, columns and split columns, against numpy, with the passes named;
knobs that select kernels or budgets of the axis passes keep them by themselves."""
import numpy as np
import pytest

import vkfft_amd as vk
from oracle import oracle as o

pytestmark = pytest.mark.gpu

F32, F64 = vk.Precision.F32, vk.Precision.F64
R, C, S1, S2 = "stockham_rows", "stockham_columns", "split_axis_pass1", "split_axis_pass2"


def _ir(dims, batch, prec, direction=vk.Direction.Forward):
    c = vk.FftConfig.new(dims).with_batch_count(batch).with_precision(prec).with_inverse_normalization(True)
    return vk.TransformIr.build(c, direction)


def _check(ctx, dims, batch, prec, names=None):
    x = o.complex_uniform(int(np.prod(dims)) * batch, 3, np.complex128 if prec == F64 else np.complex64)
    axes = tuple(range(1, len(dims) + 1))
    for direction, f in ((vk.Direction.Forward, np.fft.fftn), (vk.Direction.Inverse, np.fft.ifftn)):
        ir = _ir(dims, batch, prec, direction)
        y = ctx.execute_transform(ir, x)
        ref = f(x.astype(np.complex128).reshape([batch] + dims), axes=axes).reshape(-1)
        assert o.rel_l2(y, ref) <= (2e-13 if prec == F64 else 2e-6), (dims, direction)
        passes = ctx.plan(ir).describe()["passes"]
        if names:
            assert [p["kernel"] for p in passes] == names, dims
    return passes


@pytest.fixture
def ctx(hip_ctx):
    """A context of its own: plans read the knobs when built."""
    c = vk.HipExecutionContext(0)
    yield c
    c.close()


@pytest.mark.parametrize("dims,batch,names", [
    ([64, 48], 2, [R, C]), ([16, 12, 10], 2, [R, C, C]), ([25, 12, 8], 2, [R, C, C]), ([120, 30], 2, [R, C]),
    ([32, 16, 8], 3, [R, C, C]), ([16, 128], 5, [R, C]), ([256, 3], 2, [R, C]), ([96, 20], 2, [R, C]),
    ([360, 12], 1, [R, C]), ([12, 48, 5], 2, [R, C, C]), ([7, 640], 3, [R, C]), ([640, 3], 2, [R, C]), ([33, 12, 25], 2, [R, C, C]),
    # axes long enough to run as two passes
    ([1024, 8], 2, [R, S1, S2]), ([2048, 3], 1, [R, S1, S2]), ([1000, 6], 1, [R, S1, S2])])
@pytest.mark.parametrize("prec", [F32, F64])
def test_passes_of_small_fields(ctx, monkeypatch, dims, batch, names, prec):
    monkeypatch.setenv("VKFX_FIELD", "0")
    _check(ctx, dims, batch, prec, names)


@pytest.mark.parametrize("dims", [[64, 1], [64, 15], [64, 17], [100, 33], [512, 16], [512, 5], [33, 12, 25], [30, 7]])
@pytest.mark.parametrize("prec", [F32, F64])
def test_shared_lines_of_small_fields(ctx, monkeypatch, dims, prec):
    monkeypatch.setenv("VKFX_FIELD", "0")
    p = _check(ctx, dims, 2, prec)[-1]  # below 512 KB
    cs, inner = 16 if prec == F64 else 8, int(np.prod(dims[1:]))
    if inner == 1:
        assert p["kernel"] == R
        return
    assert p["kernel"] == C
    shared = inner * cs % 128 != 0 or p["lines_per_block"] * cs % 128 != 0
    assert p["xcd_groups"] == shared, p
    if shared and p["fixed_shape"]:
        assert p["nontemporal"] == [False, False], p


@pytest.mark.parametrize("name,value", [("VKFX_DISABLE_FIXED", "1"), ("VKFX_REGISTER_EXCHANGE", "1"),
                                        ("VKFX_LDS_BUDGET_KB", "40")])
@pytest.mark.parametrize("dims", [[120, 30], [25, 12, 8]])
def test_knobs_of_the_axis_passes(ctx, monkeypatch, name, value, dims):
    monkeypatch.setenv(name, value)
    passes = _check(ctx, dims, 2, F32, [R] + [C] * (len(dims) - 1))
    assert name != "VKFX_DISABLE_FIXED" or not any(p["fixed_shape"] for p in passes)
