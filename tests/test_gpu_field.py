"""Small 2-D and 3-D complex fields in one kernel: every radix and the shapes at
the edges of its rules (shortest axes, copied-in first stage, several fields a
block with a ragged last one, the largest fields and the first that keep the axis
passes), against numpy and against the axis passes; in place and out of place."""
import numpy as np
import pytest

import vkfft_amd as vk
from oracle import oracle as o

pytestmark = pytest.mark.gpu

# (dims, batch, one kernel in f32, in f64)
CASES = [([2, 2], 1, True, True), ([2, 2], 3001, True, True), ([3, 5], 2000, True, True), ([64, 64], 1, True, False),
         ([64, 64], 3, True, False), ([32, 32], 4099, True, True), ([13, 11], 1500, True, True), ([9, 7], 1, True, True),
         ([16, 16], 5, True, True), ([2, 1000], 2, True, True), ([1000, 2], 2, True, True), ([16, 8, 8], 700, True, True),
         ([10, 12, 15], 3, True, True), ([3, 2, 26], 4, True, True), ([49, 81], 2, True, True), ([44, 104], 2, True, False),
         ([16, 16, 16], 2, True, True), ([8, 512], 2, True, True), ([72, 72], 1, True, False), ([91, 77], 512, True, False),
         ([91, 77], 513, False, False), ([128, 128], 1, False, False), ([36, 60], 2912, True, True), ([36, 60], 2913, False, True),
         ([17, 16], 2, False, False), ([16, 1], 2, False, False)]


def _plan(ctx, dims, batch, prec, direction):
    c = vk.FftConfig.new(dims).with_batch_count(batch).with_precision(prec).with_inverse_normalization(True)
    return vk.TransformIr.build(c, direction)


@pytest.mark.parametrize("dims,batch,one32,one64", CASES)
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_fields(hip_ctx, monkeypatch, dims, batch, one32, one64, prec):
    wide = prec == vk.Precision.F64
    x = o.complex_uniform(int(np.prod(dims)) * batch, 5, np.complex128 if wide else np.complex64)
    axes = tuple(range(1, len(dims) + 1))
    # the axis passes' bound at these lengths: a few roundings a stage
    tol = 4e-15 if wide else 1e-6
    for direction, f in ((vk.Direction.Forward, np.fft.fftn), (vk.Direction.Inverse, np.fft.ifftn)):
        ir = _plan(hip_ctx, dims, batch, prec, direction)
        y = hip_ctx.execute_transform(ir, x)
        ref = f(x.astype(np.complex128).reshape([batch] + dims), axes=axes).reshape(-1)
        assert o.rel_l2(y, ref) <= tol, (dims, batch, direction)
        assert ([p["kernel"] for p in hip_ctx.plan(ir).describe()["passes"]] == ["field"]) == (one64 if wide else one32)
    monkeypatch.setenv("VKFX_FIELD", "0")
    other = vk.Plan(hip_ctx, ir)
    assert all(p["kernel"] != "field" for p in other.describe()["passes"])


# fields alone on a CU: (dims, batch, precision, one kernel by the rule of 256 CUs)
ALONE = [([20, 20, 20], 1, "f32", False), ([16, 16, 16], 1, "f64", True), ([12, 12, 20], 1, "f64", False),
         ([8, 30, 36], 255, "f32", False), ([8, 30, 36], 256, "f32", True), ([18, 18, 18], 256, "f32", False),
         ([25, 320], 1, "f32", False), ([36, 225], 1, "f32", False), ([15, 540], 300, "f32", False),
         ([8, 512], 1, "f64", False), ([8, 512], 3, "f64", True), ([8, 512], 4, "f64", False), ([8, 512], 256, "f64", True), ([45, 64], 1, "f64", False),
         ([48, 108], 1, "f32", True), ([100, 80], 1, "f32", True), ([160, 50], 1, "f32", False), ([160, 50], 256, "f32", True),
         ([1000, 8], 1, "f32", False), ([270, 30], 256, "f32", False), ([80, 60], 513, "f32", False), ([91, 77], 57, "f32", True),
         ([4, 2000], 31, "f32", False), ([4, 2000], 32, "f32", True), ([9, 792], 1, "f32", False), ([48, 98], 63, "f32", False),
         ([48, 98], 64, "f32", True), ([36, 105], 255, "f64", True), ([1024, 4], 1, "f64", True), ([2, 2, 1000], 1, "f64", True)]


@pytest.mark.parametrize("dims,batch,prec,one", ALONE)
def test_alone_on_a_cu(hip_ctx, monkeypatch, dims, batch, prec, one):
    """Both sides of the rule for fields whose LDS takes the CU, and the same
    results from the one kernel where the rule keeps the axis passes."""
    if hip_ctx.device_profile()["compute_units"] != 256:
        pytest.skip("the rule's sides are stated for 256 CUs")
    wide = prec == "f64"
    x = o.complex_uniform(int(np.prod(dims)) * batch, 5, np.complex128 if wide else np.complex64)
    axes = tuple(range(1, len(dims) + 1))
    ref = np.fft.fftn(x.astype(np.complex128).reshape([batch] + dims), axes=axes).reshape(-1)
    for env in (None, "1"):
        if env:
            monkeypatch.setenv("VKFX_FIELD", env)
        ctx = vk.HipExecutionContext(0)
        try:
            ir = _plan(ctx, dims, batch, vk.Precision.F64 if wide else vk.Precision.F32, vk.Direction.Forward)
            assert o.rel_l2(ctx.execute_transform(ir, x), ref) <= (4e-15 if wide else 1e-6)
            assert ([p["kernel"] for p in ctx.plan(ir).describe()["passes"]] == ["field"]) == (one or env == "1")
        finally:
            ctx.close()


@pytest.mark.parametrize("dims,batch", [([64, 64], 2), ([30, 14], 1100), ([8, 9, 10], 7)])
def test_in_place(hip_ctx, dims, batch):
    import torch
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.view_as_complex(torch.rand([batch] + dims + [2], generator=g, device="cuda").sub_(0.5))
    plan = vk.Plan(hip_ctx, _plan(hip_ctx, dims, batch, vk.Precision.F32, vk.Direction.Forward))
    ref = torch.fft.fftn(x.to(torch.complex128), dim=tuple(range(1, len(dims) + 1)))
    y = torch.empty_like(x)
    plan.execute_tensors(x, y)
    plan.execute_tensors(x, x)
    torch.cuda.synchronize()
    assert torch.equal(x, y)
    assert float((x - ref).abs().norm() / ref.abs().norm()) <= 1e-6


def test_no_less_precise_than_the_axis_passes(hip_ctx, monkeypatch):
    """A field's twiddles are as exact as those of one pass per axis: lengths of
    large radices (10 x 10 x 10, 12 x 4, 9 x 7 x 7 x 7), whose error grows where a
    radix's twiddles are products of one root alone (1.4 times the axis passes' at
    1000 x 2 x 2). 5%: the spread of the error over inputs."""
    for prec, dt in ((vk.Precision.F32, np.complex64), (vk.Precision.F64, np.complex128)):
        for dims, batch in (([1000, 2, 2], 8), ([64, 48], 4), ([80, 60], 4), ([720, 12], 2), ([3087, 2], 2), ([4, 40, 48], 2)):
            if prec == vk.Precision.F64 and np.prod(dims) > 4000:
                continue
            x = o.complex_uniform(int(np.prod(dims)) * batch, 5, dt)
            axes = tuple(range(1, len(dims) + 1))
            ref = np.fft.fftn(x.astype(np.clongdouble).reshape([batch] + dims), axes=axes).reshape(-1)
            err = {}
            for field in ("1", "0"):
                monkeypatch.setenv("VKFX_FIELD", field)
                ctx = vk.HipExecutionContext(0)
                try:
                    ir = _plan(ctx, dims, batch, prec, vk.Direction.Forward)
                    err[field] = float(np.linalg.norm(ctx.execute_transform(ir, x) - ref) / np.linalg.norm(ref))
                    assert (ctx.plan(ir).describe()["passes"][0]["kernel"] == "field") == (field == "1")
                finally:
                    ctx.close()
            assert err["1"] <= 1.05 * err["0"], (dims, prec, err)
