"""Strided axes of 640 to 1247 points in one pass (kf_cols_*): every registered
length, ragged last blocks and odd row pitches, and both sides of the rule that
picks one pass or two, against numpy; the fused axis-0 convolution and the
mixed-storage last pass on the same shapes."""
import numpy as np
import pytest

import vkfft_amd as vk
from oracle import oracle as o

pytestmark = pytest.mark.gpu

LENGTHS = [640, 648, 675, 720, 729, 750, 768, 800, 810, 864, 900, 960, 972, 1000, 1024, 1080, 1125, 1152, 1200, 1215]


def _run(ctx, dims, batch, prec, direction):
    wide = prec == vk.Precision.F64
    x = o.complex_uniform(int(np.prod(dims)) * batch, dims[0] + batch, np.complex128 if wide else np.complex64)
    c = vk.FftConfig.new(dims).with_batch_count(batch).with_precision(prec).with_inverse_normalization(True)
    ir = vk.TransformIr.build(c, direction)
    y = ctx.execute_transform(ir, x)
    f = np.fft.fftn if direction == vk.Direction.Forward else np.fft.ifftn
    ref = f(x.astype(np.complex128).reshape([batch] + dims), axes=tuple(range(1, 1 + len(dims)))).reshape(-1)
    assert o.rel_l2(y, ref) <= (2e-13 if wide else 2e-6), (dims, batch)
    return ctx.plan(ir).describe()["passes"]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("prec,G", [(vk.Precision.F32, 16), (vk.Precision.F64, 8)])
def test_lengths(hip_ctx, n, prec, G):
    for inner, direction in ((3 * G + 1, vk.Direction.Forward), (4 * G, vk.Direction.Inverse)):
        batch = 100 * G // inner + 1
        passes = _run(hip_ctx, [n, inner], batch, prec, direction)
        assert [p["kernel"] for p in passes] == ["stockham_rows", "stockham_columns"], (n, inner)
        assert passes[1]["fixed_shape"] and passes[1]["lines_per_block"] == G


@pytest.mark.parametrize("prec,G", [(vk.Precision.F32, 16), (vk.Precision.F64, 8)])
def test_no_less_precise_than_two_passes(hip_ctx, monkeypatch, prec, G):
    """One pass of large radices against the split axis (an LDS budget below the
    one that one pass needs): 1000 points had 1.45 times its error in f32 with
    the twiddles as products of one root. 3%: the spread of the error over inputs."""
    for n in LENGTHS:
        x = o.complex_uniform(n * G * 100, n, np.complex128 if prec == vk.Precision.F64 else np.complex64)
        c = vk.FftConfig.new([n, 4 * G]).with_batch_count(25).with_precision(prec).with_omit_dimension(1, True)
        ref = np.fft.fft(x.astype(np.clongdouble).reshape(25, n, 4 * G), axis=1).reshape(-1)
        err = []
        for budget, kernels in (("80", ["stockham_columns"]), ("79", ["split_axis_pass1", "split_axis_pass2"])):
            monkeypatch.setenv("VKFX_LDS_BUDGET_KB", budget)
            ctx = vk.HipExecutionContext(0)
            try:
                ir = vk.TransformIr.build(c, vk.Direction.Forward)
                y = ctx.execute_transform(ir, x)
                assert [p["kernel"] for p in ctx.plan(ir).describe()["passes"]] == kernels, n
            finally:
                ctx.close()
            err.append(float(np.linalg.norm(y - ref) / np.linalg.norm(ref)))
        assert err[0] <= 1.03 * err[1], (n, err)


@pytest.mark.parametrize("blocks,split", [(95, True), (96, False), (256, False), (257, True), (307, True), (308, False)])
def test_rule(hip_ctx, blocks, split):
    if hip_ctx.device_profile()["compute_units"] != 256:
        pytest.skip("the rule's sides are stated for 256 CUs")
    passes = _run(hip_ctx, [720, 16], blocks, vk.Precision.F32, vk.Direction.Forward)
    assert ("split_axis_pass1" in [p["kernel"] for p in passes]) == split


@pytest.mark.parametrize("n,inner,batch", [(768, 33, 40), (1024, 64, 2), (1215, 16, 3)])
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_convolution(hip_ctx, n, inner, batch, prec):
    wide = prec == vk.Precision.F64
    dt = np.complex128 if wide else np.complex64
    x = o.complex_uniform(n * inner * batch, 7, dt)
    k = o.complex_uniform(n * inner, 8, dt)
    conv = vk.ConvolutionIr.build(vk.FftConfig.new([n, inner]).with_batch_count(batch).with_precision(prec), k)
    y = hip_ctx.execute_convolution(conv, x)
    X = np.fft.fftn(x.astype(np.complex128).reshape(batch, n, inner), axes=(1, 2))
    ref = np.fft.ifftn(X * k.astype(np.complex128).reshape(n, inner), axes=(1, 2)).reshape(-1)
    assert o.rel_l2(y, ref) <= (2e-13 if wide else 2e-6)


@pytest.mark.parametrize("n,inner,fused", [(900, 16, True), (972, 16, False), (1080, 112, False), (1080, 120, True),
                                           (1125, 360, False), (1125, 375, True), (1215, 49, False), (1024, 16, True),
                                           (832, 16, True)])
def test_convolution_of_few_columns(hip_ctx, n, inner, fused):
    """Axes that the plain plan splits: one fused kernel per column, or the split
    passes around the multiply where few blocks would leave the CUs idle."""
    x, k = o.complex_uniform(n * inner, 7, np.complex64), o.complex_uniform(n * inner, 8, np.complex64)
    conv = vk.ConvolutionIr.build(vk.FftConfig.new([n, inner]), k)
    y = hip_ctx.execute_convolution(conv, x)
    ref = np.fft.ifft2(np.fft.fft2(x.astype(np.complex128).reshape(n, inner)) * k.astype(np.complex128).reshape(n, inner))
    assert o.rel_l2(y, ref.reshape(-1)) <= 2e-6
    plan = vk.Plan(hip_ctx, conv.ir, desc=conv.desc())
    names = [p["kernel"] for p in plan.describe()["passes"]]
    assert ("convolution_fused_axis0" in names) == fused and ("convolution_multiply" in names) != fused, names


@pytest.mark.parametrize("prec,tol", [(vk.Precision.F16StorageF32Compute, 1e-3),
                                      (vk.Precision.F64ComputeF32Storage, 1e-7)])
def test_mixed_storage(hip_ctx, prec, tol):
    n, inner, batch = 960, 48, 40
    x = o.complex_uniform(n * inner * batch, 9, np.complex64)
    c = vk.FftConfig.new([n, inner]).with_batch_count(batch).with_precision(prec)
    ir = vk.TransformIr.build(c, vk.Direction.Forward)
    y = hip_ctx.execute_transform_f32(ir, x)
    xs = x
    if prec == vk.Precision.F16StorageF32Compute:
        xs = x.real.astype(np.float16).astype(np.float64) + 1j * x.imag.astype(np.float16).astype(np.float64)
    ref = np.fft.fft2(xs.astype(np.complex128).reshape(batch, n, inner), axes=(1, 2)).reshape(-1)
    assert o.rel_l2(y, ref) <= tol


@pytest.mark.parametrize("prec,G", [(vk.Precision.F32, 16), (vk.Precision.F64, 8)])
def test_every_convolution_length_is_fused(hip_ctx, prec, G):
    """Every registered length's KK_CONV_1 shape, with a ragged last block (49
    columns a tensor): three passes, the fixed shape in the middle."""
    wide = prec == vk.Precision.F64
    dt, inner = (np.complex128 if wide else np.complex64), 49
    for n in LENGTHS:
        batch = 97 * G // inner + 1
        x = o.complex_uniform(n * inner * batch, n, dt)
        k = o.complex_uniform(n * inner, n + 1, dt)
        conv = vk.ConvolutionIr.build(vk.FftConfig.new([n, inner]).with_batch_count(batch).with_precision(prec), k)
        plan = vk.Plan(hip_ctx, conv.ir, desc=conv.desc())
        passes = plan.describe()["passes"]
        plan.close()
        assert [p["kernel"] for p in passes] == ["stockham_rows", "convolution_fused_axis0", "stockham_rows"], n
        assert passes[1]["fixed_shape"] and passes[1]["lines_per_block"] == G and passes[1]["fft_len"] == n
        y = hip_ctx.execute_convolution(conv, x)
        X = np.fft.fftn(x.astype(np.complex128).reshape(batch, n, inner), axes=(1, 2))
        ref = np.fft.ifftn(X * k.astype(np.complex128).reshape(n, inner), axes=(1, 2)).reshape(-1)
        assert o.rel_l2(y, ref) <= (2e-13 if wide else 2e-6), n


@pytest.mark.parametrize("prec,G,tol", [(vk.Precision.F16StorageF32Compute, 16, 1e-3),
                                        (vk.Precision.F64ComputeF32Storage, 8, 1e-7)])
def test_every_length_stores_half_precision(hip_ctx, prec, G, tol):
    """Every registered length's KK_PLAIN_EDGE_OUT shape: no boundary pass, the
    conversion inside the one pass over the columns (rows of 256, whose shape reads
    half precision)."""
    inner = 256
    for n in LENGTHS:
        batch = 97 * G // inner + 1
        x = o.complex_uniform(n * inner * batch, n, np.complex64)
        for direction, f in ((vk.Direction.Forward, np.fft.fft2), (vk.Direction.Inverse, np.fft.ifft2)):
            c = vk.FftConfig.new([n, inner]).with_batch_count(batch).with_precision(prec).with_inverse_normalization(True)
            ir = vk.TransformIr.build(c, direction)
            d = hip_ctx.plan(ir).describe()
            assert d["boundary"]["fused_edges"], n
            assert [(p["kernel"], p["fixed_shape"]) for p in d["passes"]] == [("stockham_rows", True), ("stockham_columns", True)], n
            assert d["passes"][1]["lines_per_block"] == G, n
            y = hip_ctx.execute_transform_f32(ir, x)
            xs = x
            if prec == vk.Precision.F16StorageF32Compute:
                xs = x.real.astype(np.float16).astype(np.float64) + 1j * x.imag.astype(np.float16).astype(np.float64)
            ref = f(xs.astype(np.complex128).reshape(batch, n, inner), axes=(1, 2)).reshape(-1)
            # inverses in binary16 are small numbers: their spacing is 2^-24 below 2^-14
            slack = 2.0 ** -25 * np.sqrt(2 * ref.size) / np.linalg.norm(ref) if prec == vk.Precision.F16StorageF32Compute else 0.0
            assert o.rel_l2(y, ref) <= tol + slack, (n, direction)
