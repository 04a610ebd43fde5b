"""Strided passes whose row segments share 128-byte memory lines with their
neighbours run in contiguous group ranges per XCD with cached accesses; aligned
ones keep round-robin groups. Both against numpy at the edges of a block's lines
and of the group ranges (fewer groups than XCDs, a remainder, many)."""
import numpy as np
import pytest

import vkfft_amd as vk
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [([64, 1], 3), ([64, 15], 1), ([64, 17], 2), ([100, 33], 9), ([360, 405], 2),
                                        ([512, 16], 5), ([512, 48], 1), ([7, 640], 3), ([2048, 45], 1), ([33, 12, 25], 2),
                                        ([34, 27], 5), ([202, 9], 2)])
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_strided_passes(hip_ctx, dims, batch, prec):
    cs = 16 if prec == vk.Precision.F64 else 8
    x = o.complex_uniform(int(np.prod(dims)) * batch, 3, np.complex128 if cs == 16 else np.complex64)
    axes = tuple(range(1, len(dims) + 1))
    for direction, f in ((vk.Direction.Forward, np.fft.fftn), (vk.Direction.Inverse, np.fft.ifftn)):
        c = vk.FftConfig.new(dims).with_batch_count(batch).with_precision(prec).with_inverse_normalization(True)
        ir = vk.TransformIr.build(c, direction)
        y = hip_ctx.execute_transform(ir, x)
        ref = f(x.astype(np.complex128).reshape([batch] + dims), axes=axes).reshape(-1)
        assert o.rel_l2(y, ref) <= (2e-13 if cs == 16 else 2e-6), (dims, direction)
    # the strided pass of a Stockham axis 0
    p = hip_ctx.plan(ir).describe()["passes"][-1]
    inner = int(np.prod(dims[1:]))
    if p["kernel"] == "stockham_columns" and inner > 1:
        shared = inner * cs % 128 != 0 or p["lines_per_block"] * cs % 128 != 0
        assert p["xcd_groups"] == shared, p
        if shared and p["fixed_shape"]:
            assert p["nontemporal"] == [False, False], p


@pytest.mark.parametrize("dims,batch,shared", [([24, 405], 6, True), ([24, 405], 7, False), ([24, 405], 539, False),
                                               ([24, 405], 540, True), ([127, 405], 2, False), ([128, 405], 2, True),
                                               ([24, 400], 540, False), ([200, 120], 4, False)])
def test_rule_by_size(hip_ctx, dims, batch, shared):
    """A last pass over short lines or pitches of half memory lines keeps the round-robin
    order and nontemporal stores from 512 KB to 40 MB, and everywhere where the row
    pitch is whole memory lines."""
    x = o.complex_uniform(int(np.prod(dims)) * batch, 3, np.complex64)
    ir = vk.TransformIr.build(vk.FftConfig.new(dims).with_batch_count(batch), vk.Direction.Forward)
    y = hip_ctx.execute_transform(ir, x)
    ref = np.fft.fft2(x.astype(np.complex128).reshape([batch] + dims)).reshape(-1)
    assert o.rel_l2(y, ref) <= 2e-6
    p = hip_ctx.plan(ir).describe()["passes"][-1]
    assert p["xcd_groups"] == shared, p
    if p["fixed_shape"]:
        assert p["nontemporal"] == [False, not shared], p


def test_passes_before_the_last_keep_their_ranges(hip_ctx):
    """Sizes whose last pass streams: the middle axis of a volume, the columns of a
    C2R, which the rows read next, and those of an R2C are dealt in ranges."""
    dims, batch = [40, 40, 45], 4
    x = o.complex_uniform(int(np.prod(dims)) * batch, 3, np.complex64)
    ir = vk.TransformIr.build(vk.FftConfig.new(dims).with_batch_count(batch), vk.Direction.Forward)
    y = hip_ctx.execute_transform(ir, x)
    ref = np.fft.fftn(x.astype(np.complex128).reshape([batch] + dims), axes=(1, 2, 3)).reshape(-1)
    assert o.rel_l2(y, ref) <= 2e-6
    passes = hip_ctx.plan(ir).describe()["passes"]
    assert [(p["kernel"], p["xcd_groups"]) for p in passes] == [("stockham_rows", False), ("stockham_columns", True),
                                                                ("stockham_columns", False)]
    c = vk.FftConfig.new([60, 90]).with_batch_count(40).with_transform(vk.TransformKind.ComplexToReal)
    names = [(p["kernel"], p["xcd_groups"]) for p in
             hip_ctx.plan(vk.TransformIr.build(c, vk.Direction.Inverse)).describe()["passes"]]
    assert names == [("stockham_columns", True), ("c2r_even_half", False)]
    c = vk.FftConfig.new([60, 90]).with_batch_count(40).with_transform(vk.TransformKind.RealToComplex)
    names = [(p["kernel"], p["xcd_groups"]) for p in
             hip_ctx.plan(vk.TransformIr.build(c, vk.Direction.Forward)).describe()["passes"]]
    assert names == [("r2c_even_half", False), ("stockham_columns", True)]
