"""One-kernel DCT / DST lines (KK_R2R_*): every form at the sizes where its
packing, pairing or block edges change, along contiguous and strided axes,
against scipy's pocketfft. f64 meets the repository's 1e-13 gate, f32 its 1e-5
gate, and f32 also 16 units of rounding (2^-24) times log2 of the FFT length:
each stage adds a few units, the phases run in f64."""
import math

import numpy as np
import pytest

import vkfft_amd as vk
from oracle import oracle as o

pytestmark = pytest.mark.gpu

KINDS = ["dct1", "dct2", "dct3", "dct4", "dst1", "dst2", "dst3", "dst4"]


def _plan(ctx, name, dims, batch, prec, direction=vk.Direction.Forward, omit=()):
    t = int(name[-1])
    kind = vk.TransformKind.dct(t) if name.startswith("dct") else vk.TransformKind.dst(t)
    c = vk.FftConfig.new(dims).with_batch_count(batch).with_precision(prec).with_transform(kind)
    for ax in omit:
        c.with_omit_dimension(ax, True)
    return vk.TransformIr.build(c, direction)


def _check(y, ref, n, prec):
    err = o.rel_l2(y, ref)
    assert err <= (1e-13 if prec == vk.Precision.F64 else min(1e-5, 16 * 2.0 ** -24 * math.log2(2 * n))), (n, err)


@pytest.mark.parametrize("name", KINDS)
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_rows(hip_ctx, name, prec):
    import scipy.fft as sf
    f = sf.dct if name.startswith("dct") else sf.dst
    # smallest, odd and even halves, fixed shapes and the runtime shape (14, 26, 1386), ragged last blocks
    for n, batch in ((2, 5), (3, 1), (4, 130), (6, 3), (14, 67), (15, 64), (26, 9), (64, 33), (100, 7), (720, 4),
                     (1000, 3), (1386, 2), (2048, 3), (16384 if prec == vk.Precision.F32 else 8192, 2)):
        if name == "dct1":
            n += 1  # the reduction of type I has n - 1 points
        if name == "dst1":
            n -= 1
        if n < 2:
            continue
        x = o.uniform(n * batch, n + batch, np.float32 if prec == vk.Precision.F32 else np.float64)
        ir = _plan(hip_ctx, name, [n], batch, prec)
        y = hip_ctx.execute_transform(ir, x)
        _check(y, f(x.astype(np.float64).reshape(batch, n), type=int(name[-1]), axis=-1).reshape(-1), n, prec)
        labels = [p["kernel"] for p in hip_ctx.plan(ir).describe()["passes"]]
        odd4 = name.endswith("4") and n % 2
        assert odd4 or labels == ["r2r_line"], (name, n, labels)


@pytest.mark.parametrize("name", KINDS)
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_strided_lines(hip_ctx, name, prec):
    import scipy.fft as sf
    f = sf.dct if name.startswith("dct") else sf.dst
    # columns below, at and above the lines of a block, odd column counts, several outer lines
    for n, inner, batch in ((2, 1, 3), (4, 31, 2), (12, 33, 3), (18, 64, 1), (30, 5, 7), (44, 37, 2), (96, 32, 2),
                            (720, 65, 1), (2048, 17, 1), (27, 35, 2)):
        if name == "dct1":
            n += 1
        if name == "dst1":
            n -= 1
        if n < 2:
            continue
        x = o.uniform(n * inner * batch, n + inner, np.float32 if prec == vk.Precision.F32 else np.float64)
        y = hip_ctx.execute_transform(_plan(hip_ctx, name, [n, inner], batch, prec, omit=(1,)), x)
        ref = f(x.astype(np.float64).reshape(batch, n, inner), type=int(name[-1]), axis=1).reshape(-1)
        _check(y, ref, n, prec)


def _shapes(prec):
    """(half length, lines a block, columns) of every registered type II / III shape."""
    import importlib.util
    import os
    src = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vkfft-rs_amd", "csrc", "gen_shape_tables.py")
    spec = importlib.util.spec_from_file_location("gen_shape_tables", src)
    g = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(g)
    rows = g.TABLES["kf_r2r_f64" if prec == vk.Precision.F64 else "kf_r2r_f32"]
    return sorted({(r[2], r[4], r[5]) for r in rows})


@pytest.mark.parametrize("name", ["dct2", "dct3", "dst2", "dst3"])
@pytest.mark.parametrize("col", [False, True])
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_every_registered_shape(hip_ctx, name, col, prec):
    """All fixed shapes of types II and III, rows and columns, one full block and a
    ragged one (columns: over two outer lines, so that blocks cross them)."""
    import scipy.fft as sf
    f = sf.dct if name.startswith("dct") else sf.dst
    dt = np.float32 if prec == vk.Precision.F32 else np.float64
    seen, unreached = 0, []
    for M, G, is_col in _shapes(prec):
        if is_col != col:
            continue
        n, seen = 2 * M, seen + 1
        dims, batch = ([n, G // 2 + 2], 2) if col else ([n], G + 1)
        x = o.uniform(int(np.prod(dims)) * batch, n, dt)
        ir = _plan(hip_ctx, name, dims, batch, prec, omit=(1,) if col else ())
        plan = vk.Plan(hip_ctx, ir)
        passes = plan.describe()["passes"]
        plan.close()
        if len(passes) != 1:
            unreached.append(M)
            continue
        (p,) = passes
        assert p["kernel"] == "r2r_line" and p["fixed_shape"] and p["lines_per_block"] == G and p["fft_len"] == M, (n, p)
        y = hip_ctx.execute_transform(ir, x)
        _check(y, f(x.astype(np.float64).reshape([batch] + dims), type=int(name[-1]), axis=1).reshape(-1), n, prec)
    assert seen >= 60 and not unreached, unreached


@pytest.mark.parametrize("name", KINDS)
def test_described_lengths_are_the_executed_ones(hip_ctx, name):
    """The description's kernel length is that of the launch: half of the reduction's
    in the packed forms of types II and III, N -+ 1 in type I."""
    t = int(name[-1])
    for n in (64, 63):
        ir = _plan(hip_ctx, name, [n], 2, vk.Precision.F32)
        d = hip_ctx.plan(ir).describe()
        kernel = d["r2r"]["kernel_fft_len"]
        if t == 4 and n % 2:
            assert kernel == d["r2r"]["fft_len"] == 2 * n and len(d["passes"]) > 1
            continue
        # DCT-I of 64 points: the even extension has 126, a Stockham length; of 63, 124 = 4 x 31 is none
        if len(d["passes"]) == 1:
            assert d["passes"][0]["kernel"] == "r2r_line" and d["passes"][0]["fft_len"] == kernel
            assert kernel == {1: n - 1 if name == "dct1" else n + 1, 2: n // 2 if n % 2 == 0 else n,
                              3: n // 2 if n % 2 == 0 else n, 4: n // 2}[t]
        else:
            assert kernel == d["r2r"]["fft_len"] and t == 1


@pytest.mark.parametrize("name", KINDS)
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_few_lines(hip_ctx, name, prec):
    """Fewer blocks than CUs on the runtime shapes: lines spread over the CUs with
    more threads than the stages need (at most the line's elements), along rows and
    columns, and the three passes for lone strided lines that fill the LDS."""
    import scipy.fft as sf
    f = sf.dct if name.startswith("dct") else sf.dst
    cus = hip_ctx.device_profile()["compute_units"]
    dt = np.float32 if prec == vk.Precision.F32 else np.float64
    for n, inner, batch in ((14, 1, 1), (28, 1, 3), (84, 1, cus), (84, 1, cus + 1), (154, 1, 3 * cus + 5), (1386, 1, 2),
                            (4158, 1, 2), (14, 5, 3), (154, 30, 7), (1386, 9, 1), (2772, 33, 1)):
        n += {"dct1": 1, "dst1": -1}.get(name, 0)
        lines = batch * inner
        x = o.uniform(n * lines, n + lines, dt)
        ir = _plan(hip_ctx, name, [n, inner] if inner > 1 else [n], batch, prec, omit=(1,) if inner > 1 else ())
        y = hip_ctx.execute_transform(ir, x)
        _check(y, f(x.astype(np.float64).reshape(batch, n, inner), type=int(name[-1]), axis=1).reshape(-1), n, prec)
        (p,) = hip_ctx.plan(ir).describe()["passes"]
        assert p["kernel"] == "r2r_line", p
        if not p["fixed_shape"] and lines < cus * 4:
            G = p["lines_per_block"]
            assert G <= -(-lines // cus) and p["block"] >= G * min(p["fft_len"], (512 if lines <= cus else 256) // G), p
    n = {"dct1": 2049, "dst1": 2047, "dct4": 4096, "dst4": 4096}.get(name)
    for inner, one in ((32, False), (33, True)) if n else ():
        passes = hip_ctx.plan(_plan(hip_ctx, name, [n, inner], 1, prec, omit=(1,))).describe()["passes"]
        assert (len(passes) == 1) == one, passes


@pytest.mark.parametrize("name", ["dct2", "dct3", "dct4", "dct1", "dst2", "dst3"])
def test_lines_stay_on_their_own(hip_ctx, name):
    """A line of NaN, of infinities or of tiny values leaves its neighbours
    bit for bit as they are alone, and a small line keeps its own relative error."""
    n, batch = 48, 9
    x = o.uniform(n * batch, 5, np.float32).reshape(batch, n)
    ir = _plan(hip_ctx, name, [n], batch, vk.Precision.F32)
    clean = hip_ctx.execute_transform(ir, x.reshape(-1)).reshape(batch, n)
    bad = x.copy()
    bad[1], bad[4], bad[6] = np.nan, np.inf, x[6] * np.float32(2.0 ** -60)
    y = hip_ctx.execute_transform(ir, bad.reshape(-1)).reshape(batch, n)
    for b in (0, 2, 3, 5, 7, 8):
        assert np.array_equal(y[b], clean[b]), b
    assert np.array_equal(y[6], clean[6] * np.float32(2.0 ** -60))
    assert not np.isfinite(y[1]).any() and not np.isfinite(y[4]).all()


@pytest.mark.parametrize("name", KINDS)
def test_one_kernel_matches_the_three_passes(hip_ctx, name, monkeypatch):
    """The same plans with VKFX_R2R_FUSED=0 (pre pass, complex FFT, post pass)."""
    dims, batch = [36, 50], 3
    x = o.uniform(36 * 50 * batch, 8, np.float64)
    for direction in (vk.Direction.Forward, vk.Direction.Inverse):
        ir = _plan(hip_ctx, name, dims, batch, vk.Precision.F64, direction)
        y = hip_ctx.execute_transform(ir, x)
        monkeypatch.setenv("VKFX_R2R_FUSED", "0")
        ctx = vk.HipExecutionContext(0)
        try:
            z = ctx.execute_transform(ir, x)
            assert any(p["kernel"] == "r2r_pre" for p in ctx.plan(ir).describe()["passes"])
        finally:
            ctx.close()
            monkeypatch.delenv("VKFX_R2R_FUSED")
        assert o.rel_l2(y, z) <= 1e-14


@pytest.mark.parametrize("name", KINDS)
@pytest.mark.parametrize("prec", [vk.Precision.F32, vk.Precision.F64])
def test_no_less_precise_than_the_three_passes(hip_ctx, name, prec, monkeypatch):
    """The half-length FFTs' twiddles and the phases are as exact as the full-length
    FFT's and sincospi: with products of one root f32 DST-II of 8192 points had 1.45
    times the error of the three passes. f32 5%: the spread over inputs; f64 15%: the
    packing's own roundings at short lines (1.08 at DCT-III of 60 points), which f32
    lines do in f64."""
    import scipy.fft as sf
    f = sf.dct if name.startswith("dct") else sf.dst
    dt, slack = (np.float32, 1.05) if prec == vk.Precision.F32 else (np.float64, 1.15)
    for n, batch in ((40, 300), (84, 200), (616, 40), (2048, 16), (8192, 4)):
        n += {"dct1": 1, "dst1": -1}.get(name, 0)
        if n > 8192:
            continue
        x = o.uniform(n * batch, n, dt)
        ref = f(x.astype(np.longdouble).reshape(batch, n), type=int(name[-1]), axis=-1).reshape(-1)
        err = {}
        for fused in ("1", "0"):
            monkeypatch.setenv("VKFX_R2R_FUSED", fused)
            ctx = vk.HipExecutionContext(0)
            try:
                ir = _plan(ctx, name, [n], batch, prec)
                y = ctx.execute_transform(ir, x)
                assert (len(ctx.plan(ir).describe()["passes"]) == 1) == (fused == "1")
            finally:
                ctx.close()
            err[fused] = float(np.linalg.norm(y - ref) / np.linalg.norm(ref))
        assert err["1"] <= slack * err["0"], (n, err)
