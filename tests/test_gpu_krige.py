"""GPU tier: the kriging calculators (krige.rs:24-118) against the reference's
golden values and the FP64 oracle.

Tolerance: the reference's own tests allow 6 ulps (krige.rs:208, 220, 243);
the GPU sums in another order (tiles of 128 conditions, FMA), so random cases
are held to 1e-12 of the largest term of the sum, i.e. FP64 rounding only.
"""
from __future__ import annotations

import json
import os

import numpy as np
import pytest

import oracle
import gstools_core
from conftest import GOLDEN
from gstools_core import _native

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def krige_rs():
    with open(os.path.join(GOLDEN, "krige_rs_fixture.json")) as f:
        d = json.load(f)
    return {k: (np.array(v, dtype=np.float64) if k != "source" else v) for k, v in d.items()}


def ulps(a, b):
    return np.abs(a - b) / np.spacing(np.abs(b))


def test_golden_values(krige_rs):
    m, v, c = krige_rs["krig_mat"], krige_rs["krig_vecs"], krige_rs["cond"]
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    assert np.max(ulps(f, krige_rs["field"])) <= 6
    assert np.max(ulps(e, krige_rs["error"])) <= 6
    f2 = gstools_core.calc_field_krige(m, v, c)
    assert np.max(ulps(f2, krige_rs["field"])) <= 6


def _scale(m, v, c):
    # largest term of the sums: |c_i| |fac_i| and |v_ij| |fac_i|
    fac = np.abs(m).T @ np.abs(v)
    return max(float(np.max(np.abs(c)[:, None] * fac, initial=0.0)),
               float(np.max(np.abs(v) * fac, initial=0.0)), 1e-300)


@pytest.mark.parametrize("n,N", [(1, 1), (3, 6), (63, 65), (64, 64), (65, 1000), (130, 63),
                                 (127, 129), (128, 128), (129, 300), (257, 2000),
                                 (200, 5000), (1, 777)])
def test_random_against_oracle(n, N):
    rng = np.random.default_rng(1000 * n + N)
    a = rng.normal(size=(n, n))
    m = a @ a.T / n + np.eye(n)
    v = rng.normal(size=(n, N))
    c = rng.normal(size=n)
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    rf, re = oracle.calc_field_krige_and_variance(m, v, c)
    tol = 1e-12 * n * _scale(m, v, c)
    assert np.abs(f - rf).max() <= tol
    assert np.abs(e - re).max() <= tol
    f2 = gstools_core.calc_field_krige(m, v, c)
    assert np.abs(f2 - rf).max() <= tol


def test_strided_views_and_reproducibility():
    rng = np.random.default_rng(7)
    m = rng.normal(size=(90, 90))
    v = rng.normal(size=(90, 3000))
    c = rng.normal(size=90)
    f, e = gstools_core.calc_field_krige_and_variance(m[::-1, ::-1], v[::-1, ::2], c[::-1])
    rf, re = oracle.calc_field_krige_and_variance(m[::-1, ::-1], v[::-1, ::2], c[::-1])
    tol = 1e-12 * 90 * _scale(m, v, c)
    assert np.abs(f - rf).max() <= tol and np.abs(e - re).max() <= tol
    f2, e2 = gstools_core.calc_field_krige_and_variance(m[::-1, ::-1], v[::-1, ::2], c[::-1])
    np.testing.assert_array_equal(f, f2)
    np.testing.assert_array_equal(e, e2)


def test_large_against_oracle_subset():
    rng = np.random.default_rng(8)
    n, N = 1000, 100_000
    a = rng.normal(size=(n, n)) / np.sqrt(n)
    m = a @ a.T
    v = rng.normal(size=(n, N))
    c = rng.normal(size=n)
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    sub = np.sort(rng.choice(N, 500, replace=False))
    rf, re = oracle.calc_field_krige_and_variance(m, np.ascontiguousarray(v[:, sub]), c)
    tol = 1e-12 * n * _scale(m, v[:, sub], c)
    assert np.abs(f[sub] - rf).max() <= tol
    assert np.abs(e[sub] - re).max() <= tol


def test_device_entry_point_matches_host():
    rng = np.random.default_rng(9)
    n, N = 150, 4000
    m = rng.normal(size=(n, n))
    v = rng.normal(size=(n, N))
    c = rng.normal(size=n)
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    lib = _native.lib()
    dm = _native.DeviceBuffer.from_array(m)
    dv = _native.DeviceBuffer.from_array(v)
    dc = _native.DeviceBuffer.from_array(c)
    out = _native.DeviceBuffer(16 * N)
    nb = lib.gsc_krige_workspace_bytes(n, N, 1)
    work = _native.DeviceBuffer(nb)
    opts = _native.make_opts()
    import ctypes
    _native.check(lib.gsc_krige_dev(n, N, dm.ptr, dv.ptr, N, dc.ptr, out.ptr, out.ptr + 8 * N,
                                    work.ptr, nb, ctypes.byref(opts), None))
    _native.synchronize()
    res = out.to_array(np.float64, 2 * N)
    np.testing.assert_array_equal(res[:N], f)
    np.testing.assert_array_equal(res[N:], e)
    # a workspace that is too small is refused
    with pytest.raises(ValueError):
        _native.check(lib.gsc_krige_dev(n, N, dm.ptr, dv.ptr, N, dc.ptr, out.ptr, out.ptr + 8 * N,
                                        work.ptr, nb - 8, ctypes.byref(opts), None))
    for b in (dm, dv, dc, out, work):
        b.free()


@pytest.mark.parametrize("with_error", [True, False])
def test_device_entry_point_row_pitch(with_error):
    # krig_vecs rows with a pitch above N (a view of a wider array): the same
    # results as the dense host call, bit for bit
    import ctypes
    rng = np.random.default_rng(10)
    n, N, pitch = 140, 1000, 1037
    m = rng.normal(size=(n, n))
    wide = rng.normal(size=(n, pitch))
    c = rng.normal(size=n)
    f, e = gstools_core.calc_field_krige_and_variance(m, np.ascontiguousarray(wide[:, :N]), c)
    if not with_error:
        f = gstools_core.calc_field_krige(m, np.ascontiguousarray(wide[:, :N]), c)
    lib = _native.lib()
    dm = _native.DeviceBuffer.from_array(m)
    dv = _native.DeviceBuffer.from_array(wide)
    dc = _native.DeviceBuffer.from_array(c)
    out = _native.DeviceBuffer(16 * N)
    nb = lib.gsc_krige_workspace_bytes(n, N, 1 if with_error else 0)
    work = _native.DeviceBuffer(nb)
    opts = _native.make_opts()
    _native.check(lib.gsc_krige_dev(n, N, dm.ptr, dv.ptr, pitch, dc.ptr, out.ptr,
                                    out.ptr + 8 * N if with_error else None, work.ptr, nb,
                                    ctypes.byref(opts), None))
    _native.synchronize()
    res = out.to_array(np.float64, 2 * N)
    np.testing.assert_array_equal(res[:N], f)
    if with_error:
        np.testing.assert_array_equal(res[N:], e)
    for b in (dm, dv, dc, out, work):
        b.free()


def test_empty_and_shape_errors():
    f, e = gstools_core.calc_field_krige_and_variance(np.zeros((0, 0)), np.zeros((0, 4)),
                                                      np.zeros(0))
    np.testing.assert_array_equal(f, np.zeros(4))
    np.testing.assert_array_equal(e, np.zeros(4))
    f, e = gstools_core.calc_field_krige_and_variance(np.eye(2), np.zeros((2, 0)), np.ones(2))
    assert f.shape == (0,) and e.shape == (0,)
    with pytest.raises(ValueError):
        gstools_core.calc_field_krige(np.eye(3), np.zeros((2, 4)), np.ones(3))
    with pytest.raises(ValueError):
        gstools_core.calc_field_krige(np.zeros((3, 2)), np.zeros((3, 4)), np.ones(3))
    with pytest.raises(ValueError):
        gstools_core.calc_field_krige(np.eye(3), np.zeros((3, 4)), np.ones(2))


@pytest.mark.parametrize("n,N", [(16, 600), (17, 600), (128, 8500), (129, 8500), (137, 30_011),
                                 (250, 40_000), (256, 70_000), (385, 250_000)])
def test_triangle_form(n, N):
    # sizes at which the error is summed over the lower triangle (one row
    # block, several, several splits), with an unsymmetric matrix; tolerance:
    # FP64 rounding, as for the random cases above
    rng = np.random.default_rng(n)
    m = rng.normal(size=(n, n)) + np.eye(n)
    v = rng.normal(size=(n, N))
    c = rng.normal(size=n)
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    sub = np.unique(np.concatenate([np.arange(130), np.arange(N - 130, N),
                                    rng.choice(N, 300, replace=False)]))
    rf, re = oracle.calc_field_krige_and_variance(m, np.ascontiguousarray(v[:, sub]), c)
    tol = 1e-12 * n * _scale(m, v[:, sub], c)
    assert np.abs(f[sub] - rf).max() <= tol
    assert np.abs(e[sub] - re).max() <= tol


def test_triangle_form_nan_stays_in_its_column():
    n, N = 130, 20_000
    rng = np.random.default_rng(3)
    m = rng.normal(size=(n, n))
    v = rng.normal(size=(n, N))
    c = rng.normal(size=n)
    f0, e0 = gstools_core.calc_field_krige_and_variance(m, v, c)
    v[n - 1, 5] = np.nan
    v[3, N - 1] = np.inf
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    bad = [5, N - 1]
    assert np.isnan(f[5]) and np.isnan(e[5])
    assert not np.isfinite(f[N - 1]) and not np.isfinite(e[N - 1])
    np.testing.assert_array_equal(np.delete(f, bad), np.delete(f0, bad))
    np.testing.assert_array_equal(np.delete(e, bad), np.delete(e0, bad))


@pytest.mark.parametrize("n", [63, 64, 65, 137])
@pytest.mark.parametrize("N", [1, 63, 64, 65, 32768, 32769])
def test_field_rows_split_over_waves(n, N):
    # the field alone: rows shared by the waves of a block from 64 rows up and up
    # to 32768 targets, a wave per 64 targets otherwise
    rng = np.random.default_rng(n + N)
    m, v, c = rng.normal(size=(n, n)), rng.normal(size=(n, N)), rng.normal(size=n)
    v[3, N // 2] = np.nan  # reaches its own target only
    f = gstools_core.calc_field_krige(m, v, c)
    ok = np.arange(N) != N // 2
    assert np.isnan(f[~ok]).all()
    if N == 1:
        return
    ref = oracle.calc_field_krige(m, v[:, ok], c)
    assert np.max(np.abs(f[ok] - ref)) <= 1e-12 * _scale(m, v[:, ok], c)
    np.testing.assert_array_equal(f, gstools_core.calc_field_krige(m, v, c))


@pytest.mark.parametrize("n,N", [(400, 73_000), (700, 100_000), (1000, 70_000)])
def test_triangle_form_is_no_less_accurate(n, N):
    # the error over the lower triangle (many targets) against extended precision:
    # rms no larger than the full form's (the same targets alone; at 400 targets
    # either rms is known to about 5 %); so the field
    rng = np.random.default_rng(n)
    t = 400
    xc, xt = rng.uniform(0.0, 100.0, size=(n, 2)), rng.uniform(0.0, 100.0, size=(t, 2))
    cov = lambda a, b: np.exp(-np.hypot(*(a[:, None] - b[None]).transpose(2, 0, 1)) / 20.0)  # noqa: E731
    m = np.linalg.inv(cov(xc, xc) + 0.05 * np.eye(n))
    v, c = cov(xc, xt), rng.normal(size=n)
    w = m.T.astype(np.longdouble) @ v.astype(np.longdouble)
    refs = ((c[:, None] * w).sum(axis=0), (v * w).sum(axis=0))
    wide = np.ascontiguousarray(np.tile(v, (1, N // t + 1))[:, :N])
    tri = gstools_core.calc_field_krige_and_variance(m, wide, c)
    full = gstools_core.calc_field_krige_and_variance(m, v, c)
    assert not np.array_equal(tri[1][:t], full[1])  # two forms indeed
    for a, b, r in zip(tri, full, refs):
        rms = [float(np.sqrt(np.mean((x[:t] - r) ** 2))) for x in (a, b)]
        print(n, N, rms)
        assert rms[0] <= 1.1 * rms[1]


@pytest.mark.parametrize("n,N,tri", [(128, 100_000, False), (256, 70_000, False),
                                     (290, 28_766, False), (257, 60_001, True),
                                     (400, 50_000, True), (513, 30_011, True),
                                     (640, 42_017, True)])
def test_forms_by_size(n, N, tri):
    # the triangle form where it takes less time than the full one (one row block,
    # or unequal splits, do not), in one split or two; unsymmetric matrix
    rng = np.random.default_rng(n)
    t = 311
    m, c, v = rng.normal(size=(n, n)) + np.eye(n), rng.normal(size=n), rng.normal(size=(n, t))
    wide = np.ascontiguousarray(np.tile(v, (1, N // t + 1))[:, :N])
    f, e = gstools_core.calc_field_krige_and_variance(m, wide, c)
    f1, e1 = gstools_core.calc_field_krige_and_variance(m, v, c)
    assert np.array_equal(e[:t], e1) != tri
    rf, re = oracle.calc_field_krige_and_variance(m, v, c)
    tol = 1e-12 * n * _scale(m, v, c)
    assert np.abs(f - np.tile(rf, N // t + 1)[:N]).max() <= tol
    assert np.abs(e - np.tile(re, N // t + 1)[:N]).max() <= tol


@pytest.mark.parametrize("n,N", [(257, 60_001), (400, 73_000)])
def test_non_finite_results_of_both_forms(n, N):
    # targets whose results are not finite are those of the full form, which the
    # same targets take alone: signed infinities where all terms agree, NaN otherwise
    rng = np.random.default_rng(n)
    t = 300
    m = rng.uniform(0.5, 1.0, size=(n, n))
    v = rng.uniform(0.5, 1.0, size=(n, t))
    c = rng.uniform(0.5, 1.0, size=n)
    v[3, 7] = np.inf  # rows above it see no infinity in the triangle
    v[n - 2, 9] = -np.inf
    v[5, 130] = np.nan
    v[:, 299] *= 1e160  # the error overflows
    wide = lambda: np.ascontiguousarray(np.tile(v, (1, N // t + 1))[:, :N])  # noqa: E731
    for cond in (c, np.where(np.arange(n) == 4, np.inf, c), np.where(np.arange(n) == 4, -np.inf, c)):
        f, e = gstools_core.calc_field_krige_and_variance(m, wide(), cond)
        f1, e1 = gstools_core.calc_field_krige_and_variance(m, v, cond)
        assert np.isposinf(e1[7]) and np.isnan(e1[130]) and np.isposinf(e1[299])
        bad = ~(np.isfinite(f1) & np.isfinite(e1))
        assert bad[[7, 9, 130, 299]].all() and (bad.all() or np.isfinite(cond).all())
        np.testing.assert_array_equal(f[:t][bad], f1[bad])
        np.testing.assert_array_equal(e[:t][bad], e1[bad])
        if np.isfinite(cond).all():
            assert not np.array_equal(e[:t][~bad], e1[~bad])  # two forms indeed
        else:
            assert (f1[:5] == cond[4]).all()
    m[2, 6] = m[6, 2] = 1e308  # their sum overflows, mat and the results do not
    v = rng.uniform(0.5, 1.0, size=(n, t)) * np.where(np.arange(n) == 6, 1e-20, 1.0)[:, None]
    f, e = gstools_core.calc_field_krige_and_variance(m, wide(), c)
    f1, e1 = gstools_core.calc_field_krige_and_variance(m, v, c)
    assert np.isfinite(e1).all()
    np.testing.assert_allclose(e[:t], e1, rtol=1e-12)


@pytest.mark.parametrize("n", [20, 64, 65, 140, 298])
def test_rows_past_the_last_condition(n):
    # the full form's idle rows read the last column of the matrix: nothing of it,
    # infinities included, may reach the sums
    rng = np.random.default_rng(n)
    N = 259
    m, c, v = rng.normal(size=(n, n)), rng.normal(size=n), rng.normal(size=(n, N))
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    rf, re = oracle.calc_field_krige_and_variance(m, v, c)
    tol = 1e-12 * n * _scale(m, v, c)
    assert max(np.abs(f - rf).max(), np.abs(e - re).max()) <= tol
    m, c, v = np.abs(m), np.abs(c), np.abs(v)
    m[n // 2, n - 1] = np.inf
    c[n - 1], v[n - 1, 5] = 0.0, 0.0  # inf * 0 in every field and in one target's error
    f, e = gstools_core.calc_field_krige_and_variance(m, v, c)
    assert np.isnan(f).all() and np.isnan(e[5]) and np.isposinf(np.delete(e, 5)).all()
