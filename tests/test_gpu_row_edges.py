"""GPU: softmax, rms_norm and index_select where their row kernels change: one
wave, one workgroup or several parts per row, rows that start at any element,
and the values a mask or an overflow leaves."""
import numpy as np
import pytest

import affon_amd as A
from tests.helpers import HipRuntime, storage, widened

pytestmark = pytest.mark.gpu

# Columns around 256, 2048 and 4096 vectors (f32: 4 values, bf16: 8) and part ends; rows around the cut.
WIDTHS = [1, 3, 7, 255, 1024, 1025, 4095, 4097, 8192, 8193, 16384, 16391, 40001]


def upload(session, x, dtype):
    return session.from_bytes(x, A.TensorSpec(dtype, x.shape))


def softmax_f64(x):
    with np.errstate(invalid="ignore", over="ignore"):
        e = np.exp(x - np.fmax.reduce(x, axis=1, keepdims=True))
        return e / e.sum(1, keepdims=True)


def check(got, want, dtype):
    # f32: expf and the quotient to an ulp or two each, the sum over a few
    # levels of partial sums; bf16: that and one rounding of the result.
    rtol = 2e-6 if dtype == "f32" else 2.0 ** -8 + 2e-6
    np.testing.assert_allclose(widened(got), want, rtol=rtol, atol=1e-38)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows", [1, 5, 127, 128])
def test_row_kernels_at_their_edges(session, dtype, rows, rng):
    for cols in WIDTHS:
        x = storage(rng.standard_normal((rows, cols)) * 3, dtype)
        t, v = upload(session, x, dtype), widened(x)
        check(A.softmax(t, -1).storage(), softmax_f64(v), dtype)
        check(A.rms_norm(t, -1).storage(), v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-5), dtype)


@pytest.mark.parametrize("cols", [70, 3000, 20001])
def test_softmax_of_masks_and_specials(session, cols, rng):
    """Masked values (-inf, the type's lowest) give zeros; a row of them alone
    at -inf, a NaN and a +inf make their row NaN, as the quotient says."""
    x = rng.standard_normal((6, cols)).astype(np.float32)
    x[0, cols // 3:] = -np.inf
    x[1, : cols - 1] = np.finfo(np.float32).min
    x[2] = -np.inf
    x[3, cols // 2] = np.nan
    x[4, cols - 1] = np.inf
    x[5] = np.finfo(np.float32).min
    check(A.softmax(upload(session, x, "f32"), -1).storage(), softmax_f64(x.astype(np.float64)), "f32")


def test_softmax_captured_without_scratch(rng):
    """On a session whose workspace is empty and cannot grow, a long row runs
    in one workgroup; every replay gives the same result."""
    x = rng.standard_normal((3, 50000)).astype(np.float32)
    hip = HipRuntime()
    with A.Session("rocm") as session:
        t = upload(session, x, "f32")
        kept = []
        import ctypes
        from affon_amd import _native
        out = session.empty("f32", x.shape)
        graph = hip.capture(session.stream, lambda: kept.append(_native.load().affon_rocm_softmax(
            session._handle, ctypes.c_void_p(t.data_ptr), _native.F32, *x.shape, ctypes.c_void_p(out.data_ptr))))
        assert kept == [0], _native.last_error()
        try:
            for _ in range(3):
                hip.replay(session.stream, graph)
                check(out.storage(), softmax_f64(x.astype(np.float64)), "f32")
                A.softmax(t, -1)
                session.synchronize()
        finally:
            hip.destroy(graph)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_index_select_rows_in_pieces(session, dtype, rng):
    """Rows of whole 16-byte pieces, of elements, and more than one workgroup
    wide; indices outside select zeros."""
    for cols in (1, 8, 12, 513, 4096, 4098):
        x = storage(rng.standard_normal((9, cols)), dtype)
        index = np.array([0, 8, 9, -1, 3, 3, 2 ** 40], np.int64)
        want = np.where(((index >= 0) & (index < 9))[:, None], x[np.clip(index, 0, 8)], 0)
        got = A.index_select(upload(session, x, dtype), 0, session.tensor(index, "i64")).storage()
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_short_rows_at_the_edges_of_their_shapes(session, dtype, rng):
    """Rows of a value per lane, rows that share a wave and rows that a wave or
    a workgroup holds: columns on both sides of every line between them and
    with a part of a vector at the end, rows around the line between few and
    many and around the waves and workgroups that rows share."""
    w = 4 if dtype == "f32" else 8  # values of a vector
    short = [1, 2, w + 1, 4 * w, 4 * w + 1, 8 * w, 8 * w + 3, 64, 65, 16 * w, 16 * w + 1, 128, 129, 32 * w, 32 * w + 1,
             40 * w, 40 * w + 1]
    long = [64 * w, 64 * w + 1, 128 * w, 128 * w + 3, 256 * w, 256 * w + 1, 512 * w, 512 * w + 1, 1024 * w, 1024 * w + 1]
    for rows, widths in ((3, short + long), (8192, short), (8193, short), (8209, short[-4:] + long[:2]), (67, long)):
        for cols in widths:
            x = storage(rng.standard_normal((rows, cols)) * 3, dtype)
            x[rows // 2, cols // 2] = storage([-np.inf], dtype)[0] if cols > 1 else x[rows // 2, 0]
            t, v = upload(session, x, dtype), widened(x)
            check(A.softmax(t, -1).storage(), softmax_f64(v), dtype)
            x[rows // 2, cols // 2] = 0
            t, v = upload(session, x, dtype), widened(x)
            check(A.rms_norm(t, -1).storage(), v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-5), dtype)


@pytest.mark.parametrize("rows,cols", [(6, 20), (6, 100), (6, 200), (8196, 20), (8196, 70), (6, 1000), (6, 3000)])
def test_short_softmax_of_masks_and_specials(session, rows, cols, rng):
    """As for long rows: masked values give zeros, a NaN, a +inf or -inf alone a
    row of NaNs, and no row touches its neighbours."""
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    x[0, cols // 3:] = -np.inf
    x[1, : cols - 1] = np.finfo(np.float32).min
    x[2] = -np.inf
    x[3, cols // 2] = np.nan
    x[4, cols - 1] = np.inf
    x[5] = np.finfo(np.float32).min
    check(A.softmax(upload(session, x, "f32"), -1).storage(), softmax_f64(x.astype(np.float64)), "f32")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_index_select_of_many_rows(session, dtype, rng):
    """Rows shorter and longer than a workgroup, many of them: pieces of 16, 4
    and 2 bytes, workgroups that begin inside a row and end in another."""
    for cols in (1, 2, 3, 7, 20, 255, 256, 257, 511, 1020, 1024, 1028, 2056):
        x = storage(rng.standard_normal((301, cols)), dtype)
        index = rng.integers(-3, 305, 777)
        want = np.where(((index >= 0) & (index < 301))[:, None], x[np.clip(index, 0, 300)], 0)
        got = A.index_select(upload(session, x, dtype), 0, session.tensor(index, "i64")).storage()
        np.testing.assert_array_equal(got, want)
