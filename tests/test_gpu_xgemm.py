"""GPU: the general matrix-core kernels (f32 activations split into three bf16
planes, any group that is a multiple of 32, any K of whole groups) at the edges
of their tiles, K units and parameter windows."""
import ctypes

import numpy as np
import pytest

import affon_amd as A
from affon_amd import _native, ops
from tests.helpers import HipRuntime, pack_codes, storage, widened

pytestmark = pytest.mark.gpu

# Rows around the kernels' tiles of 16, 32, 64 and 128; columns around their 64, 128 and 256.
SHAPES = [(2, 65), (5, 1), (16, 64), (17, 63), (32, 130), (33, 127), (64, 129), (65, 300), (129, 257)]
# The same rows with columns enough that the matrix-core kernels, and not the VALU kernel, run them at every
# width of codes.
WIDE = [(2, 8200), (5, 2100), (16, 1090), (17, 1650), (32, 1030), (33, 460), (64, 300), (65, 301), (129, 257)]
# (K, group): half a step at the end, one unit and less, odd blocks per group,
# more groups than one parameter window, K ranges over workgroups; at 2 bits 96, 160, 1376 and 2592 end in
# half of a lane's 64 codes.
DEPTHS = [(64, 32), (160, 32), (96, 96), (576, 192), (1376, 32), (1344, 64), (2560, 128), (2592, 96), (4160, 64)]


def operands(rng, M, N, K, bits, group, x_dtype, p_dtype):
    q = rng.integers(0, 1 << bits, size=(N, K))
    x = storage(rng.standard_normal((M, K)), x_dtype)
    s = storage(rng.uniform(0.5, 1.5, (N, K // group)) / (1 << bits), p_dtype)
    b = storage(rng.standard_normal((N, K // group)), p_dtype)
    return x, q, s, b


def upload_all(session, x, q, s, b, bits, x_dtype, p_dtype):
    return (session.from_bytes(x, A.TensorSpec(x_dtype, x.shape)),
            session.from_bytes(pack_codes(q, bits), A.TensorSpec("u32", (q.shape[0], q.shape[1] * bits // 32))),
            session.from_bytes(s, A.TensorSpec(p_dtype, s.shape)), session.from_bytes(b, A.TensorSpec(p_dtype, b.shape)))


def runs_matrix_cores(desc):
    """Whether the gemv candidate runs the matrix-core kernels for a descriptor."""
    runs = ctypes.c_int(-1)
    _native.check(_native.load().affon_rocm_kernel_supports(ctypes.byref(desc), b"xgemm", ctypes.byref(runs)))
    return runs.value == 1


def expected_and_bound(x, q, s, b, group):
    """The product in f64, and what f32 sums of its terms may be off by: a
    term is rounded in its product with s or b and once per addition above
    it, at most one per 16 values of k in its K part, the planes' three
    chains and the parts' reduction."""
    x, s, b = (widened(v).astype(np.float64) for v in (x, s, b))
    s, b = np.repeat(s, group, 1), np.repeat(b, group, 1)
    depth = x.shape[1] / 16 + 32
    return x @ (s * q + b).T, depth * 2.0 ** -24 * (np.abs(x) @ (s * q + np.abs(b)).T)


@pytest.mark.parametrize("x_dtype,p_dtype", [("f32", "f32"), ("f32", "bf16"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_edges_against_f64(session, bits, x_dtype, p_dtype, rng):
    for i, (K, group) in enumerate(DEPTHS):
        for M, N in SHAPES[i % 2::2] if K > 600 else SHAPES:
            x, q, s, b = operands(rng, M, N, K, bits, group, x_dtype, p_dtype)
            t = upload_all(session, x, q, s, b, bits, x_dtype, p_dtype)
            out = session.tensor(np.full((M, N), np.nan, np.float32))
            A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
            want, bound = expected_and_bound(x, q, s, b, group)
            err = np.abs(out.numpy() - want)
            assert (err <= bound).all(), (M, N, K, group, float((err / bound).max()))
            # Far below the bound in norm: no plane, block or part is missing.
            assert np.linalg.norm(err) <= 2e-6 * np.linalg.norm(want), (M, N, K, group)


@pytest.mark.parametrize("x_dtype,p_dtype", [("f32", "f32"), ("f32", "bf16"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_edges_of_the_matrix_core_kernels(session, bits, x_dtype, p_dtype, rng):
    """As above, with columns enough that the matrix-core kernels run it all:
    each tile, row count and end of K, every third pair of them."""
    for i, (K, group) in enumerate(DEPTHS):
        if x_dtype == "bf16" and bits == 4 and group % 64 == 0 and K % 256 == 0:
            continue  # the direct-transfer kernels'
        for M, N in [WIDE[0]] * (K < 200) + WIDE[1 + i % 3::3]:
            x, q, s, b = operands(rng, M, N, K, bits, group, x_dtype, p_dtype)
            t = upload_all(session, x, q, s, b, bits, x_dtype, p_dtype)
            out = session.tensor(np.full((M, N), np.nan, np.float32))
            desc = ops._descriptor(*t, bits, group, out, "gemv", "backend_equivalent")
            assert runs_matrix_cores(desc), (M, N, K, group)
            A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
            want, bound = expected_and_bound(x, q, s, b, group)
            err = np.abs(out.numpy() - want)
            assert (err <= bound).all(), (M, N, K, group, float((err / bound).max()))
            assert np.linalg.norm(err) <= 2e-6 * np.linalg.norm(want), (M, N, K, group)


@pytest.mark.parametrize("M", [3, 40, 200])
def test_extreme_activations(session, M):
    """One nonzero activation per row: the largest finite f32 (no plane
    overflows), one with all 24 bits set, a small normal one, infinities and a
    NaN; codes 1 with scale 2^-10 and bias 0 give x * 2^-10 exactly."""
    N, K, group = 70, 320, 64
    values = np.array([np.finfo(np.float32).max, np.float32(1.0 + 2.0 ** -23), -np.float32(2.0 ** -100 * (2 - 2.0 ** -23)),
                       np.inf, -np.inf, np.nan], np.float32)
    x = np.zeros((M, K), np.float32)
    picked = values[np.arange(M) % len(values)]
    x[np.arange(M), np.arange(M) * 7 % K] = picked
    q, s, b = np.ones((N, K), np.int64), np.full((N, K // group), 2.0 ** -10, np.float32), np.zeros((N, K // group), np.float32)
    t = upload_all(session, x, q, s, b, 4, "f32", "f32")
    out = session.empty("f32", (M, N))
    A.quantized_matmul_into(out, *t, bits=4, group_size=group, implementation="gemv")
    # The bias term 0 * sum(x) makes an infinite row NaN, as on the VALU kernel.
    want = np.where(np.isfinite(picked), picked * np.float32(2.0 ** -10), np.nan).astype(np.float32)
    np.testing.assert_array_equal(out.numpy(), np.broadcast_to(want[:, None], (M, N)))
    # With a positive bias an infinite row stays infinite.
    t = t[:3] + (session.tensor(np.full_like(b, 0.25)),)
    A.quantized_matmul_into(out, *t, bits=4, group_size=group, implementation="gemv")
    rows = np.isinf(picked)
    np.testing.assert_array_equal(out.numpy()[rows], np.broadcast_to(picked[rows, None], (rows.sum(), N)))


@pytest.mark.parametrize("M", [3, 40, 200])
def test_smallest_activations(session, M):
    """One nonzero f32 activation per row: its planes hold what of it lies above
    2^-133, the smallest bf16 value, so that all bits are there from 2^-110 on;
    below, the error stays under 2^-133."""
    N, K, group = 70, 320, 64
    picked = np.array([2.0 ** -109 * (2 - 2.0 ** -23), -(2.0 ** -118) * (2 - 2.0 ** -23), 2.0 ** -126, 2.0 ** -130, 2.0 ** -149],
                      np.float32)[np.arange(M) % 5]
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), np.arange(M) * 7 % K] = picked
    q, s, b = np.ones((N, K), np.int64), np.full((N, K // group), 2.0 ** 30, np.float32), np.zeros((N, K // group), np.float32)
    t = upload_all(session, x, q, s, b, 4, "f32", "f32")
    out = session.empty("f32", (M, N))
    A.quantized_matmul_into(out, *t, bits=4, group_size=group, implementation="gemv")
    err = np.abs(out.numpy() * 2.0 ** -30 - picked[:, None].astype(np.float64))
    assert (err < 2.0 ** -133).all() and (err[np.abs(picked) >= 2.0 ** -110] == 0).all()


@pytest.mark.parametrize("M", [6, 24, 100, 300])
def test_epilogues_and_repeats(session, M, rng):
    """Output bias and SiLU-gated product through the K ranges' reduction and
    without it; repeated runs are bit-identical."""
    for N, K in ((200, 4096), (96, 192)):
        x, q, s, b = operands(rng, M, N, K, 4, 64, "f32", "f32")
        t = upload_all(session, x, q, s, b, 4, "f32", "f32")
        y = A.quantized_matmul(*t, bits=4, group_size=64).numpy()
        np.testing.assert_array_equal(A.quantized_matmul(*t, bits=4, group_size=64).numpy(), y)
        bias = rng.standard_normal(N).astype(np.float32)
        fused = A.quantized_linear(*t, session.tensor(bias), bits=4, group_size=64).numpy()
        np.testing.assert_array_equal(fused, y + bias)
        _, q2, s2, b2 = operands(rng, M, N, K, 4, 64, "f32", "f32")
        up = upload_all(session, x, q2, s2, b2, 4, "f32", "f32")
        u = A.quantized_matmul(*up, bits=4, group_size=64).numpy().astype(np.float64)
        g = y.astype(np.float64)
        want = g / (1 + np.exp(-g)) * u
        got = A.quantized_silu_gate(t[0], t[1:], up[1:], bits=4, group_size=64).numpy()
        # expf, the division and the product: a few roundings of the result.
        assert (np.abs(got - want) <= 8 * 2.0 ** -24 * np.abs(want) + 1e-30).all()


@pytest.mark.parametrize("M", [8, 128])
def test_capture_without_scratch(M, rng):
    """Captured on a session whose workspace is still empty, the product runs
    in one K range; replays give the same bits each time, within the bound."""
    N, K, group = {8: 4400, 128: 1056}[M], 4160, 64
    x, q, s, b = operands(rng, M, N, K, 8, group, "f32", "bf16")
    hip = HipRuntime()
    with A.Session("rocm") as session:
        t = upload_all(session, x, q, s, b, 8, "f32", "bf16")
        out = session.empty("f32", (M, N))
        desc = ops._descriptor(*t, 8, group, out, "auto", "backend_equivalent")
        assert runs_matrix_cores(desc)
        lib = _native.load()

        def enqueue():
            assert lib.affon_rocm_quantized_matmul(session._handle, ctypes.byref(desc)) == 0, _native.last_error()

        graph = hip.capture(session.stream, enqueue)
        try:
            want, bound = expected_and_bound(x, q, s, b, group)
            first = None
            for _ in range(3):
                zeros = np.zeros((M, N), np.float32)
                _native.check(lib.affon_rocm_memcpy_h2d(session._handle, out.data_ptr, zeros.ctypes.data, zeros.nbytes),
                              "clear")
                hip.replay(session.stream, graph)
                session.synchronize()
                got = out.numpy()
                assert (np.abs(got - want) <= bound).all()
                first = got if first is None else first
                np.testing.assert_array_equal(got, first)
                A.quantized_matmul(*t, bits=8, group_size=group)
        finally:
            hip.destroy(graph)


@pytest.mark.parametrize("M", [3, 40, 200])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_bf16_products_start_from_their_sums(session, bits, M):
    """bf16 activations: rows of one value, whose products and sums are all
    exact, so that nothing of the start -2^(bits-1) * sum(x) may remain; an
    infinite row stays infinite with positive scales and biases."""
    N, K, group = 70 if bits == 4 else 8200, 320, 32
    x = np.zeros((M, K), np.float32)
    picked = np.array([1.5, -2.0 ** 60, np.inf, -np.inf, np.nan, 2.0 ** -100], np.float32)[np.arange(M) % 6]
    x[np.arange(M), np.arange(M) * 7 % K] = picked
    q = np.full((N, K), (1 << bits) - 1, np.int64)
    s, b = np.full((N, K // group), 2.0 ** -10, np.float32), np.full((N, K // group), 0.25, np.float32)
    t = upload_all(session, storage(x, "bf16"), q, s, b, bits, "bf16", "f32")
    out = session.empty("f32", (M, N))
    assert runs_matrix_cores(ops._descriptor(*t, bits, group, out, "gemv", "backend_equivalent"))
    A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
    want = picked * np.float32(q[0, 0] * 2.0 ** -10 + 0.25)
    np.testing.assert_array_equal(out.numpy(), np.broadcast_to(want[:, None], (M, N)))


@pytest.mark.parametrize("M,N", [(2, 1), (3, 1), (2, 3), (33, 1), (35, 3), (33, 67), (40, 64)])
def test_reductions_of_many_ranges(session, M, N, rng):
    """32 K ranges and their ordered sum, for counts of outputs below four and
    of every remainder by four."""
    K, bits, group = 16384, 4, 64
    x, q, s, b = operands(rng, M, N, K, bits, group, "f32", "f32")
    t = upload_all(session, x, q, s, b, bits, "f32", "f32")
    out = session.tensor(np.full((M, N), np.nan, np.float32))
    assert runs_matrix_cores(ops._descriptor(*t, bits, group, out, "gemv", "backend_equivalent"))
    A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
    want, bound = expected_and_bound(x, q, s, b, group)
    err = np.abs(out.numpy() - want)
    assert (err <= bound).all() and np.linalg.norm(err) <= 2e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("bits,group,x_dtype,K", [(8, 64, "f32", 8192), (8, 64, "f32", 8256), (2, 32, "bf16", 2624),
                                                  (4, 32, "bf16", 2048), (4, 32, "bf16", 2080), (4, 32, "bf16", 8224)])
def test_sides_of_the_few_passes_rule(session, bits, group, x_dtype, K, rng):
    """Rows and columns on both sides of the lines between the VALU and the
    matrix-core kernels."""
    for M, N in ((2, 70), (4, 2048), (5, 1024), (5, 1025), (8, 2048), (8, 2049)):
        x, q, s, b = operands(rng, M, N, K, bits, group, x_dtype, "bf16")
        t = upload_all(session, x, q, s, b, bits, x_dtype, "bf16")
        out = session.tensor(np.full((M, N), np.nan, np.float32))
        A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
        want, bound = expected_and_bound(x, q, s, b, group)
        err = np.abs(out.numpy() - want)
        assert (err <= bound).all() and np.linalg.norm(err) <= 2e-6 * np.linalg.norm(want), (M, N)


LOWEST_BF16 = -(2.0 ** 127) * (2 - 2.0 ** -7)


@pytest.mark.parametrize("M,N,K", [(5, 2060, 352), (24, 1030, 352), (70, 1030, 352), (130, 2060, 16032)])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_large_bf16_activations(session, bits, M, N, K):
    """Where 2^(bits-1) * sum(x) or a group's 2^(bits-1) * scale overflows, on
    every kernel: one nonzero activation per row, negative, zero and positive
    biases, codes on both sides of the middle. A result that f32 holds as
    s * (q*x) + b*x lies within its terms' roundings; a row that is infinite
    gives its true sign or, where the two terms' signs differ, a NaN; no row
    changes another."""
    group, c = 32, 2.0 ** (bits - 1)
    picked = np.array([LOWEST_BF16, -LOWEST_BF16, 2.0 ** 121, -2.0 ** 122, 2.0 ** 123, 2.0 ** 124, -2.0 ** 125, 2.0 ** 126,
                       np.inf, -np.inf, np.nan, 1.5, -2.0 ** 60])[np.arange(M) % 13]
    at = np.arange(M) * 37 % K
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), at] = picked
    q = np.arange(N) % (1 << bits)  # a column's code
    large = np.arange(N) % 5 == 4  # scales whose 2^(bits-1) times overflows at 8 bits
    s = np.where(large, 2.0 ** 122, 2.0 ** -10)
    b = s * np.where(large, 0.25, np.array([-(c - 0.5), 0.0, 0.25, -0.5 - c, c])[np.arange(N) // 3 % 5])
    t = (session.from_bytes(storage(x, "bf16"), A.TensorSpec.bf16((M, K))),
         session.from_bytes(np.repeat(pack_codes(np.repeat(q[:, None], 32 // bits, 1), bits), K * bits // 32, 1),
                            A.TensorSpec.u32((N, K * bits // 32))),
         *(session.from_bytes(storage(np.repeat(v[:, None], K // group, 1), "f32"), A.TensorSpec.f32((N, K // group)))
           for v in (s, b)))
    out = session.tensor(np.full((M, N), 7.0, np.float32))
    A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
    got, v = out.numpy(), picked[:, None]
    assert runs_matrix_cores(ops._descriptor(*t, bits, group, out, "gemv", "backend_equivalent"))
    with np.errstate(over="ignore", invalid="ignore"):
        qx, bx = (q * v).astype(np.float32), (b * v).astype(np.float32)
        plain = s.astype(np.float32) * qx + bx
        exact = (s * q + b) * v
        bound = 4 * 2.0 ** -24 * (s * (q + 2 * c) + 2 * np.abs(b)) * np.abs(v)
        held = np.isfinite(plain)
        assert held.any() and (np.abs(got.astype(np.float64) - exact)[held] <= bound[held]).all()
        infinite = np.isinf(v) & (s * q + b != 0)
        assert (np.isnan(got) | (got == exact))[infinite].all()
    assert (got == exact)[infinite & (b * q > 0)].all()  # both terms of one sign
    assert np.isnan(got[np.isnan(picked)]).all()


@pytest.mark.parametrize("M,N,bits", [(8, 1030, 4), (24, 1030, 4), (40, 256, 4), (40, 2200, 4), (130, 1500, 8)])
def test_capture_without_scratch_on_both_sides(M, N, bits, rng):
    """Captured on a session whose workspace is still empty: one K range, or
    the VALU kernel where that is ahead of it (few columns for K); eager calls
    then take several ranges. Every replay gives the same bits, within the bound."""
    K, group = 4160, 64
    x, q, s, b = operands(rng, M, N, K, bits, group, "f32", "f32")
    hip = HipRuntime()
    with A.Session("rocm") as session:
        t = upload_all(session, x, q, s, b, bits, "f32", "f32")
        out = session.tensor(np.full((M, N), np.nan, np.float32))
        desc = ops._descriptor(*t, bits, group, out, "auto", "backend_equivalent")
        assert runs_matrix_cores(desc)
        lib = _native.load()

        def enqueue():
            assert lib.affon_rocm_quantized_matmul(session._handle, ctypes.byref(desc)) == 0, _native.last_error()

        graph = hip.capture(session.stream, enqueue)
        try:
            want, bound = expected_and_bound(x, q, s, b, group)
            hip.replay(session.stream, graph)
            first = out.numpy()
            assert (np.abs(first - want) <= bound).all()
            for _ in range(2):
                enqueue()
                assert (np.abs(out.numpy() - want) <= bound).all()
                hip.replay(session.stream, graph)
                np.testing.assert_array_equal(out.numpy(), first)
        finally:
            hip.destroy(graph)


@pytest.mark.parametrize("bits", [2, 4, 8])
def test_errors_of_many_rows_have_no_sign(session, bits, rng):
    """f32 activations at groups of 32 in tiles of 64 rows: the products round
    down, and the steps' errors must cancel instead of adding up. Of n errors
    without a sign the mean is about rms / sqrt(n), here with what the outputs
    of a row and a column share; rounding down alone gives 0.8 rms."""
    M, N, K, group = 260, 512, 8960, 32
    x, q, _, _ = operands(rng, M, N, K, bits, group, "f32", "f32")
    s = np.full((N, K // group), 0.02 / (1 << bits), np.float32)
    b = np.float32(-0.5 * ((1 << bits) - 1)) * s
    t = upload_all(session, x, q, s, b, bits, "f32", "f32")
    out = session.empty("f32", (M, N))
    assert runs_matrix_cores(ops._descriptor(*t, bits, group, out, "gemv", "backend_equivalent"))
    A.quantized_matmul_into(out, *t, bits=bits, group_size=group, implementation="gemv")
    want, _ = expected_and_bound(x, q, s, b, group)
    err = out.numpy() - want
    assert abs(err.mean()) <= 0.2 * np.sqrt((err ** 2).mean())
    assert np.linalg.norm(err) <= 2.6e-7 * np.linalg.norm(want)
