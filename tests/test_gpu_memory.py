"""GPU: memory that a session keeps between allocations is bounded, is handed
out again only when nothing can still use it, and is given back."""
import ctypes
import gc
import threading

import numpy as np
import pytest

import affon_amd as A
from affon_amd import _native, ops
from affon_amd.decoder import QuantizedDecoderBlock
from tests.helpers import HipRuntime
from tests.test_gpu_decoder import BITS, GROUP, SHAPE, block_checkpoint

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def raw_alloc(session, nbytes):
    ptr = ctypes.c_void_p()
    _native.check(_native.load().affon_rocm_alloc(session._handle, nbytes, ctypes.byref(ptr)), "alloc")
    return ptr.value


def test_kept_memory_is_bounded_and_given_back():
    hip = HipRuntime()
    with A.Session("rocm") as session:
        lib = _native.load()
        before = hip.free_bytes()
        for size in (200 * MIB, 120 * MIB, 300 * MIB, 7 * MIB):  # 300 MiB: over what is kept
            blocks = [raw_alloc(session, size) for _ in range(6)]
            assert len(set(blocks)) == 6
            for b in blocks:
                assert lib.affon_rocm_free(session._handle, b) == 0
            assert hip.free_bytes() >= before - 1100 * MIB, size
        # Freed once: not this session's any more, whether kept or not.
        assert lib.affon_rocm_free(session._handle, blocks[0]) == _native.CORE_FAILURE
    assert hip.free_bytes() >= before - 64 * MIB


def test_held_results_keep_their_values(session, rng):
    """A loop of products whose results are dropped two rounds later, so that
    their memory goes round: those still held keep their values."""
    x = session.tensor(rng.standard_normal((64, 4096)).astype(np.float32))
    w = A.quantize(session.tensor(rng.standard_normal((4096, 4096)).astype(np.float32)), bits=4, group_size=64,
                   param_dtype="f32")
    want = A.quantized_matmul(x, *w, bits=4, group_size=64).numpy()
    recent = []
    for i in range(60):
        recent.append(A.quantized_matmul(x, *w, bits=4, group_size=64))
        if len(recent) > 2:
            recent.pop(0)
        if i % 20 == 19:
            for t in recent:
                np.testing.assert_array_equal(t.numpy(), want)


def test_frees_from_other_threads(session):
    """Tensors dropped on other threads while this one allocates: addresses of
    live tensors never coincide, and their contents stay."""
    stop, errors = threading.Event(), []
    dropped = []

    def drop():
        while not stop.is_set():
            try:
                dropped.pop(0)
            except IndexError:
                pass
            except Exception as e:  # noqa: BLE001 - reported below
                errors.append(e)

    threads = [threading.Thread(target=drop) for _ in range(2)]
    for t in threads:
        t.start()
    try:
        live = []
        for i in range(400):
            t = session.tensor(np.full(1000 + i % 3, i, np.float32))
            live.append((i, t))
            assert len({v._buffer.ptr for _, v in live}) == len(live)
            if len(live) > 8:
                j, old = live.pop(0)
                assert (old.numpy() == j).all()
                dropped.append(old)
                del old
    finally:
        stop.set()
        for t in threads:
            t.join()
        dropped.clear()
        gc.collect()
    assert not errors


def test_memory_of_a_captured_program_stays_its_own(tmp_path, rng):
    """A captured feed-forward frees its gated product inside the region, and
    its output is dropped after it. Every replay writes to both: tensors made
    since then keep their values."""
    hip, rows = HipRuntime(), 32
    path, _ = block_checkpoint(tmp_path)
    with A.Session("rocm") as session:
        block = QuantizedDecoderBlock.from_checkpoint(session, path, 3, SHAPE, bits=BITS, group_size=GROUP)
        x = session.from_bytes(A.core.bf16_bits(rng.standard_normal((rows, SHAPE.width)).astype(np.float32)),
                               A.TensorSpec.bf16((rows, SHAPE.width)))
        want = block.feed_forward(x).numpy()
        for _ in range(3):
            block.feed_forward(x)
            session.synchronize()
        # Blocks of both sizes are ready to be handed out within the region.
        for width in (SHAPE.inner_width, SHAPE.width):
            session.empty("f32", (rows, width))
        kept = []
        graph = hip.capture(session.stream, lambda: kept.append(block.feed_forward(x)))
        try:
            hip.replay(session.stream, graph)
            np.testing.assert_array_equal(kept[0].numpy(), want)
            kept.clear()
            session.synchronize()
            tensors = [session.tensor(np.full((rows, width), i, np.float32))
                       for i in range(24) for width in (SHAPE.inner_width, SHAPE.width)]
            for _ in range(3):
                hip.replay(session.stream, graph)
                block.feed_forward(x)
                for i, t in enumerate(tensors):
                    assert (t.numpy() == i // 2).all(), i
        finally:
            hip.destroy(graph)


def test_memory_used_on_another_stream(rng):
    """A block freed while another session's stream still writes to it is
    handed out only after that work has ended."""
    M, N, K = 512, 4096, 4096
    with A.Session("rocm") as one, A.Session("rocm") as other:
        x = other.tensor(rng.standard_normal((M, K)).astype(np.float32))
        w = A.quantize(other.tensor(rng.standard_normal((N, K)).astype(np.float32)), bits=4, group_size=64,
                       param_dtype="f32")
        A.quantized_matmul(x, *w, bits=4, group_size=64)
        other.synchronize()
        block = raw_alloc(one, M * N * 4)
        desc = ops._descriptor(x, *w, 4, 64, None, "auto", "backend_equivalent")
        desc.output, desc.output_bytes = block, M * N * 4
        for _ in range(100):  # some milliseconds
            assert _native.load().affon_rocm_quantized_matmul(other._handle, ctypes.byref(desc)) == 0
        assert _native.load().affon_rocm_free(one._handle, block) == 0
        tensors = [one.tensor(np.full((M, N), i, np.float32)) for i in range(3)]
        other.synchronize()
        for i, t in enumerate(tensors):
            assert (t.numpy() == i).all()


def test_scratch_between_threads(session, rng):
    """Calls that keep partial results in the session's scratch memory between
    two launches (softmax of few long rows, a batch in K ranges), from two
    threads at once: each gets the result that it gets alone."""
    errors = []

    def softmax(seed):
        x = session.tensor(np.random.default_rng(seed).standard_normal((3, 40000)).astype(np.float32))
        return lambda: A.softmax(x, -1).numpy()

    def batch(seed):
        r = np.random.default_rng(seed)
        x = session.tensor(r.standard_normal((40, 4096)).astype(np.float32))
        w = A.quantize(session.tensor(r.standard_normal((512, 4096)).astype(np.float32)), bits=4, group_size=64,
                       param_dtype="f32")
        return lambda: A.quantized_matmul(x, *w, bits=4, group_size=64).numpy()

    calls = [softmax(1), batch(2), softmax(3), batch(4)]
    alone = [call() for call in calls]

    def work(mine):
        try:
            for _ in range(100):
                for i in mine:
                    np.testing.assert_array_equal(calls[i](), alone[i])
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(mine,)) for mine in ((0, 1), (2, 3))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_capture_beside_another_sessions_work(rng):
    """A capture on one session's stream while another session allocates, takes
    its first scratch memory, runs and drops results, on the same thread: the
    capture ends well, and replays give the eager result."""
    hip = HipRuntime()
    with A.Session("rocm") as one, A.Session("rocm") as other:
        x = one.tensor(rng.standard_normal((8, 1024)).astype(np.float32))
        w = A.quantize(one.tensor(rng.standard_normal((512, 1024)).astype(np.float32)), bits=4, group_size=64,
                       param_dtype="f32")
        out = one.empty("f32", (8, 512))
        run = lambda: A.quantized_matmul_into(out, x, *w, bits=4, group_size=64)
        run()
        want = out.numpy()
        rows = other.tensor(rng.standard_normal((3, 40000)).astype(np.float32))  # takes scratch memory

        def enqueue():
            run()
            for i in range(40):
                result = A.softmax(rows, -1)
                if i % 10 == 9:
                    result.numpy()
            run()

        graph = hip.capture(one.stream, enqueue)
        try:
            for _ in range(3):
                _native.check(_native.load().affon_rocm_memcpy_h2d(
                    one._handle, out.data_ptr, np.zeros_like(want).ctypes.data, want.nbytes), "clear")
                hip.replay(one.stream, graph)
                np.testing.assert_array_equal(out.numpy(), want)
                A.softmax(rows, -1)
        finally:
            hip.destroy(graph)
