"""int8-mode calls of 17 to 63 tokens in one launch: the same bits as the
register-staged kernel's 16-token launches, at the edges of its tiles (rows of
64, gated 32; token tiles of 16), of its column chunks (one block, fewer than
eight, an odd number, not a multiple of eight), with its tiles whole and with
their chunks split over workgroups, fused and gated. The oracle side is
test_i8_mode_batched (17 and 35 tokens) and the block-dot routes (40)."""
import numpy as np
import pytest

import mdma_amd.backend as bm
from mdma_amd import synth
from mdma_amd.backend import Gfx950Backend

pytestmark = pytest.mark.gpu
Q8, Q4K, Q6K = 8, 12, 14
CANARY = np.float32(123456.25)


@pytest.fixture
def i8(backend):
    backend.set_act_mode(bm.ACT_I8)
    yield backend
    backend.set_act_mode(bm.ACT_F32)


def both(be, sizes, call):
    """call(outs) with the AUTO and the STAGED kernel: the outputs' bits."""
    got = []
    for kind in (bm.BATCH_AUTO, bm.BATCH_STAGED):
        be.set_batch_kernel(kind)
        outs = [be.f32_buf(np.full(n + 8, CANARY, np.float32)) for n in sizes]
        call(outs)
        res = [be.download_f32(o) for o in outs]
        for r, n in zip(res, sizes):
            assert np.all(r[n:] == CANARY), "wrote past the output"
        got.append(np.concatenate([r[:n] for r, n in zip(res, sizes)]).view(np.uint32))
    be.set_batch_kernel(bm.BATCH_AUTO)
    return got


@pytest.mark.parametrize("dtype", [Q4K, Q6K, Q8])
@pytest.mark.parametrize("rows,k", [((1, 64, 65), 256), ((129, 16, 63), 1280), ((96, 32, 32), 4096), ((70, 1, 1), 14336),
                                    ((16500, 40, 8), 768)])
@pytest.mark.parametrize("T", [17, 19, 34, 35, 48, 63])
def test_projections_equal_staged(i8, dtype, rows, k, T):
    ws = [i8.upload_weight(synth.weight(dtype, r, k, 7 + r, True), dtype, (r, k)) for r in rows]
    x = i8.f32_buf(synth.normal_f32(T * k, T + k))
    a, b = both(i8, [T * r for r in rows], lambda o: i8.qmatmul_qkv(*ws, x, *o))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype", [Q4K, Q6K, Q8])
@pytest.mark.parametrize("rows,k", [(33, 768), (200, 4096), (8300, 512)])
@pytest.mark.parametrize("T", [18, 19, 32, 49, 51])
def test_gate_up_equal_staged(i8, dtype, rows, k, T):
    ws = [i8.upload_weight(synth.weight(dtype, rows, k, s, True), dtype, (rows, k)) for s in (1, 2)]
    x = i8.f32_buf(synth.normal_f32(T * k, T) * 0.1)
    gs, us = i8.alloc(T * rows * 4), i8.alloc(T * rows * 4)
    a, b = both(i8, [T * rows], lambda o: i8.ffn_gate_up(ws[0], ws[1], x, gs, us, o[0]))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("T", [17, 18, 40, 50])
def test_captured_call_gives_the_eager_bits(T):
    # A capture has no space for the chunk sums: 16 tokens a launch, the last
    # one or two included.
    be = Gfx950Backend(0)
    be.set_act_mode(bm.ACT_I8)
    rows, k = 200, 2048
    w = be.upload_weight(synth.weight(Q6K, rows, k, 1, True), Q6K, (rows, k))
    x, y = be.f32_buf(synth.normal_f32(T * k, 2)), be.alloc(T * rows * 4)
    be.qmatmul(w, x, y)
    ref = be.download_f32(y)
    graph = be.capture(lambda: be.qmatmul(w, x, y))
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        graph.launch()
        assert np.array_equal(be.download_f32(y).view(np.uint32), ref.view(np.uint32))
    graph.close()
    be.close()


def test_captured_and_over_budget_run_unsplit():
    # No space for the split tiles' chunk sums: 16 tokens a launch, the same bits.
    be = Gfx950Backend(0)
    be.set_act_mode(bm.ACT_I8)
    rows, k, T = 256, 2048, 40
    be.set_buffer_budget(device=64 << 20)
    w = be.upload_weight(synth.weight(Q4K, rows, k, 1, True), Q4K, (rows, k))
    x, y, want = be.f32_buf(synth.normal_f32(T * k, 2)), be.alloc(T * rows * 4), be.alloc(T * rows * 4)
    be.set_batch_kernel(bm.BATCH_STAGED)
    be.qmatmul(w, x, want)
    ref = be.download_f32(want)
    be.set_batch_kernel(bm.BATCH_AUTO)
    graph = be.capture(lambda: be.qmatmul(w, x, y))
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        graph.launch()
        assert np.array_equal(be.download_f32(y), ref)
    used, limit = be.buffer_usage(bm.DOMAIN_DEVICE)
    be.qmatmul(w, x, y)  # split
    assert be.buffer_usage(bm.DOMAIN_DEVICE)[0] > used
    assert np.array_equal(be.download_f32(y), ref)
    rest = be.alloc(limit - used)  # the split's space gives way
    be.upload(y, 0, np.zeros(T * rows, np.float32))
    be.qmatmul(w, x, y)
    assert np.array_equal(be.download_f32(y), ref)
    rest.close()
    graph.close()
    be.close()


def test_int8_buffer_is_not_grown_past_16_tokens():
    # 63 tokens of 14336 values do not fit the int8 buffer's first megabyte,
    # 16 do: the call neither grows it (under a capture or a full budget it
    # could not, and growth ends graphs) nor refuses.
    be = Gfx950Backend(0)
    be.set_act_mode(bm.ACT_I8)
    be.set_buffer_budget(device=64 << 20)
    rows, k, T = 100, 14336, 63
    w = be.upload_weight(synth.weight(Q6K, rows, k, 1, True), Q6K, (rows, k))
    x, y, want = be.f32_buf(synth.normal_f32(T * k, 2)), be.alloc(T * rows * 4), be.alloc(T * rows * 4)
    be.reserve_scratch(1 << 19)
    be.set_batch_kernel(bm.BATCH_STAGED)
    be.qmatmul(w, x, want)
    ref = be.download_f32(want)
    be.set_batch_kernel(bm.BATCH_AUTO)
    graph = be.capture(lambda: be.qmatmul(w, x, y))

    def same(call):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        call()
        assert np.array_equal(be.download_f32(y), ref)

    used, limit = be.buffer_usage(bm.DOMAIN_DEVICE)
    rest = be.alloc(limit - used)
    for _ in range(2):
        same(lambda: be.qmatmul(w, x, y))  # a full budget: 16 tokens a launch
        same(graph.launch)
    rest.close()
    for _ in range(2):
        same(lambda: be.qmatmul(w, x, y))  # one launch, its int8 form beside the chunk sums
        same(graph.launch)
    assert be.buffer_usage(bm.DOMAIN_DEVICE)[0] > used
    be.reserve_scratch(8 << 20)
    graph.close()
    graph = be.capture(lambda: be.qmatmul(w, x, y))  # one launch, in the scratch
    for _ in range(3):
        same(graph.launch)
        same(lambda: be.qmatmul(w, x, y))
    graph.close()
    be.close()


@pytest.mark.parametrize("room", [100, 300])
def test_int8_buffer_and_chunk_sums_on_a_budget(room):
    # A first call with room for the int8 buffer's megabyte and little more: the
    # chunk sums' 192 KB fit beside it or not, and neither takes the other's.
    be = Gfx950Backend(0)
    be.set_act_mode(bm.ACT_I8)
    rows, k, T = 100, 2048, 40
    raw = synth.weight(Q4K, rows, k, 1, True)
    be.set_buffer_budget(device=64 << 20)
    w = be.upload_weight(raw, Q4K, (rows, k))
    x, y = be.f32_buf(synth.normal_f32(T * k, 2)), be.alloc(T * rows * 4)
    used, limit = be.buffer_usage(bm.DOMAIN_DEVICE)
    rest = be.alloc(limit - used - (1 << 20) - (room << 10))
    got = []
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        be.qmatmul(w, x, y)
        got.append(be.download_f32(y).view(np.uint32))
    free = limit - be.buffer_usage(bm.DOMAIN_DEVICE)[0]
    assert (free == room << 10) if room < 192 else (free < room << 10)
    rest.close()
    be.set_batch_kernel(bm.BATCH_STAGED)
    be.qmatmul(w, x, y)
    assert all(np.array_equal(g, be.download_f32(y).view(np.uint32)) for g in got)
    be.close()
