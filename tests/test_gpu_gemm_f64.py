"""The f32 mode's several-token kernels (f64 matrix cores) at the sizes where
their tiles, blocks and work split have remainders, against the f64 dot
product of the dequantized weights: every output must be as close to it as the
CPU's sequential f32 sum is (assert_parity, correctly_rounded), which a sum in
f64 rounded once meets."""
import numpy as np
import pytest

import npq
from conftest import assert_parity, f32_exact
from mdma_amd import synth
from mdma_amd.backend import DOMAIN_DEVICE, BackendError, Gfx950Backend
from oracle import ffi

pytestmark = pytest.mark.gpu
Q8, Q4K, Q6K = 8, 12, 14
CANARY = np.float32(123456.25)


def out_buf(be, n):
    return be.f32_buf(np.full(n + 8, CANARY, np.float32))


def check(be, buf, T, dtype, raw, rows, k, x, what):
    got = be.download_f32(buf)
    assert np.all(got[T * rows:] == CANARY), f"{what}: wrote past the output"
    exact = f32_exact(npq.dequantize(dtype, raw, rows, k), x)
    assert_parity(got[:T * rows], ffi.qmatmul(dtype, raw, rows, k, x), exact, 1e-5, what=what, correctly_rounded=True)


@pytest.mark.parametrize("dtype,k", [(Q4K, 256), (Q4K, 2304), (Q6K, 256), (Q6K, 2560), (Q8, 32), (Q8, 288), (Q8, 2048)])
@pytest.mark.parametrize("T", [2, 4, 5, 8, 9, 16, 17, 33, 49, 64, 65, 130])
def test_projections_at_tile_edges(backend, dtype, k, T):
    # Three jobs per launch: one row, one tile of rows and one more, several.
    rows = (129, 1, 300)
    raws = [synth.weight(dtype, r, k, 3 * r + k, True) for r in rows]
    x = synth.normal_f32(T * k, T + k)
    outs = [out_buf(backend, T * r) for r in rows]
    backend.qmatmul_qkv(*(backend.upload_weight(raw, dtype, (r, k)) for raw, r in zip(raws, rows)),
                        backend.f32_buf(x), *outs)
    for raw, r, o in zip(raws, rows, outs):
        check(backend, o, T, dtype, raw, r, k, x, f"dtype={dtype} k={k} T={T} rows={r}")


@pytest.mark.parametrize("dtype,k", [(Q4K, 1280), (Q6K, 512), (Q8, 288)])
@pytest.mark.parametrize("T", [2, 4, 7, 16, 40, 100])
def test_gate_up_at_tile_edges(backend, dtype, k, T):
    # silu(gate) * up of outputs rounded once: equal to the separate calls' up
    # to the few ulps of silu_mul's own roundings.
    rows = 97
    raws = [synth.weight(dtype, rows, k, s, True) for s in (5, 6)]
    w = [backend.upload_weight(r, dtype, (rows, k)) for r in raws]
    x = backend.f32_buf(synth.normal_f32(T * k, T) * 0.1)
    g, u, gs, us = (backend.alloc(T * rows * 4) for _ in range(4))
    y, want = out_buf(backend, T * rows), backend.alloc(T * rows * 4)
    backend.ffn_gate_up(w[0], w[1], x, gs, us, y)
    backend.qmatmul(w[0], x, g)
    backend.qmatmul(w[1], x, u)
    backend.silu_mul(g, u, want)
    got, ref = backend.download_f32(y), backend.download_f32(want)
    assert np.all(got[T * rows:] == CANARY)
    assert np.allclose(got[:T * rows], ref, rtol=6 * 2.0**-24, atol=0)


@pytest.mark.parametrize("rows,T", [(200, 70), (200, 9), (200, 128), (200, 129), (16700, 12)])
def test_captured_launch_without_partials_space(rows, T):
    # Under capture the partial tiles' space cannot be made: the launch takes 8
    # tokens at a time (and a last one alone), or whole tiles where these are
    # many or the tokens more than 128, and its replays give the eager results.
    be = Gfx950Backend(0)
    k = 1024
    raw = synth.weight(Q6K, rows, k, 1, True)
    w, x_h = be.upload_weight(raw, Q6K, (rows, k)), synth.normal_f32(T * k, 2)
    x, y = be.f32_buf(x_h), out_buf(be, T * rows)
    graph = be.capture(lambda: be.qmatmul(w, x, y))
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        be.qmatmul(w, x, be.alloc(T * rows * 4))  # eager: makes the space; the graph does not hold it
        graph.launch()
        check(be, y, T, Q6K, raw, rows, k, x_h, "captured")
    graph.close()
    be.close()


@pytest.mark.parametrize("T", [9, 23])
def test_captured_gate_up_without_partials_space(T):
    be = Gfx950Backend(0)
    rows, k = 150, 1024
    w = [be.upload_weight(synth.weight(Q4K, rows, k, s, True), Q4K, (rows, k)) for s in (5, 6)]
    x = be.f32_buf(synth.normal_f32(T * k, T) * 0.1)
    g, u, want = (be.alloc(T * rows * 4) for _ in range(3))
    y = out_buf(be, T * rows)
    graph = be.capture(lambda: be.ffn_gate_up(w[0], w[1], x, g, u, y))
    be.ffn_gate_up(w[0], w[1], x, g, u, want)
    ref = be.download_f32(want)
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        graph.launch()
        got = be.download_f32(y)
        assert np.all(got[T * rows:] == CANARY)
        # Both are sums in f64 rounded once, then silu_mul's own roundings.
        assert np.allclose(got[:T * rows], ref, rtol=6 * 2.0**-24, atol=0)
    graph.close()
    be.close()


def test_partials_space_gives_way_to_the_budget():
    be = Gfx950Backend(0)
    rows, k, T = 200, 1024, 70
    raw = synth.weight(Q4K, rows, k, 1, True)
    be.set_buffer_budget(device=80 << 20)
    w, x_h = be.upload_weight(raw, Q4K, (rows, k)), synth.normal_f32(T * k, 2)
    x, y = be.f32_buf(x_h), out_buf(be, T * rows)
    before, limit = be.buffer_usage(DOMAIN_DEVICE)
    be.qmatmul(w, x, y)
    assert be.buffer_usage(DOMAIN_DEVICE)[0] > before  # charged as it grew
    rest = be.alloc(limit - before)  # all that the caller had left
    assert be.buffer_usage(DOMAIN_DEVICE)[0] == limit
    be.upload(y, 0, np.zeros(T * rows, np.float32))
    be.qmatmul(w, x, y)  # no space: unsplit
    check(be, y, T, Q4K, raw, rows, k, x_h, "over budget")
    rest.close()
    be.close()


@pytest.mark.parametrize("full", [False, True])
def test_captured_partials_space_outlives_its_growth(full):
    # A graph of a launch that splits eagerly replays after a larger call
    # replaced the partial tiles' space, or found no room in the budget for
    # more of it, and after a caller's allocation took the space back: no graph
    # points into it.
    be = Gfx950Backend(0)
    be.set_buffer_budget(device=512 << 20)
    rows, k, T, big_rows, big_T = 200, 1024, 20, 2100, 100
    raw, big_raw = synth.weight(Q6K, rows, k, 1, True), synth.weight(Q6K, big_rows, k, 3, True)
    w, bw = be.upload_weight(raw, Q6K, (rows, k)), be.upload_weight(big_raw, Q6K, (big_rows, k))
    x_h, bx_h = synth.normal_f32(T * k, 2), synth.normal_f32(big_T * k, 4)
    x, bx, y, by = be.f32_buf(x_h), be.f32_buf(bx_h), out_buf(be, T * rows), out_buf(be, big_T * big_rows)
    be.qmatmul(w, x, y)  # makes the space
    used = be.buffer_usage(DOMAIN_DEVICE)[0]
    graph = be.capture(lambda: be.qmatmul(w, x, y))
    filler = be.alloc(((512 << 20) - used) // 4096 * 4096 - 4096) if full else None
    used = be.buffer_usage(DOMAIN_DEVICE)[0]
    for _ in range(3):
        be.qmatmul(bw, bx, by)
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        graph.launch()
        check(be, y, T, Q6K, raw, rows, k, x_h, "replayed")
        check(be, by, big_T, Q6K, big_raw, big_rows, k, bx_h, "grown")
    now, limit = be.buffer_usage(DOMAIN_DEVICE)
    assert (now == used) if full else (now > used)
    rest = be.alloc((limit - now) // 4096 * 4096 + 8192)
    assert be.buffer_usage(DOMAIN_DEVICE)[0] - rest.len < now  # the space went
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        graph.launch()
        check(be, y, T, Q6K, raw, rows, k, x_h, "replayed without the space")
    rest.close()
    if filler:
        filler.close()
    graph.close()
    be.close()


def test_nan_and_infinity_stay_in_their_token(backend):
    rows, k, T = 64, 512, 20
    raw = synth.weight(Q6K, rows, k, 1, True)
    w, x_h = backend.upload_weight(raw, Q6K, (rows, k)), synth.normal_f32(T * k, 2)
    clean, y = backend.alloc(T * rows * 4), backend.alloc(T * rows * 4)
    backend.qmatmul(w, backend.f32_buf(x_h), clean)
    bad = x_h.reshape(T, k).copy()
    bad[3, 17], bad[18, 300] = np.nan, np.inf
    backend.qmatmul(w, backend.f32_buf(bad), y)
    got, ref = backend.download_f32(y).reshape(T, rows), backend.download_f32(clean).reshape(T, rows)
    keep = [t for t in range(T) if t not in (3, 18)]
    assert np.array_equal(got[keep], ref[keep])
    assert np.isnan(got[3]).all() and not np.isfinite(got[18]).any()



def test_captured_launch_splits_into_the_scratch():
    # With room in the reserved scratch a captured launch splits as an eager
    # one does: the same bits, whatever else uses the scratch in between.
    be = Gfx950Backend(0)
    rows, k, T = 300, 1024, 70
    raw = synth.weight(Q6K, rows, k, 1, True)
    w, x_h = be.upload_weight(raw, Q6K, (rows, k)), synth.normal_f32(T * k, 2)
    x, y, e = be.f32_buf(x_h), out_buf(be, T * rows), out_buf(be, T * rows)
    be.qmatmul(w, x, e)
    be.reserve_scratch(64 << 20)
    graph = be.capture(lambda: be.qmatmul(w, x, y))
    for _ in range(3):
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        be.greedy(x)  # writes the scratch
        graph.launch()
        assert np.array_equal(be.download_f32(y), be.download_f32(e))
    graph.close()
    be.close()


def test_refused_allocation_leaves_partials_and_graphs():
    # A request that the budget has no room for even without the partials'
    # space is refused and changes nothing.
    be = Gfx950Backend(0)
    be.set_buffer_budget(device=256 << 20)
    rows, k, T = 200, 1024, 20
    raw = synth.weight(Q6K, rows, k, 1, True)
    w, x_h = be.upload_weight(raw, Q6K, (rows, k)), synth.normal_f32(T * k, 2)
    x, y = be.f32_buf(x_h), out_buf(be, T * rows)
    be.qmatmul(w, x, y)  # makes the space
    graph = be.capture(lambda: be.qmatmul(w, x, y))
    used, limit = be.buffer_usage(DOMAIN_DEVICE)
    for n in (limit, limit + 1, 2**64 - 1 - limit, 2**64 - 300):
        with pytest.raises(BackendError):
            be.alloc(n)
        assert be.buffer_usage(DOMAIN_DEVICE)[0] == used
        be.upload(y, 0, np.zeros(T * rows, np.float32))
        graph.launch()
        check(be, y, T, Q6K, raw, rows, k, x_h, "replayed")
    graph.close()
    be.close()


@pytest.mark.parametrize("partials", [False, True])
def test_launches_after_an_allocation_the_device_refused(partials):
    # The refused hipMalloc's error does not meet the next launch, and the
    # partials' space, which could not have made the room, stays.
    be = Gfx950Backend(0)
    rows, k, T = 200, 1024, 20
    raw = synth.weight(Q6K, rows, k, 1, True)
    w, x_h = be.upload_weight(raw, Q6K, (rows, k)), synth.normal_f32(T * k, 2)
    x, y = be.f32_buf(x_h), out_buf(be, T * rows)
    if partials:
        be.qmatmul(w, x, y)
    used = be.buffer_usage(DOMAIN_DEVICE)[0]
    with pytest.raises(BackendError, match="hipMalloc"):
        be.alloc(1 << 50)
    assert be.buffer_usage(DOMAIN_DEVICE)[0] == used
    be.silu_mul(x, x, x)  # a launch whose check reads the last error
    be.upload(x, 0, x_h)
    be.qmatmul(w, x, y)
    check(be, y, T, Q6K, raw, rows, k, x_h, "after the refusal")
    be.close()


@pytest.mark.parametrize("k", [288, 32, 512])
@pytest.mark.parametrize("T", [2, 4, 8, 20])
@pytest.mark.parametrize("fused", [False, True])
def test_infinity_in_a_rows_last_columns(backend, k, T, fused):
    # A row of blocks that do not fill the last 256 columns: what stands in the
    # rest is no input. The sums are infinite (NaN for a zero weight), as the
    # CPU's are.
    rows = 97
    raw = synth.weight(Q8, rows, k, 1, True)
    x_h = synth.normal_f32(T * k, 2).reshape(T, k)
    x_h[0, k - 1], x_h[T - 1, k - 4] = np.inf, -np.inf
    w, x, y = backend.upload_weight(raw, Q8, (rows, k)), backend.f32_buf(x_h), out_buf(backend, T * rows)
    want = ffi.qmatmul(Q8, raw, rows, k, x_h).reshape(T, rows)
    if fused:
        g, u = backend.alloc(T * rows * 4), backend.alloc(T * rows * 4)
        backend.ffn_gate_up(w, w, x, g, u, y)
        with np.errstate(all="ignore"):
            want = want / (1 + np.exp(-want)) * want
    else:
        backend.qmatmul(w, x, y)
    got = backend.download_f32(y)[:T * rows].reshape(T, rows)
    bad = [0, T - 1]
    assert np.isinf(want[bad]).sum() > rows // 2  # (few weights are zero; silu(-inf) is NaN)
    assert np.array_equal(got[bad], want[bad], equal_nan=True)
    assert np.allclose(got[1:T - 1], want[1:T - 1], rtol=1e-4, atol=1e-4)


def test_partials_space_is_no_use_of_the_budget():
    # With every buffer of the caller's freed the ledger counts as unused (the
    # f32 mode's calls leave nothing else): a budget can be installed.
    be = Gfx950Backend(0)
    rows, k, T = 200, 1024, 70
    w = be.upload_weight(synth.weight(Q4K, rows, k, 1, True), Q4K, (rows, k))
    x, y = be.f32_buf(synth.normal_f32(T * k, 2)), out_buf(be, T * rows)
    be.qmatmul(w, x, y)
    with pytest.raises(BackendError):
        be.set_buffer_budget(device=1 << 20)
    for b in (w.buf, x, y):
        b.close()
    be.set_buffer_budget(device=1 << 20)
    assert be.buffer_usage(DOMAIN_DEVICE) == (0, 1 << 20)
    be.close()
