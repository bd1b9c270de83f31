"""Sizes at which the kernels' tiles and dispatch rules change: MXFP4 prefill GEMM job tiles and row
units, the router's two forms, and the one-token layer call."""
import ctypes as C

import numpy as np
import pytest

import helpers as H
from test_gpu_layer import Layer
from test_gpu_prefill import unit_scale_activations, unit_scale_mxfp4, unit_scale_q8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("type_id", [H.MX, H.Q8])
@pytest.mark.parametrize("rows,k", [(288, 576), (544, 256)])
def test_gemm_job_counts_around_the_tile_edges_exact(gpu, orc, type_id, rows, k):
    """One expert per job count: 1, 15..17 and 63..65 jobs (fragment columns of 16, job tiles of 64), 130
    jobs, and experts without any; rows past the 256-row units. Unit scales: every fp32 sum is an exact
    integer, so any order gives the oracle's bits."""
    counts = [1, 0, 15, 16, 17, 63, 64, 65, 130, 0, 33, 48, 96, 97]
    ids = np.repeat(np.arange(len(counts)), counts).astype(np.int32)
    rng = np.random.default_rng(11 + rows)
    rng.shuffle(ids)
    ids = ids.reshape(-1, 1)
    tokens = ids.shape[0]
    w = (unit_scale_mxfp4 if type_id == H.MX else unit_scale_q8)(len(counts), rows, k, rng)
    bank = H.make_bank(type_id, w, len(counts), rows, k)
    x = unit_scale_activations(tokens, k, rng).reshape(tokens, 1, k)
    got = H.mul_mat_id(bank, len(counts), x, gpu.TYPE_F32, 1, ids, 1, order=gpu.ORDER_FAST)
    ref = orc.mul_mat_id(type_id, w, k, rows, len(counts), 0, x, 1, ids, 1, tokens, 1, threads=8)
    assert H.bits_equal(got, ref), H.diff_report(got, ref)
    bank.destroy()


@pytest.mark.parametrize("type_id", [H.MX, H.Q8])
@pytest.mark.parametrize("units", [5, 8, 9, 13, 22, 23])
def test_gemm_tile_splits_exact(gpu, orc, type_id, units):
    """23 job tiles of 16 experts over bank rows of 5 to 23 workgroups each: tiles in quarters (115 items), in halves
    though quarters are allowed (184), in halves (207), whole with even shares though halves are allowed (299), whole with
    even shares (506) and whole (529). Unit scales: every fp32 sum is an exact integer."""
    counts = [1, 0, 15, 16, 17, 33, 48, 63, 64, 65, 80, 81, 96, 97, 128, 129]
    assert sum(-(-c // 64) for c in counts) == 23 and 32 < sum(counts) // len(counts) <= 64
    ids = np.repeat(np.arange(len(counts)), counts).astype(np.int32)
    rng = np.random.default_rng(units)
    rng.shuffle(ids)
    ids = ids.reshape(-1, 1)
    tokens, rows, k = ids.shape[0], 256 * units - 160, 192
    w = (unit_scale_mxfp4 if type_id == H.MX else unit_scale_q8)(len(counts), rows, k, rng)
    bank = H.make_bank(type_id, w, len(counts), rows, k)
    x = unit_scale_activations(tokens, k, rng).reshape(tokens, 1, k)
    got = H.mul_mat_id(bank, len(counts), x, gpu.TYPE_F32, 1, ids, 1, order=gpu.ORDER_FAST)
    ref = orc.mul_mat_id(type_id, w, k, rows, len(counts), 0, x, 1, ids, 1, tokens, 1, threads=8)
    assert H.bits_equal(got, ref), H.diff_report(got, ref)
    bank.destroy()


def test_gemv_fold_check_sees_every_wave(gpu, orc):
    """One exponent too large to fold, in each expert in another 1 KiB part of the tile pair's exponents (the
    part one wave checks), at every chunk width: folded all the same, its weights overflow to infinity."""
    rows, k, experts = 64, 4096, 8
    rng = np.random.default_rng(8)
    w = H.synth_weights(H.MX, 17, 3, experts, rows, k).reshape(experts, rows, k // 32, 17)
    for e in range(experts):
        w[e, 8 * e + int(rng.integers(8)), int(rng.integers(k // 32)), 0] = 150
    bank = H.make_bank(H.MX, w.reshape(-1), experts, rows, k)
    for tokens in (1, 2, 4, 7):
        ids = np.tile(np.arange(experts, dtype=np.int32), (tokens, 1))
        x = gpu.synth_normal(17, 4, tokens, tokens * k).reshape(tokens, 1, k)
        got = H.mul_mat_id(bank, experts, x, gpu.TYPE_F32, 1, ids, experts)
        ref = orc.mul_mat_id(H.MX, w.reshape(-1), k, rows, experts, 0, x, 1, ids, experts, tokens, experts, threads=8)
        assert H.bits_equal(got, ref), (tokens, H.diff_report(got, ref))
    bank.destroy()


@pytest.mark.parametrize("hidden", [32, 64, 96, 160, 256, 288, 512, 736, 31])
@pytest.mark.parametrize("n_expert,tokens", [(8, 5), (128, 65)])
def test_router_logits_row_ends_bitwise(gpu, orc, n_expert, tokens, hidden):
    """Rows of 1, 2, 3, 5 and 8 steps (their own batch widths), of 9, 16 and 23 (full batches and a rest), and of
    none, in both forms of the kernel."""
    w = gpu.synth_normal(16, 1, 0, n_expert * hidden, 0.0, 0.02).reshape(n_expert, hidden)
    x = gpu.synth_normal(16, 2, 0, tokens * hidden).reshape(tokens, hidden)
    dw, dx = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x)
    dl, di, dwt = (gpu.DeviceBuffer(4 * tokens * n) for n in (n_expert, 2, 2))
    gpu.call("vbm_router_topk_softmax", dw.ptr, None, dx.ptr, hidden, dl.ptr, n_expert, tokens, 2, di.ptr, dwt.ptr, None)
    logits, ids, _ = orc.router(router_w=w, x=x, n_expert=n_expert, n_tokens=tokens, top_k=2, hidden=hidden)
    assert H.bits_equal(dl.download(np.float32, (tokens, n_expert)), logits)
    assert np.array_equal(di.download(np.int32, (tokens, 2)), ids)


@pytest.mark.parametrize("n_expert,tokens,hidden", [(8, 3, 1000), (32, 1, 2880), (33, 250, 2880), (32, 257, 100), (64, 128, 960)])
def test_router_logits_bitwise(gpu, orc, n_expert, tokens, hidden):
    """One token per weight row and, from 8192 (expert, token) pairs on, four: ragged token counts, rows of
    one batch of steps and of several, and rows with a remainder past the last 32 (summed serially)."""
    w = gpu.synth_normal(15, 1, 0, n_expert * hidden, 0.0, 0.02).reshape(n_expert, hidden)
    x = gpu.synth_normal(15, 2, 0, tokens * hidden).reshape(tokens, hidden)
    dw, dx = gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x)
    dl, di, dwt = (gpu.DeviceBuffer(4 * tokens * n) for n in (n_expert, 2, 2))
    gpu.call("vbm_router_topk_softmax", dw.ptr, None, dx.ptr, hidden, dl.ptr, n_expert, tokens, 2, di.ptr, dwt.ptr, None)
    logits, ids, _ = orc.router(router_w=w, x=x, n_expert=n_expert, n_tokens=tokens, top_k=2, hidden=hidden)
    assert H.bits_equal(dl.download(np.float32, (tokens, n_expert)), logits)
    assert np.array_equal(di.download(np.int32, (tokens, 2)), ids)


def kernels_of(gpu, call):
    """Kernel launches that call(stream) records into a captured graph (not run)."""
    with open("/proc/self/maps") as maps:                       # the runtime the library itself runs on
        hip = C.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    stream, graph, count = C.c_void_p(), C.c_void_p(), C.c_size_t()
    gpu.call("vbm_stream_create", C.byref(stream))
    assert hip.hipStreamBeginCapture(stream, 2) == 0            # relaxed
    call(stream.value)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(count)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    gpu.call("vbm_stream_destroy", stream.value)
    return count.value


@pytest.mark.parametrize("type_id,hidden,inter,experts,top_k,act,biases,decode", [
    (H.MX, 2880, 2880, 32, 4, 1, True, True), (H.Q8, 2048, 768, 128, 8, 0, False, True), (H.MX, 64, 4096, 300, 3, 0, True, True),
    (H.Q8, 4096, 64, 9, 9, 1, True, True), (H.MX, 448, 192, 5, 1, 1, False, True),
    # top_k and top_k + 1 at the line between the paths, up to 128, 256 and more experts
    (H.MX, 128, 512, 64, 32, 1, True, True), (H.MX, 128, 512, 64, 33, 1, True, False),
    (H.Q8, 64, 512, 200, 25, 0, False, True), (H.Q8, 64, 512, 200, 26, 0, False, False),
    (H.MX, 64, 512, 300, 16, 1, False, True), (H.MX, 64, 512, 300, 17, 1, False, False)])
def test_one_token_layer_takes_either_path(gpu, orc, type_id, hidden, inter, experts, top_k, act, biases, decode):
    """A one-token call runs the decode kernels (three launches) when its input is 16-byte aligned and its
    routing small, and the batched path (four) otherwise: the oracle's bits from both, and the same ids and weights."""
    layer = Layer(gpu, type_id, hidden, inter, experts, top_k, seed=91, router=False, biases=biases, activation=act,
                  q8_scale=(1e-4, 1e-3))
    x = gpu.synth_normal(91, 6, 0, hidden).reshape(1, hidden)
    logits = gpu.synth_normal(91, 7, 0, experts).reshape(1, experts)
    logits[0, : experts // 2] = np.round(logits[0, : experts // 2])          # ties
    ref = layer.forward_cpu(orc, x, logits)
    d = layer.desc()
    need = C.c_size_t()
    gpu.call("vbm_moe_layer_workspace", C.byref(d), 1, C.byref(need))
    work = gpu.DeviceBuffer(need.value)
    dx = gpu.DeviceBuffer.from_array(x)
    off = gpu.DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), x[0]]))
    dl = gpu.DeviceBuffer.from_array(logits)
    weights = []
    for src, launches in ((dx.ptr, 3 if decode else 4), (off.ptr + 4, 4)):
        out, ids, w = gpu.DeviceBuffer(4 * hidden), gpu.DeviceBuffer(4 * top_k), gpu.DeviceBuffer(4 * top_k)

        def forward(stream):
            gpu.call("vbm_moe_layer_forward", C.byref(d), src, dl.ptr, 1, out.ptr, ids.ptr, w.ptr, work.ptr, need.value, stream)

        assert kernels_of(gpu, forward) == launches
        forward(None)
        gpu.call("vbm_stream_synchronize", None)
        assert np.array_equal(ids.download(np.int32, (1, top_k)), ref["ids"])
        weights.append(w.download(np.float32, (1, top_k)))
        assert np.allclose(weights[-1], ref["weights"], rtol=1e-6, atol=0)
        got = out.download(np.float32, (1, hidden))
        assert H.bits_equal(got, ref["out"]), H.diff_report(got, ref["out"])
    assert H.bits_equal(*weights)
    layer.destroy()


def test_nan_logits_route_alike_on_every_path(gpu):
    """NaN logits rank as -inf: valid ids, and the same ids, weights and output from the decode kernels, the
    batched path and a row of a batch, with as many numbers as picks, fewer, none, and real -inf among them."""
    experts, top_k, hidden = 20, 4, 128
    layer = Layer(gpu, H.MX, hidden, 128, experts, top_k, seed=37, router=False)
    inf, nan = np.float32(np.inf), np.float32(np.nan)
    logits = np.full((5, experts), nan, np.float32)
    logits[0] = gpu.synth_normal(37, 7, 0, experts)
    logits[0, ::3] = nan
    logits[1, [3, 17]] = 1.0, 2.0
    logits[3, [0, 9, 12]] = -inf, 0.5, -inf
    logits[4, 5:] = -inf
    x = gpu.synth_normal(37, 6, 0, 5 * hidden).reshape(5, hidden)
    want = np.argsort(-np.where(np.isnan(logits), -inf, logits), axis=1, kind="stable")[:, :top_k]
    batch = layer.forward_gpu(x, logits)
    assert np.array_equal(batch[1], want)
    d = layer.desc()
    need = C.c_size_t()
    gpu.call("vbm_moe_layer_workspace", C.byref(d), 1, C.byref(need))
    work = gpu.DeviceBuffer(need.value)
    for t in range(5):
        dl = gpu.DeviceBuffer.from_array(logits[t:t + 1])
        for pad in (0, 1):
            dx = gpu.DeviceBuffer.from_array(np.concatenate([np.zeros(pad, np.float32), x[t]]))
            out, ids, w = gpu.DeviceBuffer(4 * hidden), gpu.DeviceBuffer(4 * top_k), gpu.DeviceBuffer(4 * top_k)
            gpu.call("vbm_moe_layer_forward", C.byref(d), dx.ptr + 4 * pad, dl.ptr, 1, out.ptr, ids.ptr, w.ptr, work.ptr, need.value, None)
            gpu.call("vbm_stream_synchronize", None)
            for got, ref in ((out.download(np.float32, (hidden,)), batch[0][t]), (ids.download(np.int32, (top_k,)), batch[1][t]),
                             (w.download(np.float32, (top_k,)), batch[2][t])):
                assert np.array_equal(got, ref, equal_nan=got.dtype == np.float32), (t, pad)
    assert np.all(batch[2][1, 2:] == 0) and np.all(np.isnan(batch[0][2])) and not np.any(np.isnan(batch[0][[0, 1, 3]]))
    layer.destroy()


@pytest.mark.parametrize("hidden,inter,top_k", [(2048, 1024, 20), (2048, 1024, 21), (1024, 512, 16), (1024, 512, 17), (704, 512, 3)])
def test_decode_q8_ring_depths_bitwise(gpu, orc, hidden, inter, top_k):
    """Q8_0 gate_up on both sides of the lines between its two ring depths: 1280 workgroups of the unrolled
    kernel, 512 of the rolled one, and a row too short for the deep ring."""
    layer = Layer(gpu, H.Q8, hidden, inter, top_k, top_k, seed=61, router=False, biases=False, activation=0, q8_scale=(1e-4, 1e-3))
    x = gpu.synth_normal(61, 6, 0, hidden).reshape(1, hidden)
    logits = gpu.synth_normal(61, 7, 0, top_k).reshape(1, top_k)
    ref = layer.forward_cpu(orc, x, logits)
    plan = C.c_void_p()
    gpu.call("vbm_decode_plan_create", (gpu.MoeLayerDesc * 1)(layer.desc()), 1, C.byref(plan))
    dx, dl, out = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer.from_array(logits), gpu.DeviceBuffer(4 * hidden)
    gpu.call("vbm_decode_step", plan.value, dx.ptr, dl.ptr, out.ptr, None, None, None, None)
    gpu.call("vbm_stream_synchronize", None)
    got = out.download(np.float32, (1, hidden))
    assert H.bits_equal(got, ref["out"]), H.diff_report(got, ref["out"])
    gpu.call("vbm_decode_plan_destroy", plan.value)
    layer.destroy()


@pytest.mark.parametrize("top_k,hidden", [(1, 320), (8, 256), (9, 320), (17, 64)])
def test_decode_step_finish_matches_layer_calls(gpu, top_k, hidden):
    """The step's last launch combines the ranks in batches of eight and hands out ids and weights: two
    chained layers against two one-token layer calls, bit for bit, with and without the optional outputs."""
    experts, inter, L = 20, 128, 2
    layers = [Layer(gpu, H.MX, hidden, inter, experts, top_k, seed=33, layer=l, router=False) for l in range(L)]
    x = gpu.synth_normal(33, 6, 0, hidden).reshape(1, hidden)
    logits = gpu.synth_normal(33, 7, 0, L * experts).reshape(L, experts)
    want, want_ids, want_w = x, [], []
    for l in range(L):
        want, i, w = layers[l].forward_gpu(want, logits[l:l + 1])
        want_ids.append(i), want_w.append(w)
    plan = C.c_void_p()
    gpu.call("vbm_decode_plan_create", (gpu.MoeLayerDesc * L)(*[l.desc() for l in layers]), L, C.byref(plan))
    dx, dl = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer.from_array(logits)
    for outputs in (True, False):
        out, ids, w = gpu.DeviceBuffer(4 * hidden), gpu.DeviceBuffer(4 * L * top_k), gpu.DeviceBuffer(4 * L * top_k)
        gpu.call("vbm_decode_step", plan.value, dx.ptr, dl.ptr, out.ptr, ids.ptr if outputs else None, w.ptr if outputs else None, None, None)
        gpu.call("vbm_stream_synchronize", None)
        assert H.bits_equal(out.download(np.float32, (1, hidden)), want)
        if outputs:
            assert np.array_equal(ids.download(np.int32, (L, top_k)), np.concatenate(want_ids))
            assert H.bits_equal(w.download(np.float32, (L, top_k)), np.concatenate(want_w))
    gpu.call("vbm_decode_plan_destroy", plan.value)
    for l in layers:
        l.destroy()
