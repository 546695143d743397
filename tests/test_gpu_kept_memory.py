"""Device memory that a context keeps from destroyed handles and zr_free (csrc/zr_runtime.hip): reuse in stream order, the errors there were, and
nothing kept where another context or a caller's stream could still use a block."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import Layer
from zoph_rnn_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def raw_free(ctx, ptr):
    return capi.load().zr_free(ctx.h, ctypes.c_void_p(ptr))


def test_a_freed_block_is_handed_out_again_and_freeing_it_twice_is_an_error(ctx):
    a = ctx.zeros((1 << 20,))
    ptr = a.ptr
    a.free()
    assert raw_free(ctx, ptr) != 0
    b = ctx.empty((1 << 20,))
    assert b.ptr == ptr
    small = ctx.empty((1000,))
    assert small.ptr != ptr
    b.free()


def test_weights_packed_again_while_the_old_ones_are_in_use(ctx):
    """A training loop's pack: the new weights' block is the old one's, which a queued sweep still reads."""
    H, mb, T, V, L = 200, 24, 40, 64, 2
    cfgs = [synth.encoder_config(H=H, mb=mb, T=T, V=V, L=L) for _ in range(2)]
    g = synth.rng(900, 1)
    for ly in cfgs[1]["layers"]:
        for k in ("M", "Wh"):
            ly[k] = [np.asfortranarray(synth.uniform(g, (H, H))) for _ in range(4)]
    embed, ids = ctx.array(cfgs[0]["embed"]), ctx.array(np.abs(cfgs[0]["ids"]).reshape(-1).astype(np.int32))
    ones, z = ctx.array(np.ones(mb * T, np.int32)), ctx.zeros((H, mb))
    mats = [[Layer(ctx, ly) for ly in c["layers"]] for c in cfgs]  # (matrices on the device; packed again below)

    def pack(which):
        return [ctx.lstm_pack(ly.M, ly.Wh, ly.b, H) for ly in mats[which]]

    def sweep(w, h, c):
        ctx.lstm_stack_forward(w, embed, V, ids, ones, T, mb, [z] * L, [z] * L, h, c)

    def buffers():
        return [ctx.empty((H * mb * T,)) for _ in range(L)], [ctx.empty((H * mb * T,)) for _ in range(L)]

    want = []
    for which in (0, 1):
        w, (h, c) = pack(which), buffers()
        sweep(w, h, c)
        ctx.sync()
        want.append([a.get() for a in h + c])
        for x in w:
            ctx.lstm_weights_destroy(x)
    assert not np.array_equal(want[0][-1], want[1][-1])
    outs = [buffers() for _ in range(8)]
    w = pack(0)
    for i, (h, c) in enumerate(outs):  # no wait in between
        sweep(w, h, c)
        for x in w:
            ctx.lstm_weights_destroy(x)
        w = pack((i + 1) % 2)
    ctx.sync()
    for i, (h, c) in enumerate(outs):
        for a, b in zip(h + c, want[i % 2]):
            assert np.array_equal(a.get(), b)
    for x in w + [ly.w for m in mats for ly in m]:
        ctx.lstm_weights_destroy(x)


def test_beyond_the_bound_blocks_are_given_back(ctx):
    """Freeing 80 blocks of 24 MiB keeps at most 512 MiB of them."""
    blocks = [ctx.empty((6 << 20,)) for _ in range(80)]
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for b in blocks:
        b.free()
    given_back = torch.cuda.mem_get_info()[0] - before
    assert given_back >= 80 * (24 << 20) - (512 << 20) - (64 << 20)


def test_nothing_is_kept_with_another_context_or_stream(ctx):
    a = ctx.empty((12 << 20,))
    other = capi.Context(0)
    before = torch.cuda.mem_get_info()[0]
    a.free()
    assert torch.cuda.mem_get_info()[0] - before >= 40 << 20
    other.close()
    b = ctx.empty((12 << 20,))
    b.free()  # kept now
    before = torch.cuda.mem_get_info()[0]
    s = torch.cuda.Stream()
    capi._chk(capi.load().zr_ctx_set_stream(ctx.h, ctypes.c_void_p(s.cuda_stream)))
    assert torch.cuda.mem_get_info()[0] - before >= 40 << 20
    c = ctx.empty((12 << 20,))
    before = torch.cuda.mem_get_info()[0]
    c.free()
    assert torch.cuda.mem_get_info()[0] - before >= 40 << 20
    ctx.sync()
    capi._chk(capi.load().zr_ctx_set_stream(ctx.h, None))


def free_bytes():
    return torch.cuda.mem_get_info()[0]


MIB = 1 << 20


def keep(ctx, mib, blocks=1):
    for b in [ctx.empty((mib << 18,)) for _ in range(blocks)]:
        b.free()


def test_another_context_has_what_was_kept_given_back(ctx):
    keep(ctx, 200)
    before = free_bytes()
    other = capi.Context(0)
    assert free_bytes() - before >= 150 * MIB
    other.close()


def test_an_output_layer_is_prepared_with_memory_that_was_kept(ctx):
    """Memory for the copy of the matrix, which is no kept block's size, only with what the context keeps."""
    V, H = 380000, 1000
    need = (V + 31) // 32 * 32 * H * 4
    D = torch.zeros((H, V), device="cuda")
    torch.cuda.synchronize()
    keep(ctx, 200, 2)
    hog = []
    try:
        while free_bytes() > need - 150 * MIB and len(hog) < 8:
            hog.append(torch.empty(free_bytes() - need + 200 * MIB, dtype=torch.uint8, device="cuda"))
        assert free_bytes() < need
        ctx.softmax_prepare(D.data_ptr(), V, H)
        ctx.sync()
        ctx.softmax_release(D.data_ptr())
    finally:
        del hog
        torch.cuda.empty_cache()


def test_a_sweeps_memory_serves_an_allocation_that_fails_without_it(ctx):
    L, H, mb, T = 4, 512, 128, 40
    r = np.random.default_rng(11)
    draw = lambda *shape: ctx.array(r.random(shape, np.float32))
    mats = [[ctx.array(synth.uniform(synth.rng(901, i), (H, H))) for _ in range(4)] for i in range(2)]
    layers = [ctx.lstm_train_create(mats[0], mats[1], H) for _ in range(L)]
    ones, top, c0 = ctx.array(np.ones(mb * T, np.int32)), draw(H * mb * T), [draw(H * mb) for _ in range(L)]
    c, gates = [draw(H * mb * T) for _ in range(L)], [draw(4 * H * mb * T) for _ in range(L)]
    dg, eh, ec = [[ctx.empty((k * H * mb,)) for _ in range(L)] for k in (4 * T, 1, 1)]

    def sweep():
        ctx.lstm_stack_backward(layers, T, mb, ones, c0, c, gates, top, dg, eh, ec)
        ctx.sync()
        return [x.get() for x in dg + eh + ec]

    want = sweep()
    path = ctx.query(capi.ZR_QUERY_LSTM_BACKWARD_PATH)
    scratch = ctx.query(capi.ZR_QUERY_SCRATCH_KIB) << 10
    assert path == capi.ZR_LSTM_BACKWARD_PATH_RESIDENT and scratch >= 150 * MIB
    hog = []
    try:
        while free_bytes() > 600 * MIB and len(hog) < 8:
            hog.append(torch.empty(free_bytes() - 512 * MIB, dtype=torch.uint8, device="cuda"))
        need = free_bytes() + scratch // 2
        p = ctypes.c_void_p()
        assert capi.load().zr_malloc(ctx.h, ctypes.c_size_t(need), ctypes.byref(p)) == 0
        assert ctx.query(capi.ZR_QUERY_SCRATCH_KIB) == 0
        assert raw_free(ctx, p.value) == 0
    finally:
        del hog
        torch.cuda.empty_cache()
    for a, b in zip(sweep(), want):
        assert np.array_equal(a, b)
    for w in layers:
        ctx.lstm_train_destroy(w)


def test_nothing_is_kept_without_the_option(ctx):
    keep(ctx, 200)
    before = free_bytes()
    ctx.set_option(capi.ZR_OPT_KEEP_MEMORY, 0)
    assert free_bytes() - before >= 150 * MIB
    a = ctx.empty((50 << 20,))
    before = free_bytes()
    a.free()
    assert free_bytes() - before >= 150 * MIB
    ctx.set_option(capi.ZR_OPT_KEEP_MEMORY, 1)


def hip():
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    return ctypes.CDLL(path)


def test_memory_of_another_allocator_is_not_kept(ctx):
    torch.cuda.synchronize()
    p = ctypes.c_void_p()
    assert hip().hipMalloc(ctypes.byref(p), ctypes.c_size_t(200 * MIB)) == 0
    before = free_bytes()
    assert raw_free(ctx, p.value) == 0
    assert free_bytes() - before >= 150 * MIB


def test_freeing_waits_for_work_on_any_stream(ctx):
    a = ctx.empty((1 << 20,))
    s = torch.cuda.Stream()
    done = torch.cuda.Event()
    with torch.cuda.stream(s):
        torch.cuda._sleep(100_000_000)
        done.record()
    assert not done.query()
    a.free()
    assert done.query()


def test_freeing_during_a_relaxed_capture_of_another_stream(ctx):
    """As with hipFree, which such a capture allows."""
    a = ctx.zeros((1 << 20,))
    ctx.sync()
    x = torch.zeros(1000, device="cuda")
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="relaxed"):
        x.add_(1)
        freed = raw_free(ctx, a.ptr)
        a.ptr = 0
        b = ctx.empty((1 << 20,))
        x.add_(1)
    assert freed == 0
    for i in range(3):
        g.replay()
        b.set(np.full(1 << 20, i, np.float32))
        torch.cuda.synchronize()
        assert x[0].item() == 2.0 * (i + 1) and b.get()[5] == i


def test_destroying_a_handle_returns_the_error_of_its_wait(ctx):
    """On a stream that is being captured there is no waiting: an error, after which the handle is still there."""
    H, beam = 64, 3
    mats = [[ctx.zeros((H, H)) for _ in range(4)] for _ in range(2)]
    vec = [ctx.zeros((H,)) for _ in range(4)]
    L = capi.load()
    handles = [(L.zr_lstm_weights_destroy, ctx.lstm_pack(mats[0], mats[1], vec, H)), (L.zr_lstm_train_destroy, ctx.lstm_train_create(mats[0], mats[1], H)),
               (L.zr_attn_destroy, ctx.attn_create(H, beam, 2, mats[0][0], mats[0][1], vec[0], vec[1], mats[0][2], mats[0][3], [ctx.zeros((H, beam))])),
               (L.zr_beam_destroy, ctx.beam_create(beam, 100, 1, 10, 0.0))]
    ctx.sync()
    lib, stream, graph = hip(), ctypes.c_void_p(), ctypes.c_void_p()
    assert lib.hipStreamCreate(ctypes.byref(stream)) == 0
    capi._chk(L.zr_ctx_set_stream(ctx.h, stream))
    for destroy, handle in handles:
        assert lib.hipStreamBeginCapture(stream, 2) == 0  # relaxed
        assert destroy(ctx.h, handle) == -2
        lib.hipStreamEndCapture(stream, ctypes.byref(graph))
        lib.hipGetLastError()
    capi._chk(L.zr_ctx_set_stream(ctx.h, None))
    for destroy, handle in handles:
        assert destroy(ctx.h, handle) == 0
    ctx.sync()
    assert lib.hipStreamDestroy(stream) == 0
