"""The work this library is used for, as cases with sizes: what each pass needs in hand, the pass itself through the
public entry points (zoph_rnn_amd.capi, zoph_rnn_amd.driver), the bytes and operations it cannot do without, and how far
two correct implementations may lie apart.

Kinds of case
  lm_logprobs   a language model scored in full: stack forward and the whole matrix of log-probabilities
  lm_loss       force decoding: stack forward and the summed log-probability of the given words
  encode        the encoder sweep over a minibatch of (ragged, left-padded) source sentences
  decode_step   one decoder time step to the output distribution, with attention and feed-input
  translate     a batch of sentences from token ids to finished hypotheses, beam search on the device
  lm_train      one SGD step of a language model: forward, backward, gradients, clipped update of every parameter
  nmt_train     one SGD step of an encoder-decoder model with attention and feed-input
"""
import math

import numpy as np
import torch

from zoph_rnn_amd import capi, driver

INIT = 0.08  # weights are drawn from U(-0.08, 0.08), the range models are initialised with


# ---- cases --------------------------------------------------------------------------------------------------------

def listed():
    return [
        # The smallest model in use: one layer, 8 sentences of 20 words.  Launches and latency decide.
        dict(name="lm_logprobs_h100_8x20", kind="lm_logprobs", H=100, L=1, mb=8, T=20, V=10000),
        # Scoring text with a mid-sized language model, a batch that is no multiple of a tile and an odd vocabulary.
        dict(name="lm_loss_h500_20x35", kind="lm_loss", H=500, L=2, mb=20, T=35, V=33333),
        # The encoder over a full minibatch: 6400 tokens through four layers.
        dict(name="encode_h1000_128x50", kind="encode", H=1000, L=4, mb=128, T=50, V=50000),
        # A decoder step over a full minibatch with attention over every source position, probabilities out.
        dict(name="decode_step_h1000_128", kind="decode_step", H=1000, L=4, mb=128, S=50, D=50, V=50000, weights="f32", terms=2),
        # The same step with a small model, an odd number of columns and the default attention window.
        dict(name="decode_step_h500_37", kind="decode_step", H=500, L=2, mb=37, S=23, D=10, V=30011, weights="f32", terms=2),
        # Reduced-precision weights at the largest size they are used at, activations rounded to bf16 once.
        dict(name="decode_step_bf16_h2000_256", kind="decode_step", H=2000, L=4, mb=256, S=50, D=50, V=80000, weights="bf16", terms=1),
        # Reduced-precision weights with activations as two bf16 terms (the default), a mid-sized model.
        dict(name="decode_step_bf16_h1024_64", kind="decode_step", H=1024, L=2, mb=64, S=30, D=10, V=40000, weights="bf16", terms=2),
        # One sentence translated on its own, as an interactive user does: 12 columns, every launch counts.
        dict(name="translate_1x12", kind="translate", H=1000, L=4, n_sent=1, beam=12, S=25, steps=30, D=10, V=50000),
        # A batch of 16 sentences, 192 columns, the throughput setting of translation.
        dict(name="translate_16x12", kind="translate", H=1000, L=4, n_sent=16, beam=12, S=50, steps=60, D=10, V=50000),
        # Training a small language model: ragged batch, hidden size off the wide layouts' multiples.
        dict(name="lm_train_h300_20x35", kind="lm_train", H=300, L=2, mb=20, T=35, V=10001),
        # Training the large language model.
        dict(name="lm_train_h1000_128x50", kind="lm_train", H=1000, L=4, mb=128, T=50, V=50000),
        # Training a translation model with attention and feed-input, where the target side goes node by node.
        dict(name="nmt_train_h500_64x20", kind="nmt_train", H=500, L=2, mb=64, S=24, T=20, D=10, V=20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _hidden(rng, lo, hi):
    h = _log_int(rng, lo, hi)
    step = rng.choice([1, 2, 4, 8, 10, 32, 50])
    return min(hi, max(lo, h // step * step))


def draw(rng):
    most = max(work(c)["flops"] for c in listed() if c.get("weights") != "bf16")
    most_bf16 = max(work(c)["flops"] for c in listed() if c.get("weights") == "bf16")
    while True:
        kind = rng.choice(["lm_logprobs", "lm_loss", "encode", "decode_step", "decode_step", "translate", "lm_train", "nmt_train"])
        c = dict(kind=kind, H=_hidden(rng, 64, 1024), L=rng.randint(1, 4))
        v = _log_int(rng, 1000, 50000)
        if kind in ("lm_logprobs", "lm_loss"):
            c.update(mb=_log_int(rng, 1, 64), T=_log_int(rng, 5, 60), V=v)
        elif kind == "encode":
            c.update(mb=_log_int(rng, 1, 256), T=_log_int(rng, 5, 100), V=v)
        elif kind == "decode_step":
            S = rng.randint(4, 60)
            c.update(mb=_log_int(rng, 1, 256), S=S, D=rng.choice([5, 10, S]), V=v, weights="f32", terms=2)
            if rng.random() < 0.4:
                c.update(H=_log_int(rng, 8, 125) * 16, weights="bf16", terms=rng.choice([1, 2]), V=_log_int(rng, 1000, 80000))
        elif kind == "translate":
            S = rng.randint(5, 50)
            c.update(n_sent=_log_int(rng, 1, 16), beam=rng.choice([1, 4, 5, 8, 10, 12]), S=S, steps=rng.randint(5, min(60, S + S // 2)), D=10, V=v)
        elif kind == "lm_train":
            c.update(mb=_log_int(rng, 4, 128), T=_log_int(rng, 5, 60), V=v)
        else:
            c.update(mb=_log_int(rng, 4, 128), S=_log_int(rng, 5, 40), T=_log_int(rng, 5, 30), D=rng.choice([5, 10]), V=v)
        columns = c.get("mb", 1) * c.get("T", 1)
        if work(c)["flops"] <= (most_bf16 if c.get("weights") == "bf16" else most) and columns * c["V"] <= 3.2e8:
            return c


# ---- device memory, random values, weights -------------------------------------------------------------------------

class Dev:
    """A torch tensor's memory in the form the binding takes addresses in."""

    def __init__(self, tensor):
        self.t = tensor
        self.ptr = tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()

    def __int__(self):
        return self.ptr

    def at(self, n):
        return self.ptr + n * self.t.element_size()

    def parts(self):
        """The entries of the leading dimension."""
        return [self.at(i * self.t.stride(0)) for i in range(self.t.shape[0])]


_ctx = None


def _context():
    # One context for the process, as a program has it: the single-launch schedules want the device to themselves.
    global _ctx
    if _ctx is None:
        _ctx = capi.Context(0)
    return _ctx


class Maker:
    """Inputs from one seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.r = np.random.default_rng(seed)

    def uniform(self, *shape, scale=INIT):
        return Dev(torch.empty(shape, device="cuda").uniform_(-scale, scale, generator=self.g))

    def normal(self, *shape, sd=1.0):
        return Dev(torch.empty(shape, device="cuda").normal_(0.0, sd, generator=self.g))

    def zipf(self, V, *shape):
        """Word ids by Zipf's law with exponent 1.1 over ranks, as int32."""
        cdf = torch.cumsum(torch.arange(1, V + 1, device="cuda", dtype=torch.float64) ** -1.1, 0)
        u = torch.rand(shape, device="cuda", dtype=torch.float64, generator=self.g) * cdf[-1]
        return torch.clamp(torch.searchsorted(cdf, u.reshape(-1)).reshape(shape), max=V - 1).to(torch.int32)

    def lengths(self, n, longest):
        """Sentence lengths of one minibatch: the longest one fills it, the others are a little shorter."""
        lens = self.r.integers(max(1, longest * 2 // 3), longest + 1, n)
        lens[self.r.integers(n)] = longest
        return torch.from_numpy(lens.astype(np.int32)).cuda()


def _empty(*shape, dtype=torch.float32):
    return Dev(torch.empty(shape, device="cuda", dtype=dtype))


def _zeros(*shape, dtype=torch.float32):
    return Dev(torch.zeros(shape, device="cuda", dtype=dtype))


class Layer:
    """One LSTM layer's matrices (gate order i, f, c, o) and the handles made from them."""

    def __init__(self, ctx, mk, H, feed=False, bf16=False, train=False, scale=INIT):
        self.ctx, self.H, self.bf16 = ctx, H, bf16
        self.M, self.Wh, self.b = mk.uniform(4, H, H, scale=scale), mk.uniform(4, H, H, scale=scale), mk.uniform(4, H)
        self.Q = mk.uniform(4, H, H, scale=scale) if feed else None
        self.w = self.train = None
        self.pack()
        if train:
            self.train = ctx.lstm_train_create(self.M.parts(), self.Wh.parts(), H)

    def pack(self):
        if self.w is not None:
            self.ctx.lstm_weights_destroy(self.w)
        self.w = self.ctx.lstm_pack(self.M.parts(), self.Wh.parts(), self.b.parts(), self.H, self.Q.parts() if self.Q else None,
                                    bf16=self.bf16)

    def __del__(self):
        if self.w is not None:
            self.ctx.lstm_weights_destroy(self.w)
        if self.train is not None:
            self.ctx.lstm_train_destroy(self.train)


class Output:
    """The output layer with its snapshot in the matrix cores' layout."""

    def __init__(self, ctx, mk, V, H, bf16=False, scale=INIT):
        self.ctx, self.V, self.H, self.bf16 = ctx, V, H, bf16
        self.D, self.b = mk.uniform(H, V, scale=scale), mk.uniform(V)
        self.prepare()

    def prepare(self):
        self.ctx.softmax_prepare(self.D, self.V, self.H, bf16=self.bf16)

    def __del__(self):
        self.ctx.softmax_release(self.D)


ATTENTION = ("W_a", "W_p", "v_p", "out_bias", "W_c1", "W_c2")


class Attention:
    def __init__(self, ctx, mk, H, mb, D, tables, bf16=False):
        self.ctx = ctx
        self.p = {k: mk.uniform(H) if k in ("v_p", "out_bias") else mk.uniform(H, H) for k in ATTENTION}
        self.a = ctx.attn_create(H, mb, D, *[self.p[k] for k in ATTENTION], tables)
        if bf16:
            ctx.attn_use_bf16_weights(self.a)
        else:
            ctx.attn_prepare(self.a)

    def __del__(self):
        self.ctx.attn_destroy(self.a)


class State:
    pass


# ---- preparation ---------------------------------------------------------------------------------------------------

def prepare(case, seed):
    s = State()
    s.ctx, s.c = _context(), dict(case)
    mk = Maker(seed)
    _PREPARE[case["kind"]](s, mk)
    torch.cuda.synchronize()
    return s


def _sweep_buffers(H, L, mb, T, train=False):
    """What a stack sweep over T steps writes."""
    b = State()
    b.zero = _zeros(mb, H)
    b.h = [_empty(T, mb, H) for _ in range(L)]
    b.c = [_empty(T, mb, H) for _ in range(L)]
    b.nn, b.mask = _empty(T * mb, dtype=torch.int32), _empty(T * mb, dtype=torch.int32)
    if train:
        b.gates = [_empty(T, 4, mb, H) for _ in range(L)]
        b.dgates = [_empty(T, mb, 4 * H) for _ in range(L)]
        b.err_h0, b.err_c0 = [_empty(mb, H) for _ in range(L)], [_empty(mb, H) for _ in range(L)]
        b.err_top, b.err_in, b.x = _zeros(T, mb, H), _empty(T, mb, H), _empty(T, mb, H)
    return b


def _target_side(ctx, mk, V, T, mb):
    """Time-major input words of a minibatch, -1 behind the end of a shorter sentence, and the words to be predicted with
    their mask, as the library's index preparation leaves them."""
    on = torch.arange(T, device="cuda")[:, None] < mk.lengths(mb, T)[None, :]
    pad = torch.full((T, mb), -1, device="cuda", dtype=torch.int32)
    ids, words = Dev(torch.where(on, mk.zipf(V, T, mb), pad)), Dev(torch.where(on, mk.zipf(V, T, mb), pad))
    mask, maskf = _empty(T * mb, dtype=torch.int32), _empty(T * mb)
    torch.cuda.synchronize()
    ctx.vocab_prep_softmax(words, T * mb, V, mask, maskf)
    ctx.sync()
    return ids, words, mask


def _source_side(mk, V, S, mb):
    """Time-major source words, left padded with -1, and the lengths and paddings the attention layer is given."""
    lens = mk.lengths(mb, S)
    on = torch.arange(S, device="cuda")[:, None] >= (S - lens)[None, :]
    ids = torch.where(on, mk.zipf(V, S, mb), torch.full((S, mb), -1, device="cuda", dtype=torch.int32))
    return Dev(ids), Dev(torch.cat([lens, S - lens]).to(torch.int32))


def _prepare_lm(s, mk):
    c, ctx = s.c, s.ctx
    H, L, mb, T, V = c["H"], c["L"], c["mb"], c["T"], c["V"]
    train = c["kind"] == "lm_train"
    s.embed = mk.uniform(V, H)
    s.layers = [Layer(ctx, mk, H, train=train) for _ in range(L)]
    s.out = Output(ctx, mk, V, H)
    s.ids, s.targets, s.tmask = _target_side(ctx, mk, V, T, mb)
    s.b = _sweep_buffers(H, L, mb, T, train)
    s.matrix = _empty(T * mb, V)
    if train:
        s.g = _gradients(s.layers, H)
        s.g_out, s.g_b, s.g_embed = _empty(H, V), _empty(V), _empty(V, H)
        s.unstacked = _empty(4, H, H)


def _gradients(layers, H):
    return [dict(M=_empty(H, 4 * H), Wh=_empty(H, 4 * H), b=_empty(4 * H), **({"Q": _empty(H, 4 * H)} if ly.Q else {})) for ly in layers]


def _prepare_encode(s, mk):
    c = s.c
    s.embed = mk.uniform(c["V"], c["H"])
    s.layers = [Layer(s.ctx, mk, c["H"]) for _ in range(c["L"])]
    s.ids, _ = _source_side(mk, c["V"], c["T"], c["mb"])
    s.b = _sweep_buffers(c["H"], c["L"], c["mb"], c["T"])


def _prepare_decode_step(s, mk):
    c, ctx = s.c, s.ctx
    H, L, mb, S, V, bf16 = c["H"], c["L"], c["mb"], c["S"], c["V"], c["weights"] == "bf16"
    s.embed = mk.uniform(V, H)
    s.layers = [Layer(ctx, mk, H, feed=(l == 0), bf16=bf16) for l in range(L)]
    s.out = Output(ctx, mk, V, H, bf16=bf16)
    s.hs = mk.normal(S, mb, H, sd=0.5)
    s.att = Attention(ctx, mk, H, mb, c["D"], s.hs.parts(), bf16=bf16)
    lens = mk.lengths(mb, S)
    s.info = Dev(torch.cat([lens, S - lens]).to(torch.int32))
    s.ids = Dev(mk.zipf(V, mb))
    s.mask = Dev(torch.ones(mb, device="cuda", dtype=torch.int32))
    s.h_prev = [mk.uniform(mb, H, scale=0.5) for _ in range(L)]
    s.c_prev = [mk.uniform(mb, H, scale=0.5) for _ in range(L)]
    s.htild_prev = mk.uniform(mb, H, scale=0.7)
    s.h, s.cell = [_empty(mb, H) for _ in range(L)], [_empty(mb, H) for _ in range(L)]
    s.htild, s.prob = _empty(mb, H), _empty(mb, V)
    slots = 2 * c["D"] + 1
    s.align, s.index = _zeros(slots, mb), _zeros(slots, mb, dtype=torch.int32)


SHARP, ENDS = 8.0, 10.0  # logits of about four units' spread


def _prepare_translate(s, mk):
    c, ctx = s.c, s.ctx
    H, L, V = c["H"], c["L"], c["V"]
    w = State()
    w.ctx, w.H, w.Vs, w.Vt, w.L = ctx, H, V, V, L
    # Values as in a trained model: embeddings of order one, states that use the range of tanh, and peaked output
    # distributions, so that the likeliest word has a probability of some per cent.  The end-of-sentence word (id 1) is
    # likely enough to end hypotheses on the way.
    x = 2.5 / math.sqrt(H)
    w.src_embed, w.tgt_embed = mk.uniform(V, H, scale=1.0), mk.uniform(V, H, scale=1.0)
    s.src_layers = [Layer(ctx, mk, H, scale=x) for _ in range(L)]
    s.tgt_layers = [Layer(ctx, mk, H, feed=(l == 0), scale=x) for l in range(L)]
    w.src, w.tgt = [ly.w for ly in s.src_layers], [ly.w for ly in s.tgt_layers]
    w.attn = {k: mk.uniform(H) if k in ("v_p", "out_bias") else mk.uniform(H, H, scale=2 * x) for k in ATTENTION}
    s.out = Output(ctx, mk, V, H, scale=SHARP * x)
    s.out.b.t[1] = ENDS
    w.D_soft, w.b_soft = s.out.D, s.out.b
    s.w = w
    n = c["n_sent"]
    s.lens = mk.lengths(n, c["S"]).cpu().numpy()
    ids = mk.zipf(V, c["S"], n).cpu().numpy()
    ids[np.arange(c["S"])[:, None] < c["S"] - s.lens[None, :]] = -1
    s.ids = ids


def _prepare_nmt_train(s, mk):
    c, ctx = s.c, s.ctx
    H, L, mb, S, T, V = c["H"], c["L"], c["mb"], c["S"], c["T"], c["V"]
    s.src_embed, s.tgt_embed = mk.uniform(V, H), mk.uniform(V, H)
    s.src_layers = [Layer(ctx, mk, H, train=True) for _ in range(L)]
    s.tgt_layers = [Layer(ctx, mk, H, feed=(l == 0), train=True) for l in range(L)]
    s.src_ids, s.info = _source_side(mk, V, S, mb)
    s.tgt_ids, s.targets, s.tmask = _target_side(ctx, mk, V, T, mb)
    s.src, s.tgt = _sweep_buffers(H, L, mb, S, True), _sweep_buffers(H, L, mb, T, True)
    s.att = Attention(ctx, mk, H, mb, c["D"], s.src.h[L - 1].parts())
    ctx.attn_set_error_tables(s.att.a, s.src.err_top.parts())
    s.out = Output(ctx, mk, V, H)
    slots = 2 * c["D"] + 1
    s.htild, s.align, s.index = _empty(T, mb, H), _zeros(T, slots, mb), _zeros(T, slots, mb, dtype=torch.int32)
    s.p_t, s.ctxv = _empty(T, mb), _empty(T, mb, H)
    s.matrix = _empty(T * mb, V)
    s.err_htild, s.err_feed, s.err_att = _empty(T, mb, H), _empty(mb, H), _empty(mb, H)
    # error to h_{t-1} and, behind it, to the layer below; two of them in turn
    s.err_h = [[_empty(2, mb, H) for _ in range(2)] for _ in range(L)]
    s.err_c = [_empty(mb, H) for _ in range(L)]
    s.g_src, s.g_tgt = _gradients(s.src_layers, H), _gradients(s.tgt_layers, H)
    s.g_att = {k: _empty(H) if k in ("v_p", "out_bias") else _empty(H, H) for k in ATTENTION}
    s.g_out, s.g_b, s.g_src_embed, s.g_tgt_embed = _empty(H, V), _empty(V), _empty(V, H), _empty(V, H)
    s.unstacked = _empty(4, H, H)


_PREPARE = {"lm_logprobs": _prepare_lm, "lm_loss": _prepare_lm, "lm_train": _prepare_lm, "encode": _prepare_encode,
            "decode_step": _prepare_decode_step, "translate": _prepare_translate, "nmt_train": _prepare_nmt_train}


# ---- one pass ------------------------------------------------------------------------------------------------------

def run(s):
    return _RUN[s.c["kind"]](s)


def _forward(s, layers, embed, ids, b, T, h0=None, c0=None, train=False):
    c, ctx = s.c, s.ctx
    ctx.vocab_prep(ids, T * c["mb"], c["V"], b.nn, b.mask)
    z = [b.zero] * c["L"]
    args = ([ly.w for ly in layers], embed, c["V"], b.nn, b.mask, T, c["mb"], h0 or z, c0 or z, b.h, b.c)
    if train:
        ctx.lstm_stack_forward_train(*args, b.gates)
    else:
        ctx.lstm_stack_forward(*args)


def _run_lm_logprobs(s):
    c = s.c
    _forward(s, s.layers, s.embed, s.ids, s.b, c["T"])
    s.ctx.softmax_forward(s.out.D, s.out.b, c["V"], c["H"], s.b.h[-1], c["T"] * c["mb"], capi.ZR_SOFTMAX_LOGPROB, s.matrix)
    return {"logprobs": s.matrix.t, "h": s.b.h[-1].t}


def _run_lm_loss(s):
    c, N = s.c, s.c["T"] * s.c["mb"]
    _forward(s, s.layers, s.embed, s.ids, s.b, c["T"])
    loss = s.ctx.softmax_loss(s.out.D, s.out.b, c["V"], c["H"], s.b.h[-1], N, s.targets, s.tmask, s.matrix)
    return {"loss": loss, "h": [h.t for h in s.b.h], "c_last": [x.t[-1] for x in s.b.c]}


def _run_encode(s):
    _forward(s, s.layers, s.embed, s.ids, s.b, s.c["T"])
    return {"h": [h.t for h in s.b.h], "c": [x.t for x in s.b.c]}


def _run_decode_step(s):
    c, ctx = s.c, s.ctx
    if c["weights"] == "bf16":
        ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, c["terms"])
    ctx.decoder_step([ly.w for ly in s.layers], s.embed, c["V"], s.ids, s.h_prev, s.c_prev, s.mask, c["mb"], s.h, s.cell,
                     s.att.a, s.info, s.htild, s.out.D, s.out.b, c["V"], capi.ZR_SOFTMAX_PROB, s.prob,
                     d_htild_prev=s.htild_prev, d_align=s.align, d_idx=s.index)
    return {"prob": s.prob.t, "h": [x.t for x in s.h], "c": [x.t for x in s.cell], "htild": s.htild.t, "align": s.align.t,
            "index": s.index.t}


def _run_translate(s):
    c = s.c
    d = driver.BeamDecode(s.ctx, s.w, c["beam"], c["n_sent"], c["S"], c["steps"], attention_D=c["D"])
    d.encode(s.ids, s.lens)
    for _ in range(c["steps"]):
        d.step()
    d.finish()
    cap = 4 * c["beam"]
    words = np.full((c["n_sent"], cap, d.max_len), -1, np.int32)
    scores = np.zeros((c["n_sent"], cap), np.float32)
    for i in range(c["n_sent"]):
        for k, (w, score) in enumerate(d.hypotheses(i, cap)):
            words[i, k, :len(w)], scores[i, k] = w, score
    d.close()
    return {"words": words, "scores": scores}


RATE, CLIP = 0.1, 5.0  # learning rate, largest norm of one matrix's gradient


def _update(s, layers, grads):
    """Clipped update of every matrix of a stack, then the copies of them that the products read."""
    ctx, H, sc = s.ctx, s.c["H"], 1.0 / s.c["mb"]
    parts = s.unstacked.parts()
    for ly, g in zip(layers, grads):
        for k in ("M", "Wh", "Q"):
            if k in g:
                ctx.unstack_gates(g[k], H, parts)
                for w, x in zip(getattr(ly, k).parts(), parts):
                    ctx.sgd_update(w, x, H * H, sc, CLIP, RATE)
        for i, w in enumerate(ly.b.parts()):
            ctx.sgd_update(w, g["b"].at(i * H), H, sc, CLIP, RATE)
        ly.pack()
        ctx.lstm_train_refresh(ly.train, ly.M.parts(), ly.Wh.parts())


def _update_rest(s, pairs):
    for w, g in pairs:
        s.ctx.sgd_update(w, g, w.t.numel(), 1.0 / s.c["mb"], CLIP, RATE)


def _side_gradients(s, layers, embed, b, T, h0, grads, g_embed):
    """Weight, bias and embedding gradients of one side from its kept pre-activation errors."""
    c, ctx, N = s.c, s.ctx, T * s.c["mb"]
    ctx.embed_gather(embed, c["H"], c["V"], b.nn, N, b.x)
    for l in range(len(layers)):
        ctx.lstm_weight_gradients(c["H"], T, c["mb"], b.dgates[l], b.x if l == 0 else b.h[l - 1], h0[l], b.h[l], grads[l]["M"],
                                  grads[l]["Wh"], grads[l]["b"])
    ctx.memset_zero(g_embed)
    ctx.embed_gradient(c["H"], c["V"], b.err_in, b.nn, b.mask, N, g_embed)


def _told(layers, grads):
    return [{k: [getattr(ly, k).t, g[k].t] for k in g} for ly, g in zip(layers, grads)]


def _run_lm_train(s):
    c, ctx, b = s.c, s.ctx, s.b
    H, L, mb, T, V, N = c["H"], c["L"], c["mb"], c["T"], c["V"], c["T"] * c["mb"]
    z = [b.zero] * L
    _forward(s, s.layers, s.embed, s.ids, b, T, train=True)
    loss = ctx.softmax_backward_loss(s.out.D, s.out.b, V, H, b.h[-1], N, s.targets, s.tmask, s.matrix, b.err_top, s.g_out, s.g_b)
    ctx.lstm_stack_backward([ly.train for ly in s.layers], T, mb, b.mask, z, b.c, b.gates, b.err_top, b.dgates, b.err_h0,
                            b.err_c0, d_err_below0=b.err_in)
    _side_gradients(s, s.layers, s.embed, b, T, z, s.g, s.g_embed)
    _update_rest(s, [(s.out.D, s.g_out), (s.out.b, s.g_b), (s.embed, s.g_embed)])
    s.out.prepare()
    _update(s, s.layers, s.g)
    return {"loss": loss, "layers": _told(s.layers, s.g), "out": [s.out.D.t, s.out.b.t, s.g_out.t, s.g_b.t],
            "embed": [s.embed.t, s.g_embed.t]}


def _run_nmt_train(s):
    c, ctx, src, tgt = s.c, s.ctx, s.src, s.tgt
    H, L, mb, S, T, V, N, n = c["H"], c["L"], c["mb"], c["S"], c["T"], c["V"], c["T"] * c["mb"], c["H"] * c["mb"]
    z = [src.zero] * L
    # encoder
    _forward(s, s.src_layers, s.src_embed, s.src_ids, src, S, train=True)
    h0, c0 = [h.at((S - 1) * n) for h in src.h], [x.at((S - 1) * n) for x in src.c]
    # decoder, step by step: every step reads the attention output of the one before
    ctx.vocab_prep(s.tgt_ids, N, V, tgt.nn, tgt.mask)
    for t in range(T):
        mask = tgt.mask.at(t * mb)
        for l in range(L):
            hp = tgt.h[l].at((t - 1) * n) if t else h0[l]
            cp = tgt.c[l].at((t - 1) * n) if t else c0[l]
            gates = [tgt.gates[l].at((4 * t + k) * n) for k in range(4)]
            h, x = tgt.h[l].at(t * n), tgt.c[l].at(t * n)
            if l == 0:
                ctx.lstm_step_embed(s.tgt_layers[0].w, s.tgt_embed, V, tgt.nn.at(t * mb), hp, cp, mask, mb, h, x,
                                    d_htild=s.htild.at((t - 1) * n) if t else None, gates=gates)
            else:
                ctx.lstm_step(s.tgt_layers[l].w, tgt.h[l - 1].at(t * n), hp, cp, mask, mb, h, x, gates=gates)
        ctx.attn_step(s.att.a, s.info, tgt.h[L - 1].at(t * n), mask, s.htild.at(t * n), s.align.at(t * s.align.t.stride(0)),
                      s.index.at(t * s.index.t.stride(0)), s.p_t.at(t * mb), s.ctxv.at(t * n))
    # loss and errors of every h~
    loss = ctx.softmax_backward_loss(s.out.D, s.out.b, V, H, s.htild, N, s.targets, s.tmask, s.matrix, s.err_htild, s.g_out, s.g_b)
    # back through the decoder
    ctx.memset_zero(src.err_top)
    ctx.memset_zero(s.g_tgt[0]["Q"])
    for k in ATTENTION:
        ctx.memset_zero(s.g_att[k])
    for t in range(T - 1, -1, -1):
        mask, last = tgt.mask.at(t * mb), t == T - 1
        if not last:
            ctx.add_inplace(s.err_htild.at(t * n), s.err_feed, n)
        ctx.attn_backward(s.att.a, s.info, tgt.h[L - 1].at(t * n), mask, s.htild.at(t * n), s.align.at(t * s.align.t.stride(0)),
                          s.index.at(t * s.index.t.stride(0)), s.p_t.at(t * mb), s.ctxv.at(t * n), s.err_htild.at(t * n),
                          s.err_att, [s.g_att[k] for k in ATTENTION])
        above = s.err_att
        for l in range(L - 1, -1, -1):
            here, after = s.err_h[l][t % 2], s.err_h[l][1 - t % 2]
            below = tgt.err_in.at(t * n) if l == 0 else here.at(n)
            ctx.lstm_node_backward(s.tgt_layers[l].train, mb, [tgt.gates[l].at((4 * t + k) * n) for k in range(4)],
                                   tgt.c[l].at(t * n), tgt.c[l].at((t - 1) * n) if t else c0[l], mask, above,
                                   None if last else after, None if last else s.err_c[l], tgt.dgates[l].at(4 * t * n), here,
                                   s.err_c[l], below)
            above = below
        if t:
            ctx.lstm_feed_backward(s.tgt_layers[0].Q.parts(), H, mb, tgt.dgates[0].at(4 * t * n), s.htild.at((t - 1) * n),
                                   s.err_feed, s.g_tgt[0]["Q"])
    _side_gradients(s, s.tgt_layers, s.tgt_embed, tgt, T, h0, s.g_tgt, s.g_tgt_embed)
    # back through the encoder: errors of the source states from the attention nodes, of the last state from the decoder
    ctx.lstm_stack_backward([ly.train for ly in s.src_layers], S, mb, src.mask, z, src.c, src.gates, src.err_top, src.dgates,
                            src.err_h0, src.err_c0, err_hT=[s.err_h[l][0] for l in range(L)], err_cT=s.err_c,
                            d_err_below0=src.err_in)
    _side_gradients(s, s.src_layers, s.src_embed, src, S, z, s.g_src, s.g_src_embed)
    _update_rest(s, [(s.out.D, s.g_out), (s.out.b, s.g_b), (s.src_embed, s.g_src_embed), (s.tgt_embed, s.g_tgt_embed)]
                 + [(s.att.p[k], s.g_att[k]) for k in ATTENTION])
    s.out.prepare()
    ctx.attn_prepare(s.att.a)
    _update(s, s.src_layers, s.g_src)
    _update(s, s.tgt_layers, s.g_tgt)
    return {"loss": loss, "src": _told(s.src_layers, s.g_src), "tgt": _told(s.tgt_layers, s.g_tgt),
            "att": [s.g_att[k].t for k in ATTENTION], "out": [s.out.D.t, s.g_out.t, s.g_b.t],
            "embed": [s.src_embed.t, s.g_src_embed.t, s.tgt_embed.t, s.g_tgt_embed.t], "htild": s.htild.t}


_RUN = {"lm_logprobs": _run_lm_logprobs, "lm_loss": _run_lm_loss, "lm_train": _run_lm_train, "encode": _run_encode,
        "decode_step": _run_decode_step, "translate": _run_translate, "nmt_train": _run_nmt_train}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def work(case):
    c = case
    H, L, V, kind = c["H"], c["L"], c["V"], c["kind"]
    hh = 4.0 * H * H  # one H x H matrix of 32-bit values

    def stack(columns, feed=0):  # multiply-adds of the LSTM products: 4 gates, input and recurrent matrix, two operations each
        return 2.0 * 4 * H * H * columns * (2 * L + feed)

    def att(columns):
        return 2.0 * 4 * H * H * columns

    logits = 2.0 * V * H
    if kind in ("lm_logprobs", "lm_loss", "encode"):
        N = c["mb"] * c["T"]
        b, f = 8 * L * hh + 4.0 * H * N, stack(N)
        if kind == "encode":
            return {"bytes": b + 8.0 * L * H * N, "flops": f}
        b += 4.0 * V * H + 4.0 * H * N
        return {"bytes": b + (4.0 * V * N if kind == "lm_logprobs" else 4.0 * L * H * N), "flops": f + logits * N}
    if kind == "decode_step":
        mb, w = c["mb"], (0.5 if c["weights"] == "bf16" else 1.0)
        slots = min(2 * c["D"] + 1, c["S"])
        b = w * ((8 * L + 4 + 4) * hh + 4.0 * V * H) + 4.0 * H * mb * (slots + 4 * L + 3) + 4.0 * V * mb
        return {"bytes": b, "flops": stack(mb, 1) + att(mb) + logits * mb}
    if kind == "translate":
        cols, n = c["n_sent"] * c["beam"], c["steps"] + 1
        slots = min(2 * c["D"] + 1, c["S"])
        step_b = (8 * L + 4 + 4) * hh + 4.0 * V * H + 4.0 * H * cols * (slots + 4 * L + 3)
        step_f = stack(cols, 1) + att(cols) + logits * cols
        return {"bytes": n * step_b + 8 * L * hh, "flops": n * step_f + stack(c["n_sent"] * c["S"])}
    if kind == "lm_train":
        N = c["mb"] * c["T"]
        weights = 8 * L * hh + 8.0 * V * H  # the stack, the output layer and the embedding
        return {"bytes": 4 * weights + 4.0 * H * N * L * 12, "flops": 3 * (stack(N) + logits * N)}
    N, M = c["mb"] * c["T"], c["mb"] * c["S"]
    weights = (16 * L + 4 + 4) * hh + 12.0 * V * H
    return {"bytes": 4 * weights + 4.0 * H * (N + M) * L * 12, "flops": 3 * (stack(N, 1) + stack(M) + att(N) + logits * N)}


def tolerance(case):
    """About four times what the path's own summation orders (other schedules, tiles and splits of the same products)
    differ by; `differ` allows for words and window positions that lie closer together than the sums' rounding."""
    if case["kind"] in ("lm_train", "nmt_train"):
        # sums over all columns of a minibatch, most of whose terms cancel: 1.7e-5, single elements 4e-4
        return {"rel": 7e-5, "max": 2e-3, "differ": 0.005}
    if case.get("weights") == "bf16":
        # Activations are rounded to bf16: a change in the last place of one that lies between two bf16 values moves it
        # by 2^-8 (one term) or 2^-16 (two terms).  Inputs changed by 2e-7 move the results by 2.4e-3, single elements
        # by 5e-2 (one term), and by 4e-6 and 4e-5 (two terms).
        return {"rel": 1e-2, "max": 0.2, "differ": 0.005} if case["terms"] == 1 else {"rel": 2e-5, "max": 2e-4, "differ": 0.005}
    # 32-bit sums of up to a few thousand terms through a few layers: 9e-7, single elements 7e-6
    return {"rel": 4e-6, "max": 4e-5, "differ": 0.005}
