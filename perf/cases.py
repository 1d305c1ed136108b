"""What a user of this framework has it do, as cases that can be timed and compared.

``listed()`` holds one case of each kind of use at a size the benchmark or the configurations name, ``draw()``
more of the same kinds over their ranges.  A kind is a way through the public entry points:

  host        one matrix-vector product through host pointers (the drop-in single-token call)
  host_batch  a batch of vectors through host pointers (the drop-in prefill call)
  gemv        one decode launch on device buffers, 1-8 vectors, any weight type
  step        the independent matmuls of a decode step as one plan launch
  chain       the dependent chain a decode step is, norms, residuals and SwiGLU inside, as one plan launch
  step_q80    the same for Q8_0 kept tile-major, 1-16 sequences decoding together
  batch       one matrix under a small batch (9-64 vectors), columns shared between workgroups
  prefill     one matrix under a prompt (65 vectors and more)
  moe         a mixture-of-experts layer from router logits to combined output

Weights are random blocks of the type in question: every code and scale uniform over its bits, the half-precision
factors |N(0, 0.02)| (Q8_0: |N(0, 0.01)|, values in -127..127; Q6_K: scales in -32..31); activations, router
logits and inputs are N(0, 1).
"""
import ctypes
import math

import numpy as np
import torch

from oxidize_amd import _lib
from oxidize_amd import matvec as mv

# type id -> (values per block, bytes per block, places of the half-precision factors)
BLOCKS = {
    3: (32, 18, (0,)), 4: (32, 20, (0, 2)), 5: (32, 22, (0,)), 6: (32, 24, (0, 2)), 7: (32, 34, (0,)),
    8: (256, 84, (80, 82)), 10: (256, 110, (108,)), 13: (256, 144, (0, 2)), 15: (256, 176, (0, 2)),
    16: (256, 210, (208,)), 18: (32, 14, (0,)), 25: (256, 110, (0,)), 26: (32, 18, (0,)), 27: (256, 136, (0,)),
    36: (256, 38, (0,)),
}
Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, AL5_XS, IQ3_S, IQ4_NL, IQ4_XS, IQ1_XXXS = (
    3, 4, 5, 6, 7, 8, 10, 13, 15, 16, 18, 25, 26, 27, 36)
F32_INPUT = (IQ4_NL, IQ4_XS)
TILE_MAJOR = {Q4_K: mv.Q4_K_T16, Q5_K: mv.Q5_K_T16, Q8_0: mv.Q8_0_T16}      # types with a tile-major form


def listed():
    return [
        # the smallest call there is: one attention output projection of the small Q8_0 model, host to host
        dict(name="host_q8_0_896", kind="host", qtype=Q8_0, rows=896, cols=896),
        # a chunk of a prompt through the drop-in batch call: copies each way, registry, quantiser, tiles
        dict(name="host_batch_q4k_64", kind="host_batch", qtype=Q4_K, rows=14336, cols=4096, n_vec=64),
        # one decode launch by itself: gate and up of a Q5_K file
        dict(name="gemv_q5k_28672", kind="gemv", qtype=Q5_K, rows=28672, cols=4096, n_vec=1),
        # configuration 1: the decode set of the 8B shapes, Q4_K with Q6_K down projections: 4.4 GB in one launch
        dict(name="step_llama3_8b", kind="step", qtype=Q4_K, qtype_down=Q6_K, hidden=4096, kv=1024, ffn=14336,
             layers=32),
        # the same matrices as the dependent chain a token really is
        dict(name="chain_llama3_8b", kind="chain", qtype=Q4_K, qtype_down=Q6_K, hidden=4096, kv=1024, ffn=14336,
             layers=32),
        # configuration 2: the small Q8_0 model with its vocabulary head, eight sequences decoding together
        dict(name="step_qwen_q8_0_b8", kind="step_q80", hidden=896, kv=128, ffn=4864, layers=24, vocab=151936,
             n_vec=8),
        # sixteen sequences over a matrix of few rows and many columns: the shape that leaves a device idle
        dict(name="batch16_q6k_down", kind="batch", qtype=Q6_K, rows=4096, cols=14336, n_vec=16),
        # configuration 3: a prompt of 512 tokens over the gate projection
        dict(name="prefill_q4k_512", kind="prefill", qtype=Q4_K, rows=14336, cols=4096, n_vec=512),
        # a prompt whose length fits no tile, over the down projection of a mixed-type file
        dict(name="prefill_q6k_333", kind="prefill", qtype=Q6_K, rows=4096, cols=14336, n_vec=333),
        # the 32-value family under a prompt
        dict(name="prefill_q8_0_512", kind="prefill", qtype=Q8_0, rows=4096, cols=4096, n_vec=512),
        # configuration 4: eight experts, top-2, sixteen decoding tokens; and the same layer under a prompt
        dict(name="moe_16", kind="moe", qtype=Q4_K, qtype_down=Q4_K, n_expert=8, top_k=2, hidden=4096, ffn=14336,
             n_tok=16),
        dict(name="moe_512", kind="moe", qtype=Q4_K, qtype_down=Q4_K, n_expert=8, top_k=2, hidden=4096, ffn=14336,
             n_tok=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, qtype, lo, hi):
    """A row length: log-uniform in whole blocks (tile-major Q8_0 takes whole runs of four)."""
    unit = BLOCKS[qtype][0]
    return max(1, _log_int(rng, lo, hi) // unit) * unit


def draw(rng):
    kind = rng.choice(("host", "host_batch", "gemv", "gemv", "step", "chain", "step_q80", "batch", "batch", "prefill",
                       "prefill", "prefill", "moe", "moe"))
    if kind == "host":
        qt = rng.choice((Q4_K, Q5_K, Q6_K, Q8_0, Q4_0, Q3_K))
        return dict(kind=kind, qtype=qt, rows=_log_int(rng, 100, 28672), cols=_cols(rng, qt, 512, 14336))
    if kind == "host_batch":
        qt = rng.choice((Q4_K, Q5_K, Q6_K, Q8_0, Q4_0, Q3_K))
        return dict(kind=kind, qtype=qt, rows=_log_int(rng, 800, 14336), cols=_cols(rng, qt, 800, 14336),
                    n_vec=_log_int(rng, 2, 512))
    if kind == "gemv":
        qt = rng.choice((Q4_K, Q4_K, Q5_K, Q6_K, Q8_0, Q2_K, Q3_K, Q4_0, Q4_1, Q5_0, Q5_1, AL5_XS, IQ3_S, IQ4_NL, IQ4_XS,
                         IQ1_XXXS))
        wide = qt in F32_INPUT or qt in (IQ3_S, IQ1_XXXS)
        cols = _cols(rng, qt, 800, 14336)
        return dict(kind=kind, qtype=qt, rows=_log_int(rng, 4096, 60000), cols=cols,
                    n_vec=1 if wide or rng.random() < 0.5 else rng.randint(2, 8 if cols <= 8192 else 4))
    if kind in ("step", "chain"):
        hidden = 256 * rng.randint(4, 20)
        qt, qd = rng.choice(((Q4_K, Q6_K), (Q4_K, Q4_K), (Q5_K, Q6_K)))
        return dict(kind=kind, qtype=qt, qtype_down=qd, hidden=hidden, kv=hidden // rng.choice((1, 2, 4)),
                    ffn=256 * max(4, int(hidden * rng.uniform(2.0, 3.2)) // 256), layers=rng.randint(4, 16))
    if kind == "step_q80":
        hidden = 128 * rng.randint(5, 16)
        return dict(kind=kind, hidden=hidden, kv=128 * rng.randint(1, 4),
                    ffn=128 * min(56, int(hidden * rng.uniform(2.5, 5.5)) // 128), layers=rng.randint(4, 24),
                    vocab=_log_int(rng, 32000, 151936), n_vec=rng.randint(1, 16))
    if kind == "batch":
        qt = rng.choice((Q4_K, Q5_K, Q6_K))
        return dict(kind=kind, qtype=qt, rows=_log_int(rng, 500, 16384), cols=_cols(rng, qt, 2048, 14336),
                    n_vec=_log_int(rng, 9, 64))
    if kind == "prefill":
        qt = rng.choice((Q4_K, Q4_K, Q5_K, Q6_K, Q6_K, Q8_0, Q8_0, Q2_K, Q3_K, Q4_0, Q4_1, Q5_0, Q5_1, AL5_XS))
        rows, cols = _log_int(rng, 800, 16384), _cols(rng, qt, 800, 14336)
        return dict(kind=kind, qtype=qt, rows=rows, cols=cols, n_vec=min(_log_int(rng, 65, 1024), 10 ** 11 // (rows * cols)))
    qt = rng.choice((Q4_K, Q4_K, Q5_K))
    hidden = 256 * rng.randint(4, 16)
    ffn, top_k = 256 * max(2, int(hidden * rng.uniform(0.7, 3.5)) // 256), rng.randint(1, 3)
    return dict(kind=kind, qtype=qt, qtype_down=rng.choice((qt, qt, Q6_K)), n_expert=rng.choice((4, 8, 8, 16)), top_k=top_k,
                hidden=hidden, ffn=ffn, n_tok=min(_log_int(rng, 1, 1024), 6 * 10 ** 10 // (top_k * hidden * ffn)))


# ─── sizes ──────────────────────────────────────────────────────────────


def _row_bytes(qt, cols):
    elems, size, _ = BLOCKS[qt]
    return cols // elems * size


def _layer_ops(c):
    """(rows of each matrix, cols, type) of a layer's four matmuls."""
    h, kv, ffn = c["hidden"], c["kv"], c["ffn"]
    qt, qd = c.get("qtype", Q8_0), c.get("qtype_down", Q8_0)
    return [([h, kv, kv], h, qt), ([h], h, qt), ([ffn, ffn], h, qt), ([h], ffn, qd)]


def work(case):
    """Packed weights and f32 inputs read once, f32 outputs written once; two operations per weight and vector."""
    c, kind = case, case["kind"]
    if kind in ("step", "chain", "step_q80"):
        nv = c.get("n_vec", 1)
        ops = _layer_ops(c) * c["layers"] + ([([c["vocab"]], c["hidden"], Q8_0)] if kind == "step_q80" else [])
        weights = sum(sum(rows) * _row_bytes(qt, cols) for rows, cols, qt in ops)
        flops = sum(2 * sum(rows) * cols * nv for rows, cols, _ in ops)
        if kind == "chain":         # what the chain takes in and gives out: the norm weights, x, f; x, f
            return dict(bytes=weights + 4 * c["hidden"] * (2 * c["layers"] + 4), flops=flops)
        return dict(bytes=weights + 4 * nv * sum(cols + sum(rows) for rows, cols, _ in ops), flops=flops)
    if kind == "moe":
        e, k, t, h, ffn = c["n_expert"], c["top_k"], c["n_tok"], c["hidden"], c["ffn"]
        hit = e * (1.0 - (1.0 - k / e) ** t)            # experts that get a token, on average
        per_expert = 2 * ffn * _row_bytes(c["qtype"], h) + h * _row_bytes(c["qtype_down"], ffn)
        return dict(bytes=hit * per_expert + 4 * t * (e + 2 * h), flops=6 * t * k * h * ffn)
    nv = c.get("n_vec", 1)
    return dict(bytes=c["rows"] * _row_bytes(c["qtype"], c["cols"]) + 4 * nv * (c["rows"] + c["cols"]),
                flops=2 * c["rows"] * c["cols"] * nv)


def tolerance(case):
    """Integer sums are exact and the order of the float steps is the framework's stated contract, so every matmul gives
    the same bits, and so does the chain (its norms are summed in one stated order; in any other order a code of the next
    input moves sooner or later, and the stream ends up 2-5 % apart).  The expert layer's silu and softmax are held to
    rounding only: inputs changed by 1e-7 of themselves move its output by up to 5e-4 (2-norm) and 0.023 of the root mean
    square (one value), through the codes that move in between."""
    return dict(rel=2e-3, max=0.1) if case["kind"] == "moe" else "exact"


# ─── inputs ─────────────────────────────────────────────────────────────


class Inputs:
    """Seeded random weights and vectors on the device."""

    def __init__(self, seed):
        _lib.check(_lib.lib().oxh_init(0))
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed * 7919 + 17)

    def weights(self, qt, rows, cols, signed=False):
        elems, size, halves = BLOCKS[qt]
        n = rows * (cols // elems)
        w = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=self.gen)
        if qt == Q8_0:
            w[w == 128] = 129                           # values in -127..127
        elif qt == Q6_K:
            sc = torch.randint(-32, 32, (n, 16), dtype=torch.int8, device="cuda", generator=self.gen)
            w[:, 192:208] = sc.view(torch.uint8)
        sigma = 0.01 if qt == Q8_0 else 0.02
        for at in halves:
            d = torch.randn(n, 1, device="cuda", generator=self.gen) * sigma
            w[:, at:at + 2] = (d if signed else d.abs()).to(torch.float16).view(torch.uint8)
        return w.view(-1)

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", generator=self.gen)


def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device="cuda")


def _floats(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _tile_major(qt, w, rows, cols):
    t = _bytes(mv.tile16_bytes(qt, rows, cols))
    torch.cuda.synchronize()
    mv.tile16(qt, w.data_ptr(), rows, cols, t.data_ptr())
    mv.sync()
    return t


def _decode_form(qt, w, rows, cols):
    """Q6_K as the decode kernels read it fastest, where the row length allows it."""
    if qt != Q6_K or cols % 2048:
        return qt, w
    g = _bytes(w.numel())
    torch.cuda.synchronize()
    mv.q6_k_group(w.data_ptr(), rows, cols, g.data_ptr())
    mv.sync()
    return mv.Q6_K_G8, g


class HostMatrix:
    """A packed matrix in host memory, registered as a model file's tensors are."""

    def __init__(self, w):
        self.data = w.cpu().numpy()
        _lib.check(_lib.lib().oxh_weight_register(ctypes.c_void_p(self.data.ctypes.data), self.data.nbytes))

    def __del__(self):
        _lib.lib().oxh_weight_unregister(ctypes.c_void_p(self.data.ctypes.data))


def prepare(case, seed):
    s = PREPARE[case["kind"]](case, Inputs(seed))
    s["case"] = case
    torch.cuda.synchronize()
    return s


def _prepare_host(c, inp):
    nv = c.get("n_vec", 1)
    s = dict(w=HostMatrix(inp.weights(c["qtype"], c["rows"], c["cols"])), x=inp.normal(nv, c["cols"]).cpu().numpy(),
             out=np.zeros((nv, c["rows"]), np.float32), temp=np.zeros(c["cols"], np.float32),
             row_bytes=_row_bytes(c["qtype"], c["cols"]))
    if c["kind"] == "host_batch":
        s["scratch"] = np.zeros(mv.batch_scratch_bytes(c["cols"]), np.uint8)
    return s


def _prepare_gemv(c, inp):
    w, x = inp.weights(c["qtype"], c["rows"], c["cols"]), inp.normal(c["n_vec"], c["cols"])
    out = _floats(c["n_vec"], c["rows"])
    qt, w = _decode_form(c["qtype"], w, c["rows"], c["cols"]) if c["n_vec"] == 1 else (c["qtype"], w)
    act = None if c["qtype"] in F32_INPUT else _bytes(c["n_vec"] * mv.act_bytes(c["qtype"], c["cols"]))
    return dict(w=w, qtype=qt, x=x, out=out, act=act, segs=mv.make_segments([(w.data_ptr(), out.data_ptr(), c["rows"], 0)]))


def _layers(c, inp, signed=False):
    """Per layer and matmul: the run type and the matrices, in the form the decode kernels read."""
    layers = []
    for _ in range(c["layers"]):
        ops = []
        for rows, cols, qt in _layer_ops(c):
            forms = [_decode_form(qt, inp.weights(qt, r, cols, signed), r, cols) for r in rows]
            ops.append((forms[0][0], [w for _, w in forms]))
        layers.append(ops)
    return layers


def _prepare_step(c, inp):
    layers = _layers(c, inp)
    shapes = _layer_ops(c)
    x = inp.normal(c["layers"], sum(cols for _, cols, _ in shapes))
    out = torch.zeros(c["layers"], sum(sum(rows) for rows, _, _ in shapes), device="cuda")
    ops = []
    for l, mats in enumerate(layers):
        at_x = at_o = 0
        for (rows, cols, _), (run, ws) in zip(shapes, mats):
            items = []
            for r, w in zip(rows, ws):
                items.append((w.data_ptr(), out[l, at_o:].data_ptr(), r, 0))
                at_o += r
            ops.append(dict(qtype=run, segs=mv.make_segments(items), cols=cols, d_x=x[l, at_x:].data_ptr()))
            at_x += cols
    torch.cuda.synchronize()
    return dict(keep=layers, x=x, out=out, plan=mv.Plan(ops))


def _prepare_chain(c, inp):
    """Per layer: q/k/v of the normalised residual stream, o, gate/up with SwiGLU, down; the q projection stands in
    for the attention output, which this framework does not compute.  The factors carry signs here: over weights that
    are all positive every row answers a vector's mean, and the gates of a layer end up all open or all shut."""
    layers = _layers(c, inp, signed=True)
    h, kv, ffn, eps = c["hidden"], c["kv"], c["ffn"], 1e-5
    g = inp.normal(c["layers"], 2, h) * 0.1 + 1.0
    x0, f0 = inp.normal(h), torch.zeros(h, device="cuda")
    res = torch.zeros(3, h, device="cuda")
    qkv, o, hid, f = (torch.zeros(n, device="cuda") for n in (h + 2 * kv, h, ffn, h))
    ops, x, add, turn = [], x0, f0, 0
    for l, mats in enumerate(layers):
        x1, x2 = res[turn % 3], res[(turn + 1) % 3]
        turn += 2
        q, k, v = mats[0][1]
        ops.append(dict(qtype=mats[0][0], cols=h, d_x=x.data_ptr(), kind=mv.PRO_RMSNORM, d_b=g[l, 0].data_ptr(), eps=eps,
                        d_add=add.data_ptr(), d_sum_out=x1.data_ptr(),
                        segs=mv.make_segments([(q.data_ptr(), qkv.data_ptr(), h, 0),
                                               (k.data_ptr(), qkv[h:].data_ptr(), kv, 0),
                                               (v.data_ptr(), qkv[h + kv:].data_ptr(), kv, 0)])))
        ops.append(dict(qtype=mats[1][0], cols=h, d_x=qkv.data_ptr(),
                        segs=mv.make_segments([(mats[1][1][0].data_ptr(), o.data_ptr(), h, 0)])))
        gate, up = mats[2][1]
        ops.append(dict(qtype=mats[2][0], cols=h, d_x=x1.data_ptr(), kind=mv.PRO_RMSNORM, d_b=g[l, 1].data_ptr(), eps=eps,
                        d_add=o.data_ptr(), d_sum_out=x2.data_ptr(),
                        segs=mv.make_segments([(gate.data_ptr(), hid.data_ptr(), ffn, 0, 0, up.data_ptr())])))
        ops.append(dict(qtype=mats[3][0], cols=ffn, d_x=hid.data_ptr(),
                        segs=mv.make_segments([(mats[3][1][0].data_ptr(), f.data_ptr(), h, 0)])))
        x, add = x2, f
    torch.cuda.synchronize()
    return dict(keep=(layers, g, x0, f0, res), plan=mv.Plan(ops), x=x, f=f, qkv=qkv, o=o, h=hid)


def _prepare_step_q80(c, inp):
    nv, keep, ops = c["n_vec"], [], []
    shapes = _layer_ops(c) * c["layers"] + [([c["vocab"]], c["hidden"], Q8_0)]
    x = inp.normal(sum(nv * cols for _, cols, _ in shapes))
    out = torch.zeros(sum(nv * sum(rows) for rows, _, _ in shapes), device="cuda")
    at_x = at_o = 0
    for rows, cols, qt in shapes:
        items, off = [], 0
        for r in rows:
            t = _tile_major(qt, inp.weights(qt, r, cols), r, cols)
            keep.append(t)
            items.append((t.data_ptr(), out[at_o + off:].data_ptr(), r, 0, nv))
            off += r
        ops.append(dict(qtype=mv.Q8_0_T16, segs=mv.make_segments(items), cols=cols, d_x=x[at_x:].data_ptr(), out_stride=off))
        at_x += nv * cols
        at_o += nv * off
    torch.cuda.synchronize()
    return dict(keep=keep, x=x, out=out, plan=mv.Plan(ops))


def _prepare_matmul(c, inp):
    qt, rows, cols, nv = c["qtype"], c["rows"], c["cols"], c["n_vec"]
    w, run = inp.weights(qt, rows, cols), qt
    if qt in (Q2_K, Q3_K):                              # rewritten once for the matrix cores
        wide = _bytes(rows * (cols // 256) * 210)
        torch.cuda.synchronize()
        (mv.q2_k_widen if qt == Q2_K else mv.q3_k_as_q6_k)(w.data_ptr(), rows, cols, wide.data_ptr())
        mv.sync()
        w, run = wide, mv.Q2_K_WIDE if qt == Q2_K else Q6_K
    s = dict(w=w, run=run, x=inp.normal(nv, cols), act=_bytes(nv * mv.act_bytes(qt, cols)), out=_floats(nv, rows))
    if c["kind"] == "batch":
        s["ws_bytes"] = mv.mmq_split_workspace(run, rows, cols, nv, rows)
        s["ws"] = _bytes(max(16, s["ws_bytes"]))
    return s


def _prepare_moe(c, inp):
    e, h, ffn, t = c["n_expert"], c["hidden"], c["ffn"], c["n_tok"]
    mats, run = [], []
    for qt, rows, cols in ((c["qtype"], ffn, h), (c["qtype"], ffn, h), (c["qtype_down"], h, ffn)):
        w = inp.weights(qt, e * rows, cols)
        mats.append(_tile_major(qt, w, e * rows, cols) if qt in TILE_MAJOR else w)
        run.append(TILE_MAJOR.get(qt, qt))
    layer = mv.MoeLayer(run[0], run[2], *[w.data_ptr() for w in mats], e, c["top_k"], h, ffn, max_tok=t)
    return dict(keep=mats, layer=layer, logits=inp.normal(t, e), x=inp.normal(t, h), out=_floats(t, h))


PREPARE = dict(host=_prepare_host, host_batch=_prepare_host, gemv=_prepare_gemv, step=_prepare_step, chain=_prepare_chain,
               step_q80=_prepare_step_q80, batch=_prepare_matmul, prefill=_prepare_matmul, moe=_prepare_moe)


# ─── one pass ───────────────────────────────────────────────────────────


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "host":
        mv.matvec_quantized(c["qtype"], s["w"].data, c["rows"], c["cols"], s["row_bytes"], s["x"], s["out"], s["temp"])
        return s["out"]
    if kind == "host_batch":
        mv.matvec_quantized_batch(c["qtype"], s["w"].data, c["rows"], c["cols"], s["row_bytes"], s["x"], c["cols"], s["out"],
                                  c["rows"], c["n_vec"], s["temp"], s["scratch"])
        return s["out"]
    if kind == "gemv":
        mv.gemv_segments_f32(s["qtype"], s["segs"], c["cols"], s["x"].data_ptr(), c["cols"],
                             None if s["act"] is None else s["act"].data_ptr(), c["n_vec"], c["rows"])
        return s["out"]
    if kind in ("step", "step_q80"):
        s["plan"].launch()
        return s["out"]
    if kind == "chain":
        s["plan"].launch()
        return {k: s[k] for k in ("x", "f", "qkv", "o", "h")}
    if kind == "moe":
        s["layer"].forward(s["logits"].data_ptr(), s["x"].data_ptr(), c["n_tok"], s["out"].data_ptr())
        return s["out"]
    mv.quantize(c["qtype"], s["x"].data_ptr(), c["cols"], c["n_vec"], c["cols"], s["act"].data_ptr())
    if kind == "batch":
        mv.mmq_split(s["run"], s["w"].data_ptr(), c["rows"], c["cols"], s["act"].data_ptr(), c["n_vec"], s["out"].data_ptr(),
                     c["rows"], s["ws"].data_ptr(), s["ws_bytes"])
    else:
        mv.mmq(s["run"], s["w"].data_ptr(), c["rows"], c["cols"], s["act"].data_ptr(), c["n_vec"], s["out"].data_ptr(),
               c["rows"])
    return s["out"]
