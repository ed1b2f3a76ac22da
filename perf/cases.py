"""The work a user of this framework has it do, as measurable cases.

Every case goes through the public Python entry points (hyperscalees_amd.kernels, .snn,
.snn_attention, .rwkv, .rwkv_lm).  Whole training steps stand beside the single layers they
are made of; sizes are the configurations of bench.py and of the tests, and ragged ones.
`exact` restates each path in float64 torch: the noise streams, the perturbed products, the
spiking dynamics, the RWKV-7 recurrence and the ES gradients.
"""
import math

import numpy as np
import torch

from hyperscalees_amd import kernels as K
from hyperscalees_amd import rwkv, rwkv_lm, snn, snn_attention

DEV = "cuda"
MATH = {"f32": K.MATH_F32, "bf16": K.MATH_BF16, "f32x": K.MATH_F32X}
ACTS = {"none": 0, "tanh": 1, "sigmoid": 2, "relu_sq": 3}


# ---- the cases ---------------------------------------------------------------------------

def listed():
    return [
        # The headline training step: SNN-MLP population of 8192, rank 128, fp32-accurate.
        dict(name="mlp_step", op="mlp_step", math="f32x", n=8192, rank=128, T=16, rows=64,
             d_in=784, hidden=128, layers=3, classes=10),
        # A small research run of the same model: fp32, rank 4, launch-bound layers.
        dict(name="mlp_step_small", op="mlp_step", math="f32", n=256, rank=4, T=8, rows=64,
             d_in=784, hidden=128, layers=3, classes=10),
        # The spiking self-attention transformer's training step: many small projections.
        dict(name="attention_step", op="attention_step", n=1024, rank=8, T=8, ntok=64, d_model=64,
             heads=4, blocks=2),
        # The RWKV-7 language model scored by a population (the forward of its ES step).
        dict(name="lm_forward", op="lm", math="bf16", n=2048, rank=1, T=128, layers=4, d_model=512,
             state=False),
        # Generation: a few members, one token per call from the carried state (latency).
        dict(name="lm_decode", op="lm", math="bf16", n=8, rank=1, T=1, layers=4, d_model=512,
             state=True),
        # One hidden spiking layer of a smaller ragged model: draw, member weights, GEMM + LIF.
        dict(name="spiking_layer", op="spiking_layer", math="f32x", n=501, rank=48, T=8, rows=32,
             b=300, a=100),
        # One square EggRoll layer in fp32 at rank 1 (16 rows per member).
        dict(name="linear_fp32", op="linear", math="f32", n=4096, rank=1, rows=16, a=1024, b=1024,
             tmm=False, bf16_x=False, act="none", bf16_y=False),
        # A feed-forward expansion in bf16 with its activation, a ragged population.
        dict(name="linear_bf16", op="linear", math="bf16", n=1000, rank=1, rows=100, a=2048, b=512,
             tmm=False, bf16_x=True, act="relu_sq", bf16_y=True),
        # A TimeMixing block in fp32 continuing from a state (prefill of odd length).
        dict(name="time_mixing", op="time_mixing", math="f32", n=48, rank=1, T=37, d_model=256,
             layer=1),
        # The ES gradient of a square layer at rank 1, and of a ragged one at a larger rank.
        dict(name="es_update", op="es_update", n=4096, rank=1, a=1024, b=1024),
        dict(name="es_update_wide", op="es_update", n=3001, rank=48, a=200, b=500),
        # Rate coding and the LIF scan outside the fused layers, any T and width.
        dict(name="encode_lif", op="encode_lif", T=20, rows=10000, b=500, h=130),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("mlp_step", "mlp_step", "attention_step", "lm", "lm", "spiking_layer", "linear",
                     "linear", "linear", "time_mixing", "es_update", "es_update", "encode_lif"))
    if op == "mlp_step":
        if rng.random() < 0.5:
            return dict(op=op, math=rng.choice(("f32x", "bf16")), n=_log(rng, 64, 4096),
                        rank=rng.choice((32, 48, 64, 96, 128)), T=rng.choice((4, 8, 16)),
                        rows=rng.choice((32, 48, 64)), d_in=_log(rng, 100, 784),
                        hidden=rng.choice((70, 96, 128)), layers=rng.choice((2, 3)),
                        classes=rng.choice((10, 17)))
        return dict(op=op, math="f32", n=_log(rng, 32, 512), rank=rng.choice((1, 2, 4, 8, 16)),
                    T=rng.randint(4, 20), rows=rng.choice((16, 25, 64)), d_in=_log(rng, 100, 784),
                    hidden=rng.choice((64, 100, 128, 200)), layers=rng.choice((2, 3)), classes=10)
    if op == "attention_step":
        return dict(op=op, n=_log(rng, 64, 1024), rank=rng.choice((1, 2, 4, 8)),
                    T=rng.choice((4, 8)), ntok=rng.choice((17, 32, 64)),
                    d_model=rng.choice((32, 64)), heads=rng.choice((2, 4)), blocks=rng.choice((1, 2)))
    if op == "lm":
        if rng.random() < 0.5:
            return dict(op=op, math=rng.choice(("bf16", "f32")), n=_log(rng, 1, 64),
                        rank=rng.choice((1, 2)), T=rng.choice((1, 1, 3)), layers=rng.choice((2, 4)),
                        d_model=rng.choice((256, 512)), state=True)
        return dict(op=op, math="bf16", n=_log(rng, 32, 1024), rank=rng.choice((1, 2)),
                    T=_log(rng, 16, 128), layers=rng.choice((1, 2, 4)),
                    d_model=rng.choice((256, 512)), state=False)
    if op == "spiking_layer":
        return dict(op=op, math=rng.choice(("f32x", "bf16")), n=_log(rng, 20, 4096),
                    rank=rng.choice((32, 48, 80, 128)), T=rng.choice((8, 16)), rows=rng.choice((32, 64)),
                    b=rng.randint(128, 784), a=rng.choice((64, 100, 128)))
    if op == "linear":
        mm = rng.choice(("f32", "f32", "bf16"))
        tmm = rng.random() < 0.25
        lo16 = mm == "bf16"
        n, a = _log(rng, 1, 2048), _log(rng, 10, 2048)
        rows = max(1, min(_log(rng, 1, 256), 131072 // n))
        rank = rng.choice((1, 2, 4, 8, 16))
        # bf16 outputs are offered by the wide-output kernels
        wide = lo16 and rows >= 64 and rank <= 4 and a >= 256
        return dict(op=op, math=mm, n=n, rank=rank, rows=rows, a=a,
                    b=_log(rng, 16, 1024) // 8 * 8 + (0 if lo16 else rng.choice((0, 0, 3))), tmm=tmm,
                    bf16_x=lo16 and rng.random() < 0.7, act=rng.choice(("none", "none", "tanh", "relu_sq")),
                    bf16_y=wide and rng.random() < 0.7)
    if op == "time_mixing":
        return dict(op=op, math=rng.choice(("f32", "bf16")), n=_log(rng, 2, 128), rank=1,
                    T=rng.randint(3, 100), d_model=rng.choice((256, 512)), layer=rng.choice((0, 1)))
    if op == "es_update":
        rank = rng.choice((1, 1, 2, 4, 8, 16, 32, 64, 128))
        return dict(op=op, n=_log(rng, 64, 4096), rank=rank, a=_log(rng, 10, 2048 // max(1, rank // 8)),
                    b=_log(rng, 10, 1024))
    return dict(op=op, T=rng.randint(2, 32), rows=_log(rng, 500, 50000), b=_log(rng, 50, 784),
                h=_log(rng, 10, 256))


# ---- inputs --------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7919 + 17)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32)


def _ints(g, hi, *shape):
    return torch.randint(0, hi, shape, generator=g, device=DEV, dtype=torch.int32)


def _key(i):
    return ((i + 1) * 0x9E3779B97F4A7C15) % 2**64


def _pixels(g, rows, width):
    """Image-like intensities: 70% exact zeros, the rest uniform."""
    p = _rand(g, rows, width)
    p[_rand(g, rows, width) < 0.7] = 0.0
    return p


def _mlp_inputs(case, seed):
    c, g = case, _gen(seed)
    dims = (c["d_in"],) + (c["hidden"],) * c["layers"] + (c["classes"],)
    cfg = snn.SnnConfig(dims=dims, T=c["T"], rows=c["rows"], n=c["n"], rank=c["rank"],
                        math=MATH[c["math"]], lr=1e-4, keys=[_key(i) for i in range(len(dims) - 1)])
    gain = (12.0,) + (18.0, 20.0)[:c["layers"] - 1] + (10.0,)
    W = [(_randn(g, a, b) * (gn / math.sqrt(b))) for a, b, gn in zip(dims[1:], dims[:-1], gain)]
    pool = _pixels(g, 20000, c["d_in"])
    labels = _ints(g, c["classes"], 20000)
    index = _ints(g, 20000, c["n"] * c["rows"])
    return cfg, W, pool, labels, index


def _lm_config(case):
    c = case
    return rwkv_lm.RwkvLmConfig(n_layer=c["layers"], d_model=c["d_model"], seq_len=c["T"], n=c["n"],
                                rank=c["rank"], math=MATH[c["math"]])


def _lm_inputs(case, seed):
    cfg, g = _lm_config(case), _gen(seed)
    C, V, F = cfg.d_model, cfg.vocab, cfg.ffn_mult * cfg.d_model

    def mat(*shape):
        return _randn(g, *shape) / math.sqrt(shape[-1])

    P = {"emb": _randn(g, V, C), "head": mat(V, C), "blocks": [_block(g, cfg) for _ in range(cfg.n_layer)]}
    for n in ("ln0", "ln_out"):
        P[n + "_w"], P[n + "_b"] = 1.0 + 0.1 * _randn(g, C), 0.1 * _randn(g, C)
    for B in P["blocks"]:
        B["ffn_key"], B["ffn_value"] = mat(F, C), mat(C, F)
    tokens = _ints(g, V, case["n"], case["T"])
    state = None
    if case["state"]:
        state = 0.3 * _randn(g, cfg.n_layer, case["n"], 2 + cfg.head_size, C)
    return cfg, P, tokens, state


def _block(g, cfg):
    """One block's TimeMixing and norm parameters."""
    C, (dw, dv, da, dg) = cfg.d_model, cfg.widths
    B = {n: _rand(g, C) for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g", "ffn_x_k")}
    B.update({n: 0.5 * _randn(g, C) for n in ("w0", "v0", "a0", "r_k")})
    B.update({n: 1.0 + 0.1 * _randn(g, C) for n in ("k_k", "k_a", "ln_w", "ln1_w", "ln2_w")})
    B.update({n: 0.1 * _randn(g, C) for n in ("ln_b", "ln1_b", "ln2_b")})
    for n in ("receptance", "key", "value", "output"):
        B[n] = _randn(g, C, C) / math.sqrt(C)
    for n1, n2, d in (("w1", "w2", dw), ("v1", "v2", dv), ("a1", "a2", da), ("g1", "g2", dg)):
        B[n1], B[n2] = _randn(g, C, d) / math.sqrt(C), _randn(g, d, C) / math.sqrt(d)
    return B


def _attention_inputs(case, seed):
    c, g = case, _gen(seed)
    cfg = snn_attention.SaConfig(ntok=c["ntok"], d_model=c["d_model"], heads=c["heads"],
                                 blocks=c["blocks"], T=c["T"], n=c["n"], rank=c["rank"], lr=1e-4)
    P = snn_attention.init_params(cfg, seed)
    vocab = np.random.default_rng(seed + 100).random((cfg.vocab, cfg.tin), dtype=np.float32)
    return cfg, P, vocab, _ints(g, cfg.vocab, c["n"], c["ntok"]), _ints(g, cfg.classes, c["n"])


def _bits(g, rows, T, width, p=0.15):
    """(rows, T, words) bit-packed spikes firing with probability p."""
    words = (width + 63) // 64
    out = torch.empty((rows, T, words), dtype=torch.int64, device=DEV)
    w = 1 << torch.arange(64, device=DEV, dtype=torch.int64)
    for r0 in range(0, rows, 8192):
        r1 = min(rows, r0 + 8192)
        x = _rand(g, r1 - r0, T, words, 64) < p
        x.view(r1 - r0, T, words * 64)[:, :, width:] = False
        out[r0:r1] = (x * w).sum(-1)
    return out


def _spiking_inputs(case, seed):
    c, g = case, _gen(seed)
    M = c["n"] * c["rows"]
    return _bits(g, M, c["T"], c["b"]), _randn(g, c["a"], c["b"]) * (8.0 / math.sqrt(c["b"]))


def _linear_inputs(case, seed):
    c, g = case, _gen(seed)
    b_in = c["b"]
    x = _randn(g, c["n"] * c["rows"], b_in)
    if c["bf16_x"]:
        x = x.to(torch.bfloat16)
    shape = (c["b"], c["a"]) if c["tmm"] else (c["a"], c["b"])
    return x, _randn(g, *shape) / math.sqrt(b_in)


def _tm_inputs(case, seed):
    c, g = case, _gen(seed)
    cfg = rwkv_lm.RwkvLmConfig(n_layer=1, d_model=c["d_model"], seq_len=c["T"], n=c["n"])
    C, S = c["d_model"], cfg.head_size
    return (_block(g, cfg), _randn(g, c["n"], c["T"], C), 0.3 * _randn(g, c["n"], 1 + S, C),
            _randn(g, c["n"], c["T"], C))


def _es_linear(c, i):
    return rwkv.EsLinear(key=_key(i), rank=c["rank"], sigma=0.01, n=c["n"])


def _lif_inputs(case, seed):
    c, g = case, _gen(seed)
    return (_pixels(g, c["rows"], c["b"]), 1.5 * _randn(g, c["T"], c["rows"], c["h"]) + 1.0,
            0.2 * _rand(g, c["rows"], c["h"]))


def prepare(case, seed):
    K.init(0)
    op, s = case["op"], {"case": case}
    if op == "mlp_step":
        cfg, W, pool, labels, index = _mlp_inputs(case, seed)
        s["es"] = snn.SnnEs(cfg, W, pool, labels, index, device=DEV)
        s["epoch"] = 0
    elif op == "attention_step":
        cfg, P, vocab, s["tokens"], s["labels"] = _attention_inputs(case, seed)
        s["es"] = snn_attention.SpikingAttentionEs(cfg, P, vocab, device=DEV)
        s["epoch"] = 0
    elif op == "lm":
        cfg, P, s["tokens"], s["state"] = _lm_inputs(case, seed)
        host = {k: v.cpu().numpy() for k, v in P.items() if k != "blocks"}
        host["blocks"] = [{k: v.cpu().numpy() for k, v in B.items()} for B in P["blocks"]]
        s["lm"] = rwkv_lm.RwkvLmEs(cfg, host, device=DEV)
    elif op == "spiking_layer":
        c = case
        s["x"], s["W"] = _spiking_inputs(case, seed)
        s["rec"] = K.factor_record(c["a"], c["b"], c["rank"], 0, c["n"])
        M, wa = c["n"] * c["rows"], K.fmt_width(K.FMT_BITS, c["a"])
        s["spikes"] = torch.empty((M, c["T"], wa), dtype=torch.int64, device=DEV)
        s["wm"] = K.member_weights(s["W"], c["rank"], 0.02, 0, c["n"], s["rec"].zero_(),
                                   math=MATH[c["math"]])
    elif op == "linear":
        s["x"], s["W"] = _linear_inputs(case, seed)
    elif op == "time_mixing":
        s["P"], s["x"], s["state"], s["v_first"] = _tm_inputs(case, seed)
        s["es"] = {n: _es_linear(case, i) for i, n in enumerate(rwkv_lm.TM_MATRICES)}
    elif op == "es_update":
        s["fit"] = _randn(_gen(seed), case["n"])
        s["out"] = torch.empty((case["a"], case["b"]), dtype=torch.float32, device=DEV)
        s["key"] = _key(seed)
    else:
        s["p"], s["cur"], s["v0"] = _lif_inputs(case, seed)
        s["seeds"] = (seed, 2, 3, 4)
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "mlp_step":
        es = s["es"]
        raw = es.step(s["epoch"])
        s["epoch"] += 1
        return {"raw": raw, "logits": es.logits, "grads": es.grads}
    if op == "attention_step":
        es = s["es"]
        raw = es.step(s["tokens"], s["labels"], s["epoch"])
        s["epoch"] += 1
        return {"raw": raw, "logits": es.logits, "grads": [es.grads[k] for k, _, _ in es.leaves]}
    if op == "lm":
        if s["state"] is None:
            return s["lm"].logits(s["tokens"])
        return s["lm"].logits(s["tokens"], state=s["state"])
    if op == "spiking_layer":
        K.pair_factors(_key(0), c["rank"], 0.02, 0, 0, 0, c["n"], c["a"], c["b"], s["rec"], None)
        wm = K.member_weights(s["W"], c["rank"], 0.02, 0, c["n"], s["rec"], math=MATH[c["math"]],
                              out=s["wm"])
        K.perturbed_linear_lif_mw(s["x"], wm, c["a"], c["b"], 0, c["n"], c["rows"], c["T"], 10.0, 1.0,
                                  math=MATH[c["math"]], spikes=s["spikes"], time_inner=True)
        return s["spikes"]
    if op == "linear":
        f = K.perturbed_linear_t if c["tmm"] else K.perturbed_linear
        return f(s["x"], s["W"], _key(0), c["rank"], 0.02, 0, 0, 0, c["n"], c["rows"],
                 x_fmt=K.FMT_BF16 if c["bf16_x"] else K.FMT_F32, math=MATH[c["math"]],
                 act=ACTS[c["act"]], out_bf16=c["bf16_y"])
    if op == "time_mixing":
        out, state, v_first = rwkv.time_mixing(s["P"], s["x"], s["state"], s["v_first"],
                                               c["d_model"] // 64, c["T"], c["layer"], es=s["es"],
                                               math=MATH[c["math"]])
        return {"out": out, "state": state, "v_first": v_first}
    if op == "es_update":
        return K.es_update(s["fit"], 0, s["key"], c["rank"], 0.02, 0, 0, c["a"], c["b"],
                           np.float32(-1.0 / math.sqrt(c["n"])), out=s["out"])
    spikes = K.poisson_encode(s["p"], c["T"], s["seeds"], K.FMT_BITS)
    out, v = K.lif_scan(s["cur"], 10.0, 1.0, v0=s["v0"], fmt=K.FMT_BITS, want_v=True)
    return {"spikes": spikes, "lif": out, "v": v}


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case):
    c, op = case, case["op"]
    if op == "mlp_step":
        dims = (c["d_in"],) + (c["hidden"],) * c["layers"] + (c["classes"],)
        M = c["n"] * c["rows"]
        flops = byts = 0
        for l, (b, a) in enumerate(zip(dims[:-1], dims[1:])):
            rows = M * (c["T"] if l < len(dims) - 2 else 1)
            # the cheaper of the factored product and the product on every member's weights
            flops += 2 * min(rows * (a * b + c["rank"] * (a + b)),
                             rows * a * b + c["n"] // 2 * a * b * c["rank"])
            flops += c["n"] * a * b * c["rank"]        # the gradient, one term per pair
            byts += 3 * 4 * a * b
        return {"bytes": byts + M * (4 * c["d_in"] + 8 + 4 * c["classes"]), "flops": flops}
    if op == "attention_step":
        cfg = snn_attention.SaConfig(ntok=c["ntok"], d_model=c["d_model"], heads=c["heads"],
                                     blocks=c["blocks"], T=c["T"], n=c["n"], rank=c["rank"])
        leaves = [a * b for _, (a, b), _ in snn_attention.leaf_names(cfg)]
        return {"bytes": 3 * 4 * sum(leaves) + c["n"] * 4 * (c["ntok"] + cfg.classes + 2),
                "flops": snn_attention.forward_flops(cfg) + c["n"] * c["rank"] * sum(leaves)}
    if op == "lm":
        cfg = _lm_config(c)
        weights = 4 * sum(int(np.prod(s)) for s in _lm_shapes(cfg))
        rows = c["n"] * c["T"]
        state = 2 * 4 * c["layers"] * c["n"] * (2 + cfg.head_size) * c["d_model"] if c["state"] else 0
        wkv = rows * c["layers"] * 8 * cfg.head_size * c["d_model"]
        return {"bytes": weights + rows * 4 * (1 + cfg.vocab) + state,
                "flops": rwkv_lm.forward_flops(cfg, c["n"]) + wkv}
    if op == "spiking_layer":
        M = c["n"] * c["rows"] * c["T"]
        return {"bytes": 8 * M * ((c["b"] + 63) // 64 + (c["a"] + 63) // 64) + 4 * c["a"] * c["b"],
                "flops": 2 * M * c["a"] * c["b"] + c["n"] * c["a"] * c["b"] * c["rank"]}
    if op == "linear":
        M = c["n"] * c["rows"]
        return {"bytes": M * (c["b"] * (2 if c["bf16_x"] else 4) + c["a"] * (2 if c["bf16_y"] else 4))
                + 4 * c["a"] * c["b"],
                "flops": 2 * M * (c["a"] * c["b"] + c["rank"] * (c["a"] + c["b"]))}
    if op == "time_mixing":
        cfg = rwkv_lm.RwkvLmConfig(n_layer=1, d_model=c["d_model"])
        C, M = c["d_model"], c["n"] * c["T"]
        low = sum(cfg.widths)
        return {"bytes": 4 * (4 * C * C + 2 * low * C + 3 * M * C + 2 * c["n"] * 65 * C),
                "flops": M * (2 * (4 * C * C + 2 * low * C) + 8 * 64 * C)}
    if op == "es_update":
        return {"bytes": 4 * (c["n"] + c["a"] * c["b"]), "flops": c["n"] * c["a"] * c["b"] * c["rank"]}
    wb, wh = (c["b"] + 63) // 64, (c["h"] + 63) // 64
    return {"bytes": c["rows"] * (4 * c["b"] + 8 * c["T"] * (wb + wh) + 4 * c["h"] * (c["T"] + 2)),
            "flops": c["rows"] * c["T"] * (8 * c["b"] + 4 * c["h"])}


def _lm_shapes(cfg):
    C, F, V = cfg.d_model, cfg.ffn_mult * cfg.d_model, cfg.vocab
    per = [(C, C)] * 4 + [(C, F)] * 2 + [(C, d) for d in cfg.widths for _ in (0, 1)] + [(C,)] * 19
    return per * cfg.n_layer + [(V, C), (V, C)] + [(C,)] * 4


def tolerance(case):
    op = case["op"]
    if op == "encode_lif":
        return {"rel": 1e-6, "max": 1e-4, "differ": 0.0}
    if op == "spiking_layer":
        # a current within rounding of the threshold may fire or not (64 neurons per word)
        return {"rel": 0.0, "differ": 1e-4}
    if op == "mlp_step":
        # a spike at the threshold moves its row's logits by about a fifth: a few rows of all
        # (8192 x 64 rows: 1.1e-3 .. 2.3e-3 off float64; 256 x 64: 1e-5 .. 4.9e-3)
        return {"rel": max(8e-3, min(0.03, 2.5 / math.sqrt(case["n"] * case["rows"]))), "max": 0.99}
    if op == "attention_step":
        # the same with a member's logits (1024 members: 8e-5 .. 1.1e-3 off float64)
        return {"rel": max(5e-3, 0.15 / math.sqrt(case["n"])), "max": 0.99}
    if op == "es_update":
        return {"rel": 2e-6, "max": 4e-5}              # 2e-7 .. 3e-7 off float64
    if op == "linear":                                 # 5e-7 (fp32) and 2.5e-3 (bf16) off float64
        return {"rel": 2e-6, "max": 4e-5} if case["math"] == "f32" else {"rel": 1e-2, "max": 0.2}
    if case["math"] == "f32":                          # 6e-7 off float64
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 2e-2, "max": 0.4}                   # 5e-3 .. 1e-2 off float64


# ---- float64 ------------------------------------------------------------------------------------

_M57, _M64 = (1 << 57) - 1, 2**64 - 1


def _seed(key, thread):
    """The stream seed of (key, epoch 0, pair)."""
    h = ((key ^ 0x9E3779B97F4A7C15) * 0xBF58476D1CE4E5B9) & _M64
    h = (((h << 17) | (h >> 47)) & _M64) ^ thread
    h ^= h >> 33
    h = (h * 0xBF58476D1CE4E5B9) & _M64
    h ^= h >> 29
    h = (h * 0x94D049BB133111EB) & _M64
    return h ^ (h >> 32)


def _apply(tables, x):
    out = tables[0][x & 255]
    for j in range(1, 8):
        out = out ^ tables[j][(x >> (8 * j)) & 255]
    return out


def _tables(cols):
    """Byte tables of a GF(2) map given by its images of the 64 unit vectors."""
    t = torch.zeros((8, 256), dtype=torch.int64, device=DEV)
    for j in range(8):
        for b in range(8):
            t[j, 1 << b:2 << b] = t[j, :1 << b] ^ cols[8 * j + b]
    return t


def _normals(key, pairs, count):
    """(pairs, count) standard normals of every pair's xorshift64 stream: the stream is linear
    over GF(2), so its states are formed by doubling."""
    unit = torch.tensor([(1 << i) - (2**64 if i == 63 else 0) for i in range(64)], dtype=torch.int64,
                        device=DEV)

    def step(x):
        x = x ^ (x << 13)
        x = x ^ ((x >> 7) & _M57)
        return x ^ (x << 17)

    s = [_seed(key, p) | 1 for p in range(pairs)]
    s = torch.tensor([v - 2**64 if v >= 2**63 else v for v in s], dtype=torch.int64, device=DEV)
    states = torch.empty((pairs, 2 * count), dtype=torch.int64, device=DEV)
    states[:, 0] = step(s)
    cols, have = step(unit), 1
    while have < 2 * count:
        t = _tables(cols)
        m = min(have, 2 * count - have)
        states[:, have:have + m] = _apply(t, states[:, :m])
        cols, have = _apply(t, cols), have + m
    k = ((states >> 40) & 0xFFFFFF).double() / 16777216.0
    u1 = k[:, 0::2].clamp_min(float(np.float32(1e-9)))
    radius = torch.sqrt((-2.0 * torch.log(u1).float()).double()).float()
    theta = (float(np.float32(2 * math.pi)) * k[:, 1::2]).float().double()
    return (radius * torch.cos(theta).float()).double()


def _factors(key, rank, sigma, n, a, b):
    """A (n, a, r) with sign and scale, B (n, b, r) of members 0..n-1."""
    bs = float(np.float32(sigma) / np.sqrt(np.float32(rank)))
    z = _normals(key, (n + 1) // 2, (a + b) * rank).view(-1, a + b, rank)
    pair = torch.arange(n, device=DEV) // 2
    sign = (1.0 - 2.0 * (torch.arange(n, device=DEV) % 2)).double().view(-1, 1, 1)
    return z[pair, b:] * (bs * sign), z[pair, :b]


def _mm(x, W, f=None, tmm=False):
    """x (n, R, in) -> x W^T + (x B) A^T, or x W + (x A) B^T."""
    y = x @ (W if tmm else W.t())
    if f is None:
        return y
    A, B = f
    return y + (x @ A) @ B.transpose(1, 2) if tmm else y + (x @ B) @ A.transpose(1, 2)


def _grad(fit, key, rank, sigma, a, b, scale):
    """scale * sum_m fit_m A_m B_m^T, by pairs."""
    bs = float(np.float32(sigma) / np.sqrt(np.float32(rank)))
    n = fit.numel()
    w = torch.zeros(n + n % 2, dtype=torch.float64, device=DEV)
    w[:n] = fit
    w = w[0::2] - w[1::2]
    g = torch.zeros((a, b), dtype=torch.float64, device=DEV)
    z = _normals(key, w.numel(), (a + b) * rank).view(-1, a + b, rank)
    for p0 in range(0, w.numel(), 256):
        zz = z[p0:p0 + 256]
        A = (zz[:, b:] * w[p0:p0 + 256].view(-1, 1, 1)).permute(1, 0, 2).reshape(a, -1)
        g += A @ zz[:, :b].permute(1, 0, 2).reshape(b, -1).t()
    return g * (scale * bs)


def _poisson(p, T, mix, row0, width):
    """(T, rows, width) spikes of the per-element xorshift32 streams of rows row0.."""
    rows = p.shape[0]
    idx = (torch.arange(rows * width, device=DEV, dtype=torch.int64) + row0 * width) & 0xFFFFFFFF
    x = (1000000007 * idx + mix + 0x9E3779B9) & 0xFFFFFFFF
    out = []
    for _ in range(T):
        x = x ^ ((x << 13) & 0xFFFFFFFF)
        x = x ^ (x >> 17)
        x = x ^ ((x << 5) & 0xFFFFFFFF)
        u = (((x >> 9) + 1).double() / 8388609.0).float()
        out.append((u.view(rows, width) < p).double())
    return torch.stack(out)


def _lif(cur, tau, vth, v=None):
    """LIF over the leading time axis: (spikes, last potential)."""
    leak = float(np.float32(1.0 / np.float32(tau)))
    v = torch.zeros_like(cur[0]) if v is None else v
    spikes = []
    for c in cur:
        v = v + (c - v) * leak
        s = (v >= vth).double()
        v = v * (1.0 - s)
        spikes.append(s)
    return torch.stack(spikes), v


def _loglik(logits, labels):
    return torch.log_softmax(logits, -1).gather(-1, labels.long().unsqueeze(-1)).squeeze(-1)


def _zscore(raw):
    return (raw - raw.mean()) / torch.sqrt((raw * raw).mean() - raw.mean() ** 2 + 1e-5)


def _exact_mlp(case, seed):
    cfg, W, pool, labels, index = _mlp_inputs(case, seed)
    c, L = case, len(cfg.dims) - 1
    W = [w.double() for w in W]
    logits = []
    step = max(2, (1 << 27) // (c["rows"] * c["T"] * c["d_in"]) // 2 * 2)
    fac = [_normals(cfg.keys[l], (c["n"] + 1) // 2, (cfg.dims[l] + cfg.dims[l + 1]) * c["rank"]).float()
           for l in range(L)]
    bs = float(np.float32(cfg.sigma) / np.sqrt(np.float32(c["rank"])))
    for m0 in range(0, c["n"], step):
        m1 = min(c["n"], m0 + step)
        m = torch.arange(m0, m1, device=DEV)
        sign = (1.0 - 2.0 * (m % 2)).double().view(-1, 1, 1)
        p = pool[index[m0 * c["rows"]:m1 * c["rows"]].long()]
        x = _poisson(p, c["T"], 0, m0 * c["rows"], c["d_in"])
        for l in range(L):
            a, b = cfg.dims[l + 1], cfg.dims[l]
            z = fac[l][m // 2].double().view(m1 - m0, a + b, c["rank"])
            Wm = W[l] + bs * sign * (z[:, b:] @ z[:, :b].transpose(1, 2))
            if l == L - 1:
                x = x.mean(0, keepdim=True)
            t = x.shape[0]
            xm = x.view(t, m1 - m0, c["rows"], b).transpose(0, 1).reshape(m1 - m0, -1, b)
            cur = (xm @ Wm.transpose(1, 2)).view(m1 - m0, t, c["rows"], a).transpose(0, 1)
            cur = cur.reshape(t, -1, a)
            x = cur if l == L - 1 else _lif(cur, cfg.tau_m, cfg.v_th)[0]
        logits.append(x[0])
    logits = torch.cat(logits)
    raw = _loglik(logits, labels[index.long()]).view(c["n"], -1).mean(1)
    z, scale = _zscore(raw), -1.0 / math.sqrt(c["n"])
    del fac
    grads = [_grad(z, cfg.keys[l], c["rank"], cfg.sigma, cfg.dims[l + 1], cfg.dims[l], scale)
             for l in range(L)]
    return {"raw": raw, "logits": logits, "grads": grads}


def _softplus(x):
    return torch.nn.functional.softplus(x, threshold=100.0)


def _exact_attention(case, seed):
    cfg, P, vocab, tokens, labels = _attention_inputs(case, seed)
    c, n, R, d, hd = case, case["n"], case["ntok"], case["d_model"], case["d_model"] // case["heads"]
    names, keys = snn_attention.leaf_names(cfg), snn_attention.leaf_keys(cfg)
    W = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV).double() for k, v in P.items()}
    sign = (1.0 - 2.0 * (torch.arange(n, device=DEV) % 2)).double()
    pair = torch.arange(n, device=DEV) // 2
    noise = {k: _normals(keys[k], (n + 1) // 2, a * b)[pair] * sign.view(-1, 1) * float(np.float32(cfg.sigma))
             for k, (a, b), cls in names if cls == snn_attention.PARAM}
    leaf = {k: W[k].reshape(1, -1) + v for k, v in noise.items()}

    def mm(x, k):
        a, b = W[k].shape
        return _mm(x, W[k], _factors(keys[k], c["rank"], cfg.sigma, n, a, b))

    p = torch.from_numpy(vocab).to(DEV)[tokens.view(-1).long()]
    s0, s1, s2, s3 = cfg.poisson_seed
    spk = _poisson(p, c["T"], s0 ^ s1 ^ s2 ^ s3, 0, cfg.tin).view(c["T"], n, R, cfg.tin)
    xin = spk.permute(1, 0, 2, 3).reshape(n, c["T"] * R, cfg.tin)
    X = 0.0
    for k in "qkv":
        cur = mm(xin, "in_" + k).view(n, c["T"], R, d).transpose(0, 1)
        X = X + _lif(cur, cfg.tau_m, _softplus(leaf[k + "_th"]).view(n, 1, 1))[0].mean(0)
    X = X / 3.0 + leaf["pos_emb"].view(n, R, d)
    beta, ath = (_softplus(leaf[k]).view(n, 1, 1) for k in ("beta", "attn_th"))
    leak = float(np.float32(1.0 / np.float32(cfg.tau_m)))
    for b in range(c["blocks"]):
        heads = []
        for h in range(c["heads"]):
            q, k, v = (mm(X, "b%d_%s%d" % (b, w, h)) for w in "qkv")
            s = beta * (q @ k.transpose(1, 2))
            s = s / (s.abs().amax(-1, keepdim=True) + 1e-6)
            u, cnt = torch.zeros_like(s), torch.zeros_like(s)
            for _ in range(cfg.n_iter):
                u = u + leak * (s - cfg.g_inh * cnt.sum(-1, keepdim=True) - u)
                f = (u >= ath).double()
                u = u * (1.0 - f)
                cnt = cnt + f
            heads.append((cnt / (cnt.sum(-1, keepdim=True) + 1e-6)) @ v)
        X = X + mm(torch.cat(heads, -1), "b%d_o" % b)
        D = mm(X, "b%d_ff1" % b)
        D = D / D.abs().amax(-1, keepdim=True).clamp_min(1e-6)
        X = X + mm((D >= _softplus(leaf["b%d_ff_th" % b]).view(n, 1, 1)).double(), "b%d_ff2" % b)
    logits = mm(X.mean(1, keepdim=True), "out").view(n, -1) * leaf["out_gain"]
    raw = _loglik(logits, labels)
    z, scale, grads = _zscore(raw), -1.0 / math.sqrt(n), []
    for k, (a, b), cls in names:
        if cls == snn_attention.PARAM:
            grads.append(((noise[k] * z.view(-1, 1)).sum(0) * scale).view(a, b))
        else:
            grads.append(_grad(z, keys[k], c["rank"], cfg.sigma, a, b, scale))
    return {"raw": raw, "logits": logits, "grads": grads}


def _norm(x, w, b, eps):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt((x * x).mean(-1, keepdim=True) - m * m + eps) * w + b


def _shift(x, prev, mix):
    return x + (torch.cat([prev.unsqueeze(1), x[:, :-1]], 1) - x) * mix


def _time_mixing(P, x, state, v_first, layer, mm):
    """x (n, T, C), state (n, 1 + S, C); mm(x, name, tmm) the member's product."""
    n, T, C = x.shape
    S, H = 64, C // 64
    mix = {k: _shift(x, state[:, 0], P["x_" + k]) for k in "rwkvag"}
    r, k, v = mm(mix["r"], "receptance"), mm(mix["k"], "key"), mm(mix["v"], "value")
    w = -_softplus(-(P["w0"] + mm(torch.tanh(mm(mix["w"], "w1", True)), "w2", True))) - 0.5
    a = torch.sigmoid(P["a0"] + mm(torch.tanh(mm(mix["a"], "a1", True)), "a2", True))
    g = mm(torch.sigmoid(mm(mix["g"], "g1", True)), "g2", True)
    if layer == 0:
        v_first = v
    else:
        v = v + (v_first - v) * torch.sigmoid(P["v0"] + mm(torch.tanh(mm(mix["v"], "v1", True)), "v2", True))
    kk = (k * P["k_k"]).view(n, T, H, S)
    kk = kk / kk.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    k = k * (P["k_a"] * (a - 1.0) + 1.0)
    r4, w4, k4, v4, a4 = (t.view(n, T, H, S) for t in (r, torch.exp(-torch.exp(w)), k, v, a))
    s, out = state[:, 1:].reshape(n, H, S, S).clone(), []
    for t in range(T):
        sa = s @ (-kk[:, t]).unsqueeze(-1)
        s = s * w4[:, t].unsqueeze(-2)
        s += v4[:, t].unsqueeze(-1) * k4[:, t].unsqueeze(-2)
        s += sa * (kk[:, t] * a4[:, t]).unsqueeze(-2)
        out.append((s @ r4[:, t].unsqueeze(-1)).squeeze(-1))
    o = torch.stack(out, 1)
    o = _norm(o, P["ln_w"].view(H, S), P["ln_b"].view(H, S), 64e-5)
    o = o + (r4 * k4 * P["r_k"].view(H, S)).sum(-1, keepdim=True) * v4
    state = torch.cat([x[:, -1:], s.reshape(n, S, C)], 1)
    return mm(o.reshape(n, T, C) * g, "output"), state, v_first


def _exact_lm(case, seed):
    cfg, P, tokens, state = _lm_inputs(case, seed)
    c, n = case, case["n"]
    D = {k: v.double() for k, v in P.items() if k != "blocks"}
    blocks = [{k: v.double() for k, v in B.items()} for B in P["blocks"]]
    keys = {ln: _key(i) for i, ln in enumerate(rwkv_lm.mm_names(cfg.n_layer))}
    st = torch.zeros((cfg.n_layer, n, 66, cfg.d_model), dtype=torch.float64, device=DEV) \
        if state is None else state.double()
    x = _norm(D["emb"][tokens.long()], D["ln0_w"], D["ln0_b"], 1e-5)
    vf, new = None, []
    for l, B in enumerate(blocks):
        def mm(t, name, tmm=False):
            W = B[name]
            return _mm(t, W, _factors(keys[(l, name)], c["rank"], cfg.sigma, n, *W.shape), tmm)
        h = _norm(x, B["ln1_w"], B["ln1_b"], 1e-5)
        d, tm, vf = _time_mixing(B, h, st[l, :, 1:], vf, l, mm)
        x = x + d
        h = _norm(x, B["ln2_w"], B["ln2_b"], 1e-5)
        kk = torch.relu(mm(_shift(h, st[l, :, 0], B["ffn_x_k"]), "ffn_key")) ** 2
        x = x + mm(kk, "ffn_value")
        new.append(torch.cat([h[:, -1:], tm], 1))
    lg = (_norm(x, D["ln_out_w"], D["ln_out_b"], 1e-5) @ D["head"].t()).view(-1, cfg.vocab)
    return lg if state is None else (lg, torch.stack(new))


def _exact_linear(case, seed):
    c = case
    x, W = _linear_inputs(case, seed)
    f = _factors(_key(0), c["rank"], 0.02, c["n"], *W.shape)
    y = _mm(x.double().view(c["n"], c["rows"], -1), W.double(), f, c["tmm"]).reshape(-1, c["a"])
    if c["act"] == "tanh":
        y = torch.tanh(y)
    elif c["act"] == "sigmoid":
        y = torch.sigmoid(y)
    elif c["act"] == "relu_sq":
        y = torch.relu(y) ** 2
    return y


def _exact_tm(case, seed):
    P, x, state, v_first = _tm_inputs(case, seed)
    P = {k: v.double() for k, v in P.items()}
    keys = {n: _key(i) for i, n in enumerate(rwkv_lm.TM_MATRICES)}

    def mm(t, name, tmm=False):
        W = P[name]
        return _mm(t, W, _factors(keys[name], case["rank"], 0.01, case["n"], *W.shape), tmm)

    out, st, vf = _time_mixing(P, x.double(), state.double(), v_first.double(), case["layer"], mm)
    return {"out": out, "state": st, "v_first": vf}


def exact(case, seed):
    op = case["op"]
    if op == "mlp_step":
        return _exact_mlp(case, seed)
    if op == "attention_step":
        return _exact_attention(case, seed)
    if op == "lm":
        return _exact_lm(case, seed)
    if op == "spiking_layer":
        return None  # spikes: whole numbers
    if op == "linear":
        return _exact_linear(case, seed)
    if op == "time_mixing":
        return _exact_tm(case, seed)
    if op == "es_update":
        fit = _randn(_gen(seed), case["n"]).double()
        return _grad(fit, _key(seed), case["rank"], 0.02, case["a"], case["b"],
                     float(np.float32(-1.0 / math.sqrt(case["n"]))))
    _, cur, v0 = _lif_inputs(case, seed)
    return {"spikes": None, "lif": None, "v": _lif(cur.double(), 10.0, 1.0, v0.double())[1]}
