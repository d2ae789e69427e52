"""The work that users of this framework give it, as cases that can be timed one by one.

A case is a dict of plain values.  ``listed()`` names the ones that are always run, ``draw(rng)``
makes further ones over the same ranges, ``prepare`` makes what a program holds before the call
(the model or the layers, and the inputs), ``run`` is one pass through the public entry points.

The paths:

  encode     QuantBert: token ids in, hidden states out (``infer`` on numpy arrays, or device
             pointers in and out as a serving process uses the model)
  translate  QuantTransformer: encoder, then beam search until every beam has ended or the
             length limit is reached
  generate   QuantGpt with a sampling model file: prompt pass, then one token a step
  score      QuantGpt with a perplexity model file: one pass over whole texts
  layer      LSTransformerEncoderLayer stacks on torch tensors
  decoder    LSTransformerDecoderLayer stacks over whole target sequences (teacher forcing)
  step       the same stacks, one incremental decoding step over their caches

The shapes are those of ``lightseq_amd.synthetic`` (BERT-base, Transformer-big, GPT-2-medium) and
of ``bench.py``.  Checkpoints cannot be downloaded, so model files are random-init ones; a few
distinct layers take turns in a stack, which keeps making the files short.
"""
import collections
import os
import tempfile

import numpy as np
import torch

from lightseq_amd import inference, layers, proto, synthetic

DEV = "cuda:0"
BERT_MAX_BATCH, BIG_MAX_BATCH = 32, 16
MOST_BERT_TOKENS = 32 * 384


def listed():
    return [
        # one short query at a time: an interactive classifier or retriever
        dict(name="encode b1 s16", path="encode", batch=1, seq=16, io="host"),
        # a small dynamic batch of sentences of any length
        dict(name="encode b7 s75", path="encode", batch=7, seq=75, io="host"),
        # the headline configuration: BERT-base, batch 32, up to 128 tokens, ids on the GPU
        dict(name="encode b32 s128", path="encode", batch=32, seq=128, io="device"),
        # passages and documents, embedded in bulk
        dict(name="encode b32 s384", path="encode", batch=32, seq=384, io="host"),
        # one sentence to translate, as typed
        dict(name="translate b1 s21", path="translate", batch=1, src=21),
        # the headline configuration: Transformer-big, 16 sentences of 64 tokens, beam 4
        dict(name="translate b16 s64", path="translate", batch=16, src=64),
        # one chat turn: a short prompt, the model file's default sampling (top 4)
        dict(name="generate b1 p45 topk4", path="generate", batch=1, prompt=45, method="topk4"),
        # the headline configuration: GPT-2-medium, 16 prompts of 512 tokens, greedy
        dict(name="generate b16 p512 greedy", path="generate", batch=16, prompt=512, method="greedy"),
        # ranking texts by perplexity, right padded to the longest
        dict(name="score b8 s384", path="score", batch=8, seq=384),
        # a Transformer-base layer inside a PyTorch model (the single-layer configuration)
        dict(name="layer base b8 s64", path="layer", batch=8, seq=64, hidden=512, inner=2048, heads=8,
             depth=1, pre_ln=False, act="relu"),
        # a decoder stack over whole target sentences: scoring and forced decoding
        dict(name="decoder big b16 t61 s64", path="decoder", batch=16, trg=61, src=64, hidden=1024,
             inner=4096, heads=16, depth=6, pre_ln=True, act="relu"),
        # one step of a PyTorch-side beam search over the same stack
        dict(name="step big b16 x4 at 31", path="step", batch=16, beam=4, at=31, src=64, hidden=1024,
             inner=4096, heads=16, depth=6, pre_ln=True, act="relu"),
    ]


def _log(rng, low, high):
    """A whole number between ``low`` and ``high``, spread evenly over its logarithm."""
    return max(low, min(high, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    path = rng.choice(["encode", "encode", "encode", "translate", "generate", "score", "layer", "layer",
                       "decoder", "step"])
    if path == "encode":
        batch = _log(rng, 1, BERT_MAX_BATCH)
        seq = _log(rng, 8, min(512, MOST_BERT_TOKENS // batch))
        return dict(path=path, batch=batch, seq=seq, io=rng.choice(["host", "host", "device"]))
    if path == "translate":
        return dict(path=path, batch=_log(rng, 1, BIG_MAX_BATCH), src=_log(rng, 6, 64))
    if path == "generate":
        return dict(path=path, batch=_log(rng, 1, BIG_MAX_BATCH), prompt=_log(rng, 8, 512),
                    method=rng.choice(["greedy", "topk4", "topp"]))
    if path == "score":
        return dict(path=path, batch=_log(rng, 1, BIG_MAX_BATCH), seq=_log(rng, 16, 512))
    hidden, inner, heads = rng.choice([(512, 2048, 8), (768, 3072, 12), (1024, 4096, 16)])
    shape = dict(hidden=hidden, inner=inner, heads=heads, depth=rng.choice([1, 6]),
                 pre_ln=rng.random() < 0.5, act=rng.choice(["relu", "gelu"]))
    if path == "layer":
        return dict(path=path, batch=_log(rng, 1, 32), seq=_log(rng, 8, 256), **shape)
    if path == "decoder":
        return dict(path=path, batch=_log(rng, 1, 16), trg=_log(rng, 6, 64), src=_log(rng, 6, 64), **shape)
    return dict(path=path, batch=_log(rng, 1, 16), beam=4, at=_log(rng, 1, 64), src=_log(rng, 6, 64), **shape)


# --------------------------------------------------------------------------------------------
# models and layers: built once for a shape and kept, as a program keeps them
# --------------------------------------------------------------------------------------------
_kept = collections.OrderedDict()
_MOST_KEPT = 16


def _keep(key, make):
    if key in _kept:
        _kept.move_to_end(key)
        return _kept[key]
    while len(_kept) >= _MOST_KEPT:
        _, old = _kept.popitem(last=False)
        if hasattr(old, "close"):
            old.close()
    _kept[key] = make()
    return _kept[key]


def _turns(stack, n):
    return [stack[i % len(stack)] for i in range(n)]


def _load(cls, parts, max_batch):
    """A model from its file, written as encoded pieces one after the other."""
    with tempfile.TemporaryDirectory() as tmp:
        path = os.path.join(tmp, "model.pb")
        with open(path, "wb") as f:
            for p in parts:
                f.write(p)
        return cls(path, max_batch)


def _bert_cfg():
    return synthetic.bert_config("bert_base")


def _bert(io):
    """With device pointers the model is the plain LSModel of the C interface, whose caller owns the
    output memory; the numpy class keeps buffers of its own."""
    def load(path, max_batch):
        if io == "host":
            return inference.QuantBert(path, max_batch)
        return inference.LSModel("QuantBert", path, max_batch)

    def make():
        cfg = _bert_cfg()
        msg = synthetic.make_quant_bert(dict(cfg, n_layer=3), seed=0)
        msg["encoder_stack"] = _turns(msg["encoder_stack"], cfg["n_layer"])
        return _load(load, [proto.encode("QuantBert", msg)], BERT_MAX_BATCH)
    return _keep("bert " + io, make)


def _transformer_cfg():
    return dict(synthetic.transformer_config("transformer_big"), max_step=128)


def _transformer():
    def make():
        cfg = _transformer_cfg()
        distinct = 2
        msg = synthetic.make_quant_transformer(dict(cfg, n_enc_layer=distinct, n_dec_layer=distinct), seed=0)
        emb, times = msg["trg_embedding"], cfg["n_dec_layer"] // distinct
        msg["encoder_stack"] = _turns(msg["encoder_stack"], cfg["n_enc_layer"])
        msg["decoder_stack"] = _turns(msg["decoder_stack"], cfg["n_dec_layer"])
        for name in ("encode_output_project_kernel_kv", "encode_output_project_bias_kv",
                     "encode_output_project_kernel_kv_clip_max"):
            emb[name] = np.tile(emb[name], times)
        return _load(inference.QuantTransformer, [proto.encode("QuantTransformer", msg)], BIG_MAX_BATCH)
    return _keep("transformer", make)


def _gpt_cfg():
    return synthetic.gpt_config("gpt2_medium")


_gpt_body = []


def _gpt(method):
    def make():
        cfg = _gpt_cfg()
        if not _gpt_body:  # everything but the settings is the same for every method
            msg = synthetic.make_quant_gpt(dict(cfg, n_layer=3), seed=0)
            msg["encoder_stack"] = _turns(msg["encoder_stack"], cfg["n_layer"])
            conf = msg.pop("model_conf")
            _gpt_body.extend([proto.encode("QuantGpt", msg), conf])
        body, conf = _gpt_body
        conf = dict(conf, **{"greedy": dict(sampling_method="topk", topk=1),
                             "topk4": dict(sampling_method="topk", topk=4),
                             "topp": dict(sampling_method="topp", topp=0.75),
                             "ppl": dict(sampling_method="ppl")}[method])
        return _load(inference.QuantGpt, [body, proto.encode("QuantGpt", {"model_conf": conf})], BIG_MAX_BATCH)
    return _keep("gpt " + method, make)


def _shape_key(case):
    return tuple(case[k] for k in ("hidden", "inner", "heads", "depth", "pre_ln", "act"))


def _layer_config(cls, case, tokens, length, **more):
    return cls.get_config(max_batch_tokens=tokens, max_seq_len=length, hidden_size=case["hidden"],
                          intermediate_size=case["inner"], nhead=case["heads"], attn_prob_dropout_ratio=0.0,
                          activation_dropout_ratio=0.0, hidden_dropout_ratio=0.0, pre_layer_norm=case["pre_ln"],
                          fp16=True, local_rank=0, activation_fn=case["act"], **more)


def _ready(layer, clips):
    """A layer as a quantised model holds it for inference: half parameters on the GPU, clip values as
    calibrated to what flows through (inputs after a layer norm, small weights)."""
    layer = layer.half().to(DEV).eval()
    layer.enable_quant()
    at = layer.para_offset[clips]
    n = layer.para_offset[clips + 1] - at
    with torch.no_grad():
        layer.para[at:at + n] = torch.tensor([4.0, 0.15, 6.0], dtype=torch.half, device=DEV).repeat(n // 3)
    return layer


def _encoder_stack(case):
    cls = layers.LSTransformerEncoderLayer

    def make():
        torch.manual_seed(0)
        cfg = _layer_config(cls, case, 32 * 256, 256)
        return [_ready(cls(cfg), 12) for _ in range(case["depth"])]
    return _keep(("encoder",) + _shape_key(case), make)


_decoders = {}


def _decoder_stack(case):
    """One decoder stack at a time: its layers are numbered from 0 in a process."""
    cls, key = layers.LSTransformerDecoderLayer, _shape_key(case)
    if key not in _decoders:
        for stack in _decoders.values():
            for layer in stack:
                layer.release()
        _decoders.clear()
        cls.new_stack()
        torch.manual_seed(0)
        cfg = _layer_config(cls, case, 16 * 64, 128, nlayer=case["depth"])
        _decoders[key] = [_ready(cls(cfg), 18) for _ in range(case["depth"])]
    return _decoders[key]


# --------------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------------
def _padded_ids(rng, batch, seq, vocab, pad):
    """Uniform ids, right padded: one sequence of full length, the others from a quarter of it up."""
    ids = rng.integers(1, vocab - 1, size=(batch, seq), dtype=np.int32)
    lens = rng.integers(max(1, seq // 4), seq + 1, size=batch)
    lens[rng.integers(batch)] = seq
    ids[np.arange(seq)[None, :] >= lens[:, None]] = pad
    return ids


def _padding(rng, batch, seq):
    """1 for padding, as the layers take it."""
    lens = rng.integers(max(1, seq // 4), seq + 1, size=batch)
    lens[rng.integers(batch)] = seq
    return torch.from_numpy((np.arange(seq)[None, :] >= lens[:, None]).astype(np.float32)).to(DEV)


def _normal(seed, *shape):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.half)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    path, s = case["path"], dict(case=case)
    if path == "encode":
        cfg, s["model"] = _bert_cfg(), _bert(case["io"])
        s["ids"] = _padded_ids(rng, case["batch"], case["seq"], cfg["vocab"], cfg["padding_id"])
        if case["io"] == "device":
            s["ids"] = torch.from_numpy(s["ids"]).to(DEV)
            s["out"] = torch.zeros(case["batch"], case["seq"], cfg["hidden"], dtype=torch.half, device=DEV)
    elif path == "translate":
        s["model"] = _transformer()
        s["ids"] = rng.integers(4, _transformer_cfg()["src_vocab"], size=(case["batch"], case["src"]), dtype=np.int32)
    elif path == "generate":
        s["model"] = _gpt(case["method"])
        s["ids"] = rng.integers(0, _gpt_cfg()["vocab"] - 1, size=(case["batch"], case["prompt"]), dtype=np.int32)
        s["seed"] = seed
    elif path == "score":
        cfg, s["model"] = _gpt_cfg(), _gpt("ppl")
        s["ids"] = _padded_ids(rng, case["batch"], case["seq"], cfg["vocab"], cfg["padding_id"])
    elif path == "layer":
        s["layers"] = _encoder_stack(case)
        s["x"] = _normal(seed, case["batch"], case["seq"], case["hidden"])
        s["mask"] = _padding(rng, case["batch"], case["seq"])
    else:
        s["layers"] = _decoder_stack(case)
        b, H = case["batch"], case["hidden"]
        s["enc"] = _normal(seed + 1, case["src"], b, H)
        s["mask"] = _padding(rng, b, case["src"])
        if path == "decoder":
            s["x"] = _normal(seed, b, case["trg"], H)
        else:
            rows, h = b * case["beam"], case["heads"]
            s["x"] = _normal(seed, rows, 1, H)
            s["caches"] = []
            for i in range(case["depth"]):
                k, v = _normal(seed + 2 + i, 2, rows, h, case["at"], H // h)
                s["caches"].append({"dec_self_k": k, "dec_self_v": v})
            s["caches"][0]["encdec_kv"] = _normal(seed + 99, case["depth"] * 2, b, case["src"] * H)
    return s


# --------------------------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    path = case["path"]
    if path == "encode":
        model = s["model"]
        if case["io"] == "host":
            return model.infer(s["ids"])
        model.set_input_ptr(0, s["ids"].data_ptr())
        model.set_input_shape(0, s["ids"].shape)
        model.set_output_ptr(0, s["out"].data_ptr())
        model.infer_device()
        return s["out"]
    if path == "translate":
        tokens, scores = s["model"].infer(s["ids"])
        return {"tokens": tokens, "scores": scores}
    if path == "generate":
        if case["method"] != "greedy":
            s["model"].set_seed(s["seed"])  # the stream of random numbers belongs to the request
        return s["model"].sample(s["ids"])
    if path == "score":
        return s["model"].ppl(s["ids"])
    with torch.no_grad():
        x = s["x"]
        if path == "layer":
            for layer in s["layers"]:
                x = layer(x, s["mask"])
            return x
        if path == "decoder":
            for layer in s["layers"]:
                x = layer(x, s["enc"], s["mask"])
            return x
        caches = [dict(c) for c in s["caches"]]  # a step replaces the entries by longer ones
        for layer, cache in zip(s["layers"], caches):
            x = layer(x, s["enc"], s["mask"], cache)
        return {"x": x, "k": [c["dec_self_k"] for c in caches], "v": [c["dec_self_v"] for c in caches]}


# --------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far another correct implementation may be off
# --------------------------------------------------------------------------------------------
def work(case):
    path, B = case["path"], case["batch"]
    if path in ("encode", "translate", "generate", "score"):
        cfg = {"encode": _bert_cfg, "translate": _transformer_cfg}.get(path, _gpt_cfg)()
        H, I = cfg["hidden"], cfg["inner"]
        mat = 4 * H * H + 2 * H * I  # an encoder layer's int8 weights, in bytes and in products a token
        if path == "encode":
            L, seq = cfg["n_layer"], case["seq"]
            tokens = B * seq if B == 1 else seq * (1 + (B - 1) * 0.625)  # of the mean length
            return {"bytes": L * mat + tokens * H + B * seq * (4 + H * (4 if case["io"] == "host" else 2)),
                    "flops": L * tokens * (2 * mat + 4 * seq * H * 0.625)}
        if path == "score":
            L, V, seq = cfg["n_layer"], cfg["vocab"], case["seq"]
            tokens = B * seq if B == 1 else seq * (1 + (B - 1) * 0.625)
            return {"bytes": L * mat + V * H + B * (4 * seq + 4),
                    "flops": tokens * (L * (2 * mat + 2 * seq * H * 0.625) + 2 * V * H)}
        if path == "generate":
            L, V, P, steps = cfg["n_layer"], cfg["vocab"], case["prompt"], cfg["extra_decode_length"]
            cache = L * B * 2 * H * (P + steps / 2)  # int8 keys and values of a step
            return {"bytes": L * mat * steps + steps * (V * H + cache) + B * 4 * (2 * P + steps),
                    "flops": 2 * B * (steps * (L * mat + V * H) + P * L * (mat + P * H)) + 2 * steps * cache}
        Le, Ld, V, S, beam = cfg["n_enc_layer"], cfg["n_dec_layer"], cfg["trg_vocab"], case["src"], cfg["beam_size"]
        steps = min(cfg["max_step"], S + cfg["extra_decode_length"]) - 2  # at most
        dec = 6 * H * H + 2 * H * I
        cache = Ld * (B * beam * H * steps + B * S * H * 4)  # int8 self, fp16 cross keys and values
        return {"bytes": Le * mat + Ld * 4 * H * H + steps * (Ld * dec + V * H + cache),
                "flops": 2 * B * (S * (Le * (mat + 2 * S * H) + Ld * 2 * H * H) + steps * beam * (Ld * dec + V * H))}
    H, I, L = case["hidden"], case["inner"], case["depth"]
    if path == "layer":
        mat, rows = 4 * H * H + 2 * H * I, B * case["seq"]
        return {"bytes": 2 * L * mat + 4 * rows * H, "flops": L * rows * (2 * mat + 4 * case["seq"] * H)}
    mat, S = 6 * H * H + 2 * H * I, case["src"]
    if path == "decoder":
        rows, T = B * case["trg"], case["trg"]
        return {"bytes": 2 * L * (mat + 2 * H * H) + 4 * rows * H + 2 * B * S * H,
                "flops": L * (rows * (2 * mat + 4 * H * (T / 2 + S)) + B * S * 4 * H * H)}
    rows, at = B * case["beam"], case["at"]
    return {"bytes": 2 * L * (mat + 2 * rows * H * (2 * at + 1) + 2 * B * S * H) + 4 * rows * H,
            "flops": L * rows * (2 * mat + 4 * H * (at + S))}


def tolerance(case):
    path = case["path"]
    if path == "encode":
        # int8 codes between the stages: a float on the edge between two codes gives one or the other,
        # and what follows drifts; a twelve-layer stack against a plain C implementation of it is off
        # by 2e-2 in the mean over outputs of about 1
        return {"rel": 0.025, "max": 0.25}
    if path == "score":
        return {"rel": 2e-3}
    if path in ("translate", "generate"):
        return {"rel": 1e-3, "differ": 0.01}  # token ids; ties
    return {"rel": 0.01 if case["depth"] == 1 else 0.02, "max": 0.3}
