"""Workloads of the transformer-encoder path, as programs that use the framework run them.

Most are one request to an `Instance` on DEVICE_ROCM made from model files: the token ids, segment ids, mask and
positions go in as Mats, `Forward`, and the last hidden state comes out as a Mat -- the loop of the engine's benchmark
tool (reference test/test.cc:101-152).  "host" is a program whose requests arrive and leave in host memory, "device" a
serving loop whose tensors stay on the card.  The model is kept from request to request, as such a program keeps it;
only the inputs change.  The other workloads are the single attention layer in fp32, and the fused attention kernel
called by itself through the operator interface.
"""
import functools

import numpy as np
import torch

from tnn_amd import host, ops, quant, tnnmodel
from tnn_amd.encoder import EncoderConfig, make_inputs, make_weights

_ID_INPUTS = ("input_ids", "token_type_ids", "input_mask", "position_ids")
# numpy type of the Mat that a device-side reader asks for: a float blob's own 16-bit form
_DEVICE_MAT = {"fp16": np.float16, "bf16": np.uint16}


def _config(case):
    return (EncoderConfig.bert_large if case["model"] == "large" else EncoderConfig.bert_base)(case["layers"])


def listed():
    def encoder(name, precision, batch, seq, io, model="base", layers=12):
        return {"name": name, "kind": "encoder", "model": model, "layers": layers, "precision": precision,
                "batch": batch, "seq": seq, "io": io}

    return [
        # one short query, answered while somebody waits: launches and host work count
        encoder("query_fp16_b1_s32", "fp16", 1, 32, "host"),
        # the reading-comprehension demo's request: ids [1,256] int32 (reference BertReadingComprehension.cc:43,73)
        encoder("reading_fp16_b1_s256", "fp16", 1, 256, "host"),
        # the headline batch of the benchmark, kept on the card
        encoder("headline_fp16_b8_s384", "fp16", 8, 384, "device"),
        # a batch as it happens to come in: no dimension a multiple of anything, bfloat16 activations
        encoder("ragged_bf16_b5_s197", "bf16", 5, 197, "host"),
        # bulk encoding with the large model, whole batches on the card (24 layers cut to 4: the layers are alike)
        encoder("large_fp16_b16_s512", "fp16", 16, 512, "device", model="large", layers=4),
        # full precision (PRECISION_HIGH), one request and a batch
        encoder("full_fp32_b1_s128", "fp32", 1, 128, "host"),
        encoder("full_fp32_b4_s384", "fp32", 4, 384, "host"),
        # int8 projections with per-channel weights: the throughput configuration and one request
        dict(encoder("int8_b16_s256", "fp16", 16, 256, "device", layers=6), kind="int8"),
        dict(encoder("int8_b1_s128", "fp16", 1, 128, "host", layers=6), kind="int8"),
        # four requests of four lengths, each with an Instance::Reshape to its own shape instead of padding
        dict(encoder("stream_fp16_s200", "fp16", 1, 200, "host"), kind="stream"),
        # a single self-attention layer in fp32: InnerProduct projections around the un-fused core, hidden states in and out
        {"name": "layer_fp32_s128", "kind": "layer", "model": "base", "layers": 1, "precision": "fp32", "batch": 1,
         "seq": 128, "io": "host"},
        # the attention operator alone on padded sequences of very different lengths
        {"name": "attention_fp16_b32_s512", "kind": "attention", "precision": "fp16", "batch": 32, "seq": 512, "heads": 12},
    ]


def _log_int(rng, lo, hi):
    """a whole number between lo and hi, even over the logarithm"""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _shape(rng, max_batch, max_tokens):
    """(batch, seq): lengths of 16 to 512 tokens, half of them as a tokenizer leaves them and half padded to eights"""
    seq = _log_int(rng, 16, min(512, max_tokens))
    if rng.random() < 0.5:
        seq = -(-seq // 8) * 8
    return _log_int(rng, 1, max(1, min(max_batch, max_tokens // seq))), seq


def draw(rng):
    kind = rng.choice(["encoder", "encoder", "encoder", "encoder", "int8", "stream", "layer", "attention"])
    if kind == "attention":
        batch, seq = _shape(rng, 32, 32 * 512)
        return {"kind": kind, "precision": rng.choice(["fp16", "bf16"]), "batch": batch, "seq": seq,
                "heads": rng.choice([12, 16])}
    case = {"kind": kind, "model": "base", "layers": 12, "precision": "fp16", "io": rng.choice(["host", "device"])}
    if kind == "encoder":
        case["precision"] = rng.choice(["fp16", "fp16", "bf16", "fp32"])
        if case["precision"] != "fp32" and rng.random() < 0.25:
            case["model"], case["layers"] = "large", 4
        max_tokens = {"fp32": 1536}.get(case["precision"], 3072)
        case["batch"], case["seq"] = _shape(rng, 32, max_tokens)
        if case["precision"] == "fp32":
            case["io"] = "host"
    elif kind == "int8":
        case["layers"] = 6
        case["batch"], case["seq"] = _shape(rng, 32, 4096)
    elif kind == "stream":
        case.update(io="host", batch=rng.choice([1, 2, 4]), seq=_log_int(rng, 24, 384))
    else:
        case.update(io="host", precision="fp32", layers=1, batch=1, seq=_log_int(rng, 16, 512))
    return case


# ---- what a program loads once ---------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _encoder_files(model, layers):
    """.tnnproto / .tnnmodel of the encoder with a batch and sequence length of the caller's choice"""
    cfg = _config({"model": model, "layers": layers})
    graph = tnnmodel.encoder_graph(cfg, make_weights(cfg, seed=20240601, bias_std=0.02), 1, 128, dynamic=True, int_mask=True,
                                   position_ids=True)
    return graph.proto(), graph.model()


@functools.lru_cache(maxsize=2)
def _int8_parts(model, layers):
    """weights and per-tensor activation scales, from one fp32 forward of the float model over calibration data"""
    cfg = _config({"model": model, "layers": layers})
    weights = make_weights(cfg, seed=20240604, bias_std=0.02)
    names = quant.calibration_outputs(cfg)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, weights, 2, 128, extra_outputs=names), "fp32")
    ids, seg, _, mask = make_inputs(cfg, 2, 128, 128, 128, seed=20240605)
    for name, value in (("input_ids", ids), ("token_type_ids", seg), ("attention_bias", mask.reshape(2, 1, 1, 128))):
        inst.set_input(name, value)
    inst.forward()
    scales = {n: quant.activation_scale(inst.output(n)) for n in names}
    inst.close()
    return weights, scales


@functools.lru_cache(maxsize=24)
def _instance(kind, model, layers, precision, batch, seq):
    case = {"model": model, "layers": layers}
    cfg = _config(case)
    if kind == "layer":
        weights = make_weights(cfg, seed=20240601, bias_std=0.02, with_embeddings=False)["layers"][0]
        graph = tnnmodel.attention_layer_graph(weights, seq, cfg.hidden, cfg.heads)
        return host.RocmInstance.from_graph(graph, precision)
    if kind == "int8":
        weights, scales = _int8_parts(model, layers)
        return host.RocmInstance.from_graph(quant.int8_encoder_graph(cfg, weights, scales, batch, seq), precision)
    proto, weights = _encoder_files(model, layers)
    return host.RocmInstance(proto, weights, precision, input_shapes={n: [batch, seq] for n in _ID_INPUTS})


# ---- one request -----------------------------------------------------------------------------------------------------
def _stream_lengths(seq):
    """sequence lengths of the stream's four requests, the longest first"""
    return [seq, max(1, seq * 5 // 8), max(1, seq // 5), max(1, seq * 3 // 4 + 1)]


def _requests(case, seed):
    """[(batch, seq, {input name: host array})]"""
    cfg, batch = _config(case), case["batch"]
    lengths = _stream_lengths(case["seq"]) if case["kind"] == "stream" else [case["seq"]]
    found = []
    for k, seq in enumerate(lengths):
        # sequences fill at least half of the padded length
        ids, seg, _, bias = make_inputs(cfg, batch, seq, max(1, (seq + 1) // 2), seq, seed=1000 * seed + k)
        feed = {"input_ids": ids, "token_type_ids": seg}
        if case["kind"] == "int8":
            feed["attention_bias"] = bias.reshape(batch, 1, 1, seq)
        else:
            feed["input_mask"] = (bias == 0).astype(np.int32)
            feed["position_ids"] = np.tile(np.arange(seq, dtype=np.int32), (batch, 1))
        found.append((batch, seq, feed))
    return found


def prepare(case, seed):
    if case["kind"] == "attention":
        return _prepare_attention(case, seed)
    inst = _instance(case["kind"], case["model"], case["layers"], case["precision"], case["batch"], case["seq"])
    state = {"case": case, "inst": inst}
    if case["kind"] == "layer":
        rng = np.random.default_rng(seed)
        state["hidden"] = rng.standard_normal((case["seq"], _config(case).hidden)).astype(np.float32)
        return state
    state["requests"] = _requests(case, seed)
    if case["io"] == "device":
        batch, seq, feed = state["requests"][0]
        state["device"] = {n: torch.from_numpy(a).cuda() for n, a in feed.items()}
    return state


def _prepare_attention(case, seed):
    batch, seq, heads = case["batch"], case["seq"], case["heads"]
    dtype = torch.float16 if case["precision"] == "fp16" else torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)

    lens = np.random.default_rng(seed).integers(min(16, seq), seq + 1, batch).astype(np.int32)
    state = {"case": case, "kv_len": torch.from_numpy(lens).cuda(),
             "out": torch.empty(batch * seq, heads * 64, device="cuda", dtype=dtype)}
    if seq % 8:
        state["qkv"] = normal(batch * seq, 3 * heads * 64)
    else:
        state["qk"] = normal(batch * seq, 2 * heads * 64)
        state["vt"] = normal(batch, heads, 64, seq)
    return state


class _DeviceMat:
    """an output Mat in device memory, for torch.as_tensor"""

    def __init__(self, address, shape, typestr):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (address, False), "version": 3}


def run(state):
    case = state["case"]
    if case["kind"] == "attention":
        return _run_attention(state)
    inst = state["inst"]
    if case["kind"] == "layer":
        inst.set_input("x", state["hidden"])
        inst.forward()
        return inst.output("y")
    if case["kind"] == "stream":
        answers = []
        for batch, seq, feed in state["requests"]:
            inst.reshape({n: [batch, seq] for n in feed})
            for name, value in feed.items():
                inst.set_input(name, value)
            inst.forward()
            answers.append(inst.output("last_hidden"))
        return answers
    if case["io"] == "device":
        for name, value in state["device"].items():
            kind = np.float32 if value.dtype == torch.float32 else np.int32
            inst.set_input_device(name, value.data_ptr(), kind, list(value.shape))
        inst.forward()
        address, shape = inst.output_device("last_hidden", _DEVICE_MAT[case["precision"]])
        if case["precision"] == "bf16":
            return torch.as_tensor(_DeviceMat(address, shape, "<i2"), device="cuda").view(torch.bfloat16)
        return torch.as_tensor(_DeviceMat(address, shape, "<f2"), device="cuda")
    for name, value in state["requests"][0][2].items():
        inst.set_input(name, value)
    inst.forward()
    return inst.output("last_hidden")


def _run_attention(state):
    case = state["case"]
    batch, seq, heads = case["batch"], case["seq"], case["heads"]
    if "qkv" in state:
        return ops.attention_packed(state["qkv"], batch, seq, heads, 0.125, kv_len=state["kv_len"], out=state["out"])
    return ops.attention_qk_vt(state["qk"], state["vt"], batch, seq, heads, 0.125, kv_len=state["kv_len"],
                               out=state["out"], vt_key_order=1 if seq % 16 == 0 else 0)


# ---- what a pass cannot do without -------------------------------------------------------------------------------------
def work(case):
    batch, seq = case["batch"], case["seq"]
    if case["kind"] == "attention":
        hidden = 64 * case["heads"]
        keys = (min(16, seq) + seq) / 2  # mean valid length: keys behind it need not be read
        return {"bytes": 2 * hidden * batch * (2 * seq + 2 * keys), "flops": 4 * hidden * batch * seq * keys}
    cfg = _config(case)
    hidden, ffn, layers = cfg.hidden, cfg.ffn, case["layers"]
    if case["kind"] == "layer":
        return {"bytes": 4 * (4 * hidden * hidden + 2 * seq * hidden),
                "flops": 8 * seq * hidden * hidden + 4 * seq * seq * hidden}
    elem = 4 if case["precision"] == "fp32" else 2
    weight_elem = 1 if case["kind"] == "int8" else elem
    answer_elem = 4 if case["io"] == "host" else 2
    found = {"bytes": 0.0, "flops": 0.0}
    for s in _stream_lengths(seq) if case["kind"] == "stream" else [seq]:
        tokens, keys = batch * s, ((s + 1) // 2 + s) / 2
        found["bytes"] += (layers * (4 * hidden * hidden + 2 * hidden * ffn) * weight_elem
                           + tokens * (16 + 3 * hidden * elem + hidden * answer_elem))
        found["flops"] += layers * tokens * (8 * hidden * hidden + 4 * hidden * ffn + 4 * keys * hidden)
    return found


def tolerance(case):
    if case["precision"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] == "attention":
        return {"rel": 1e-2 if case["precision"] == "bf16" else 1e-3}
    if case["kind"] == "int8":
        # a float part that rounds another way moves some int8 activation by one, a 127th of its range, and six layers
        # carry that on: the same graph with half and with fp32 blobs is 2.5e-2 apart
        return {"rel": 2.5e-2}
    # half-precision blobs between the layers: twelve layers end 1.1e-3 (fp16) and 8.4e-3 (bf16) from their fp32 form,
    # and two implementations that far from each other again
    return {"rel": 1.2e-2 if case["precision"] == "bf16" else 2e-3}
