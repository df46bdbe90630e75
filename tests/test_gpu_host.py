"""The C++ host (Instance::Forward on DEVICE_ROCM) fed with the same .tnnproto/.tnnmodel files the reference
engine loads: un-fused fp32 path, fused fp16 path, int8 path, error behaviour."""
import numpy as np
import pytest

import encoder_ref
import orc
from test_gpu_ops import rel_err, say, BF16_TOL, FP16_TOL, FP32_TOL, FP32_ASSERT

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _mods():
    from tnn_amd import host, tnnmodel
    from tnn_amd.encoder import EncoderConfig, make_weights, make_inputs
    return host, tnnmodel, EncoderConfig, make_weights, make_inputs


def r16w(w):
    out = {}
    for k, v in w.items():
        if k == "layers":
            out[k] = [{n: (a.astype(np.float16).astype(np.float32) if a.ndim == 2 else a) for n, a in lw.items()}
                      for lw in v]
        else:
            out[k] = v.astype(np.float16).astype(np.float32) if v.ndim == 2 else v
    return out


def test_config1_attention_layer_fp32_from_model_files():
    host, tnnmodel, EncoderConfig, make_weights, _ = _mods()
    say("host: config-1 attention layer proto, fp32")
    cfg = EncoderConfig(1, 768, 12, 3072)
    lw = make_weights(cfg, seed=1, with_embeddings=False)["layers"][0]
    x = np.random.default_rng(2).standard_normal((128, 768)).astype(np.float32)
    g = tnnmodel.attention_layer_graph(lw, 128, 768, 12)
    inst = host.RocmInstance.from_graph(g, "fp32")
    types = [t for t, _ in inst.layers()]
    say("  layers: " + " ".join(types))
    assert "RocmFusedAttention" not in types          # fp32 keeps the decomposed attention core
    assert types.count("RocmFusedLinear") == 4        # the four InnerProduct projections
    inst.set_input("x", x)
    inst.forward()
    got = inst.output("y")
    ref = encoder_ref.attention_layer(x, lw, 1, 128, 12, None)
    err = rel_err(got, ref)
    say("  max rel err %.3g" % err)
    assert got.shape == (128, 768) and err <= 1e-5 <= FP32_TOL
    inst.close()


def test_view_layers_share_their_input_buffer_and_change_nothing(monkeypatch):
    """Reshape layers that only rename dimensions copy nothing (their output shares the input's buffer in the memory
    plan); with TNN_ROCM_ALIAS_VIEWS=0 every blob has its own buffer and the layer copies.  Same graph, same input:
    bit-identical outputs over several forwards (eager, the recording forward and graph replays)."""
    host, tnnmodel, EncoderConfig, make_weights, _ = _mods()
    say("host: view layers alias their input")
    cfg = EncoderConfig(1, 768, 12, 3072)
    lw = make_weights(cfg, seed=5, with_embeddings=False)["layers"][0]
    g = tnnmodel.attention_layer_graph(lw, 128, 768, 12)
    rng = np.random.default_rng(6)
    xs = [rng.standard_normal((128, 768)).astype(np.float32) for _ in range(5)]
    outs = {}
    for alias in ("1", "0"):
        monkeypatch.setenv("TNN_ROCM_ALIAS_VIEWS", alias)
        inst = host.RocmInstance.from_graph(g, "fp32")
        assert [t for t, _ in inst.layers()].count("Reshape") >= 4
        res = []
        for x in xs:
            inst.set_input("x", x)
            inst.forward()
            res.append(inst.output("y").copy())
        outs[alias] = res
        inst.close()
    for a, b in zip(outs["1"], outs["0"]):
        assert np.array_equal(a, b)
    ref = encoder_ref.attention_layer(xs[-1], lw, 1, 128, 12, None)
    assert rel_err(outs["1"][-1], ref) <= 1e-5


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_encoder_from_model_files(precision):
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: 2-layer encoder proto with embeddings + mask, " + precision)
    cfg = EncoderConfig.bert_base(2)
    w = make_weights(cfg, seed=3, bias_std=0.02)
    B, S = 2, 96
    ids, seg, lens, mask = make_inputs(cfg, B, S, 30, 96, seed=4)
    g = tnnmodel.encoder_graph(cfg, w, B, S)
    inst = host.RocmInstance.from_graph(g, precision)
    types = [t for t, _ in inst.layers()]
    if precision == "fp16":
        # per encoder layer: attention, out-proj(+res), ffn1(+gelu), ffn2(+res); the LayerNorms are folded into the
        # projection that reads them (ffn1, the next layer's QKV); only the last one, a model output, stays a layer
        assert types.count("RocmFusedAttention") == 2 and types.count("RocmFusedLinear") == 6
        assert types.count("LayerNorm") == 1, types
        assert not any(t in ("Softmax", "Permute", "Reshape", "MatMul", "GELU") for t in types), types
    else:
        assert types.count("RocmFusedLinear") == 12 and types.count("Softmax") == 2
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    inst.forward()
    got = inst.output("last_hidden").reshape(B * S, -1)
    wr = r16w(w) if precision == "fp16" else w
    ref = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids, seg, cfg.eps), B, S, mask)
    err = rel_err(got, ref)
    say("  max rel err %.3g" % err)
    assert err <= (FP16_TOL if precision == "fp16" else 1e-4)
    # second forward with other inputs on the same instance (blob memory is reused between layers)
    ids2, seg2, lens2, mask2 = make_inputs(cfg, B, S, 30, 96, seed=9)
    inst.set_input("input_ids", ids2)
    inst.set_input("token_type_ids", seg2)
    inst.set_input("attention_bias", mask2.reshape(B, 1, 1, S))
    inst.forward()
    got2 = inst.output("last_hidden").reshape(B * S, -1)
    ref2 = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids2, seg2, cfg.eps), B, S, mask2)
    assert rel_err(got2, ref2) <= (FP16_TOL if precision == "fp16" else 1e-4)
    inst.close()


def test_int8_ffn_from_model_files_bit_exact(monkeypatch):
    host, tnnmodel, *_ = _mods()
    say("host: QuantizedInnerProduct -> GELU -> QuantizedInnerProduct, fp32 boundaries")
    rng = np.random.default_rng(0)
    T, K, F = 256, 768, 3072
    x = rng.standard_normal((T, K)).astype(np.float32)
    w1 = rng.integers(-127, 128, (F, K), dtype=np.int8)
    w2 = rng.integers(-127, 128, (K, F), dtype=np.int8)
    b1 = rng.integers(-500, 500, F).astype(np.int32)
    b2 = rng.integers(-500, 500, K).astype(np.int32)
    ws1 = (rng.uniform(0.5, 1.5, F) * 6e-5).astype(np.float32)
    ws2 = (rng.uniform(0.5, 1.5, K) * 3e-5).astype(np.float32)
    s_a, s_h, s_g, s_y = (np.float32(v) for v in (0.031, 0.045, 0.027, 0.052))
    g = tnnmodel.int8_ffn_graph(T, K, F, w1, b1, ws1, w2, b2, ws2, s_a, s_h, s_g, s_y)
    qa = orc.quantize_x86(x, s_a)
    h, _ = orc.fc_int8(qa, w1, b1, orc.fc_int8_scale(ws1, s_h, F))
    ref_act = orc.gelu(orc.dequantize(h, s_h))
    gq = orc.quantize_x86(ref_act, s_g)
    yq, _ = orc.fc_int8(gq, w2, b2, orc.fc_int8_scale(ws2, s_y, K))
    assert np.abs(h).max() > 20  # the requantisation really exercised the int8 range
    outs = {}
    # once as the explicit chain (Reformat layers as the engine inserts them), once with the Reformat layers folded
    # into their neighbours by the ROCm int8 pass
    for fuse, want in (("0", {"Reformat": 4, "QuantizedInnerProduct": 2}),
                       ("1", {"Reformat": 1, "RocmQuantLinearGelu": 1, "RocmFusedLinearInt8": 1})):
        monkeypatch.setenv("TNN_ROCM_FUSE_INT8", fuse)
        inst = host.RocmInstance.from_graph(g, "fp32")
        types = [t for t, _ in inst.layers()]
        for k, n in want.items():
            assert types.count(k) == n, types
        inst.set_input("x", x)
        inst.forward()
        got = inst.output("y")
        inst.close()
        # the two int8 GEMMs, both quantisers and the GELU between them (double erf, as the CPU path) are bit-exact
        diff = np.abs(np.rint(got / s_y) - yq.astype(np.float64))
        say("  fuse=%s mismatching int8 outputs: %d of %d" % (fuse, int((diff != 0).sum()), diff.size))
        assert diff.max() == 0
        outs[fuse] = got
    assert np.array_equal(outs["0"], outs["1"])  # folding the Reformat layers changes no value in fp32


def test_host_error_paths():
    host, tnnmodel, *_ = _mods()
    say("host: error paths")
    g = tnnmodel.Graph()
    g.add_input("x", [4, 8])
    g.add_layer("GELU", "g", ["x"], ["y"])
    g.add_output("y")
    proto, model = g.proto(), g.model()
    with pytest.raises(host.HostError, match="not supported"):
        host.RocmInstance(proto.replace("GELU g", "Convolution g"), model)   # unknown layer type
    with pytest.raises(host.HostError):
        host.RocmInstance(proto, model[: len(model) // 2] if len(model) > 16 else b"")  # truncated / empty model
    inst = host.RocmInstance(proto, model, "fp32")
    with pytest.raises(host.HostError, match="dont have the input"):
        inst.set_input("nope", np.zeros((4, 8), np.float32))
    with pytest.raises(host.HostError):
        inst.set_input("x", np.zeros((4, 9), np.float32))                    # wrong element count
    inst.close()
    # MatMul with inconsistent shapes is rejected at Init like the engine's shape inference does
    g = tnnmodel.Graph()
    g.add_input("a", [4, 8])
    g.add_input("b", [7, 5])
    g.add_layer("MatMul", "mm", ["a", "b"], ["c"], [-1])
    g.add_output("c")
    with pytest.raises(host.HostError, match="wrong shape"):
        host.RocmInstance(g.proto(), g.model(), "fp32")
    # Gather index out of range surfaces as an error from Forward (the engine returns TNNERR_MODEL_ERR)
    g = tnnmodel.Graph()
    g.add_input("ids", [1, 4], tnnmodel.DT_INT32)
    g.add_layer("Gather", "emb", ["ids"], ["e"], [0, 1, 0])
    g.res_gather("emb", np.ones((10, 8), np.float32))
    g.add_output("e")
    inst = host.RocmInstance(g.proto(), g.model(), "fp32")
    inst.set_input("ids", np.array([[0, 3, 9, 2]], np.int32))
    inst.forward()
    assert inst.output("e").shape == (1, 4, 8)
    inst.set_input("ids", np.array([[0, 3, 10, 2]], np.int32))
    with pytest.raises(host.HostError, match="invalid slice_index"):
        inst.forward()
    inst.close()


def test_graph_replay_matches_eager_on_every_replay(monkeypatch):
    """The whole-forward graph (recorded on the third Forward) must reproduce the eager result on every replay, with
    new inputs each time and unrelated eager GPU work and synchronisations between the replays."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: graph replay vs eager")
    cfg = EncoderConfig.bert_base(2)
    w = make_weights(cfg, seed=13, bias_std=0.02)
    B, S = 2, 128
    g = tnnmodel.encoder_graph(cfg, w, B, S)
    monkeypatch.setenv("TNN_ROCM_GRAPH", "0")
    eager = host.RocmInstance.from_graph(g, "fp16")
    monkeypatch.setenv("TNN_ROCM_GRAPH", "1")
    graph = host.RocmInstance.from_graph(g, "fp16")
    monkeypatch.delenv("TNN_ROCM_GRAPH")          # the library's own default (the eager loop)
    default = host.RocmInstance.from_graph(g, "fp16")
    scratch = torch.zeros(1 << 20, device="cuda")
    for it in range(7):
        ids, seg, lens, mask = make_inputs(cfg, B, S, 20, 128, seed=100 + it)
        outs = []
        for inst in (eager, graph, default):
            inst.set_input("input_ids", ids)
            inst.set_input("token_type_ids", seg)
            inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
            inst.forward()
            outs.append(inst.output("last_hidden"))
        assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2]), "replay %d differs from eager" % it
        # unrelated eager work + a device synchronisation between replays
        scratch.add_(1.0)
        assert float(scratch.sum().item()) == (it + 1) * (1 << 20)
        torch.cuda.synchronize()
    eager.close()
    graph.close()
    default.close()


def test_recorded_forwards_follow_the_store_switch(monkeypatch, capfd):
    """The form of the result stores is an argument of every launch: an instance that replays recorded forwards records again
    when the switch is set, and finds its recording when it is set back."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    from tnn_amd import capi
    lib = capi.load()
    say("host: store switch and graph replay")
    cfg, B, S = EncoderConfig.bert_base(1), 1, 64
    g = tnnmodel.encoder_graph(cfg, make_weights(cfg, seed=13, bias_std=0.02), B, S)
    monkeypatch.setenv("TNN_ROCM_GRAPH", "1")
    monkeypatch.setenv("TNN_ROCM_VERBOSE", "1")
    inst = host.RocmInstance.from_graph(g, "fp16")
    ids, seg, lens, mask = make_inputs(cfg, B, S, 20, S, seed=100)
    for n, v in (("input_ids", ids), ("token_type_ids", seg), ("attention_bias", mask.reshape(B, 1, 1, S))):
        inst.set_input(n, v)
    capfd.readouterr()
    outs, recorded = [], []
    try:
        for through in (1, 0, 1, 0):
            assert lib.tnn_rocm_debug_set_store_through(through) == 0
            for _ in range(4):
                inst.forward()
            outs.append(inst.output("last_hidden").copy())
            recorded.append(capfd.readouterr().err.count("forward recorded"))
    finally:
        lib.tnn_rocm_debug_set_store_through(1)
    assert recorded == [1, 1, 0, 0]
    assert all(np.array_equal(o, outs[0]) for o in outs)
    inst.close()


def test_two_instances_on_two_threads_match_their_sequential_results():
    """One Context per Instance, instances used from different threads at the same time (the engine's threading
    contract, source/tnn/core/instance.cc and default_network.cc:632-633: all work of an instance on its own stream,
    Forward returns after its own Synchronize).  Each thread drives its own instance through eager forwards, the
    recording forward and replays; every result must equal the one the same instance gave when it ran alone."""
    import threading
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: two instances, two threads")
    cfg = EncoderConfig.bert_base(2)
    shapes = [(2, 128), (3, 96)]
    insts, feeds, alone = [], [], []
    for k, (B, S) in enumerate(shapes):
        w = make_weights(cfg, seed=70 + k, bias_std=0.02)
        insts.append(host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "fp16"))
        feeds.append([make_inputs(cfg, B, S, 17, S, seed=300 + 10 * k + it) for it in range(6)])

    def run(k, out):
        B, S = shapes[k]
        for ids, seg, lens, mask in feeds[k]:
            insts[k].set_input("input_ids", ids)
            insts[k].set_input("token_type_ids", seg)
            insts[k].set_input("attention_bias", mask.reshape(B, 1, 1, S))
            insts[k].forward()
            out.append(insts[k].output("last_hidden").copy())

    for k in range(2):
        ref = []
        run(k, ref)
        alone.append(ref)
    together = [[], []]
    errors = []

    def guarded(k):
        try:
            run(k, together[k])
        except Exception as e:  # surfaced below: an exception in a thread would otherwise pass silently
            errors.append((k, repr(e)))

    threads = [threading.Thread(target=guarded, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors, errors
    assert all(not t.is_alive() for t in threads)
    for k in range(2):
        assert len(together[k]) == len(alone[k])
        for it, (a, b) in enumerate(zip(alone[k], together[k])):
            assert np.array_equal(a, b), "instance %d forward %d differs when another instance runs beside it" % (k, it)
    for inst in insts:
        inst.close()


def test_forward_with_callback_visits_every_layer():
    """Instance::ForwardWithCallback (default_network.cc:637-668): `before` sees every layer's input blobs, `after` its
    output blobs once the layer has finished, in layer order; the forward gives the values of a plain Forward."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: ForwardWithCallback")
    cfg = EncoderConfig.bert_base(2)
    w = make_weights(cfg, seed=90, bias_std=0.02)
    B, S = 2, 64
    ids, seg, lens, mask = make_inputs(cfg, B, S, 17, S, seed=91)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "fp16")
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    inst.forward()
    plain = inst.output("last_hidden").copy()
    seen = []
    inst.forward_with_callback(before=lambda name, typ, blobs: seen.append(("in", name, typ, blobs)),
                               after=lambda name, typ, blobs: seen.append(("out", name, typ, blobs)))
    assert np.array_equal(inst.output("last_hidden"), plain)
    layers = inst.layers()
    io = inst.layer_io()
    assert len(seen) == 2 * len(layers)
    for k, ((typ, name), layer) in enumerate(zip(layers, io)):
        b, a = seen[2 * k], seen[2 * k + 1]
        assert (b[0], b[1], b[2]) == ("in", name, typ) and (a[0], a[1], a[2]) == ("out", name, typ)
        assert [x[0] for x in b[3]] == layer["inputs"] and [x[0] for x in a[3]] == layer["outputs"]
        assert [x[1] for x in a[3]] == [int(np.prod(d)) for d in layer["output_dims"]]
    assert seen[-1][3][0][0] == "last_hidden" and seen[-1][3][0][1] == B * S * cfg.hidden
    inst.close()


def test_share_command_queue_and_cpu_threads():
    """Instance::ShareCommandQueue (instance.cc:158-160, default_network.cc:537-556; the CUDA backend's counterpart is
    cuda_context.cc:91-122): the second instance launches on the first one's stream from then on - its forwards, enqueued
    without waiting, are ordered behind the first instance's on that one stream, one synchronise covers both, and every
    result equals the one the instance gave on its own stream (eager, recording and replayed forwards).
    SetCpuNumThreads is accepted."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: two instances on one shared command queue")
    cfg = EncoderConfig.bert_base(2)
    shapes = [(2, 128), (3, 96)]
    insts, feeds = [], []
    for k, (B, S) in enumerate(shapes):
        w = make_weights(cfg, seed=80 + k, bias_std=0.02)
        insts.append(host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "fp16"))
        ids, seg, lens, mask = make_inputs(cfg, B, S, 17, S, seed=400 + k)
        feeds.append({"input_ids": ids, "token_type_ids": seg, "attention_bias": mask.reshape(B, 1, 1, S)})
        for name, arr in feeds[k].items():
            insts[k].set_input(name, arr)
    alone = []
    for inst in insts:
        inst.forward()
        alone.append(inst.output("last_hidden").copy())
    assert insts[0].stream != insts[1].stream
    insts[1].set_cpu_num_threads(4)
    insts[1].share_command_queue(insts[0])
    assert insts[0].stream == insts[1].stream
    for it in range(5):
        insts[0].forward_async()
        insts[1].forward_async()
        insts[0].sync()                      # the one stream: both forwards are done
        for k in range(2):
            assert np.array_equal(insts[k].output("last_hidden"), alone[k]), (it, k)
    insts[1].close()                         # the sharer goes first: the stream belongs to instance 0
    insts[0].forward()
    assert np.array_equal(insts[0].output("last_hidden"), alone[0])
    insts[0].close()


def test_int8_encoder_full_shape_properties(monkeypatch):
    """Benchmark config 4's per-layer shape (B16 S256, hidden 768, FFN 3072; 3 layers to keep the case short):
    calibrated on this backend's fp32 forward, then run quantised in fp16 mode.  Size-independent checks: every
    projection of the first and last layer reproduces its own int8 output bit-exactly from its own input blob (checker
    on a 192-row slice), the folded graph agrees with the explicit Reformat chain, and the quantised network stays
    close to the float one."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    import golden_util
    from tnn_amd import quant
    say("host: int8 encoder at B16 S256, properties")
    cfg = EncoderConfig.bert_base(3)
    w = make_weights(cfg, seed=41)
    B, S = 16, 256
    ids, seg, lens, mask = make_inputs(cfg, B, S, 100, 256, seed=42)
    inputs = {"input_ids": ids, "token_type_ids": seg, "attention_bias": mask.reshape(B, 1, 1, S)}
    names = quant.calibration_outputs(cfg)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S, extra_outputs=names), "fp32")
    for k, v in inputs.items():
        inst.set_input(k, v)
    inst.forward()
    scales = {n: quant.activation_scale(inst.output(n, max_elems=1 << 26)) for n in names}
    float_out = inst.output("last_hidden")
    inst.close()
    check = ["x0"] + ["l%d_%s" % (li, b) for li in (0, 2) for b in quant.CALIBRATION_BLOBS] + ["l1_x2"]
    runs = {}
    for fuse, extra in (("0", check), ("1", [])):
        monkeypatch.setenv("TNN_ROCM_FUSE_INT8", fuse)
        inst = host.RocmInstance.from_graph(quant.int8_encoder_graph(cfg, w, scales, B, S, extra_outputs=extra), "fp16")
        for k, v in inputs.items():
            inst.set_input(k, v)
        inst.forward()
        runs[fuse] = inst.output("last_hidden")
        if fuse == "0":
            blobs = {n: inst.output(n, max_elems=1 << 26) for n in extra}
        else:
            types = [t for t, _ in inst.layers()]
            assert types.count("RocmFusedAttention") == 3 and types.count("RocmFusedLinearInt8") == 6, types
        inst.close()
    n = golden_util.check_projections_bit_exact(cfg, w, scales, blobs, B * S, orc.quantize_x86, layers=(0, 2), rows=192)
    assert n == 12
    e_fused, e_float = rel_err(runs["1"], runs["0"]), rel_err(runs["1"], float_out)
    say("  folded vs explicit chain %.3g ; quantised vs float network %.3g" % (e_fused, e_float))
    # folding keeps float intermediates in fp32 where the chain rounds them to fp16: a few int8 steps may flip
    assert e_fused <= 3e-2 and e_float <= 8e-2
    valid = (np.arange(S)[None, :] < lens[:, None])
    assert np.isfinite(runs["1"]).all() and np.abs(runs["1"][valid].mean(-1)).max() < 5e-3  # LayerNorm(gamma=1, beta=0)


@pytest.mark.parametrize("name,hidden,heads,ffn,B,S,lo,hi", [("config 2 (BERT-base B8 S384)", 768, 12, 3072, 8, 384, 200, 384),
                                                             ("config 5 (BERT-large B16 S512)", 1024, 16, 4096, 16, 512, 300, 512)])
def test_encoder_full_batch_shape_against_checker_on_one_sequence(name, hidden, heads, ffn, B, S, lo, hi):
    """The benchmark configurations at their full batch and sequence length (2 layers): the whole batch runs on the
    device from model files; sequences are independent, so the checker evaluates ONE of them (the one with the shortest
    valid length, which has the most padding) and must agree with that slice of the device result."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: %s, fp16, one sequence against the checker" % name)
    cfg = EncoderConfig(2, hidden, heads, ffn)
    w = make_weights(cfg, seed=51, bias_std=0.02)
    ids, seg, lens, mask = make_inputs(cfg, B, S, lo, hi, seed=52)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "fp16")
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    for _ in range(4):  # eager, eager, graph capture, graph replay: every mode must give the same result
        inst.forward()
    got = inst.output("last_hidden", max_elems=1 << 26).reshape(B, S, hidden)
    inst.close()
    b = int(np.argmin(lens))
    w16 = r16w(w)
    x0 = encoder_ref.embed(w16, ids[b:b + 1], seg[b:b + 1], cfg.eps)
    ref = encoder_ref.encoder(w16, cfg, x0, 1, S, mask[b:b + 1])
    err = rel_err(got[b].reshape(S, hidden), ref)
    say("  sequence %d (valid length %d of %d): max rel err %.3g" % (b, lens[b], S, err))
    assert err <= FP16_TOL
    assert np.isfinite(got).all()


def test_encoder_bf16_from_model_files():
    """PRECISION_LOW: bf16 activations and weights through the same fused layers.  The bar written for this path is
    4e-2 (bf16 keeps 8 mantissa bits: one rounding is 4e-3 relative, and two encoder layers stack a few dozen)."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: 2-layer encoder, bf16")
    cfg = EncoderConfig.bert_base(2)
    w = make_weights(cfg, seed=3, bias_std=0.02)
    B, S = 2, 96
    ids, seg, lens, mask = make_inputs(cfg, B, S, 30, 96, seed=4)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "bf16")
    types = [t for t, _ in inst.layers()]
    assert types.count("RocmFusedAttention") == 2 and types.count("RocmFusedLinear") == 6, types
    assert types.count("RocmFusedEmbedding") == 1 and "Gather" not in types, types
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    inst.forward()
    got = inst.output("last_hidden").reshape(B * S, -1)
    inst.close()
    x0 = encoder_ref.embed(w, ids, seg, cfg.eps)
    ref = encoder_ref.encoder(w, cfg, x0, B, S, mask)
    err = rel_err(got, ref)
    say("  max rel err %.3g" % err)
    assert err <= 4e-2


def test_layernorm_folding_switch(monkeypatch):
    """TNN_ROCM_FOLD_LN=0 keeps every LayerNorm a launch of its own, TNN_ROCM_LN_STATS=0 keeps the output tensor of a
    folded LayerNorm for the residual that reads it, TNN_ROCM_LN_SUMS=0 makes every folding GEMM take the row statistics
    from its own operand; all four graphs agree with each other to fp16 rounding and with the checker."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: LayerNorm folding on / off, 2-layer encoder fp16")
    cfg = EncoderConfig.bert_base(2)
    w = make_weights(cfg, seed=13, bias_std=0.05)
    rng = np.random.default_rng(14)
    for lw in w["layers"]:   # non-trivial LayerNorm scale / shift
        for k in ("ln1_g", "ln2_g"):
            lw[k] = (1 + 0.2 * rng.standard_normal(cfg.hidden)).astype(np.float32)
        for k in ("ln1_b", "ln2_b"):
            lw[k] = (0.3 * rng.standard_normal(cfg.hidden)).astype(np.float32)
    B, S = 3, 104
    ids, seg, lens, mask = make_inputs(cfg, B, S, 30, S, seed=15)
    g = tnnmodel.encoder_graph(cfg, w, B, S)
    outs = {}
    for fold, n_ln in (("0", 4), ("1", 1), ("y", 1), ("s", 1)):
        monkeypatch.setenv("TNN_ROCM_FOLD_LN", "0" if fold == "0" else "1")
        monkeypatch.setenv("TNN_ROCM_LN_STATS", "0" if fold == "y" else "1")
        monkeypatch.setenv("TNN_ROCM_LN_SUMS", "0" if fold == "s" else "1")
        inst = host.RocmInstance.from_graph(g, "fp16")
        types = [t for t, _ in inst.layers()]
        assert types.count("LayerNorm") == n_ln, types
        inst.set_input("input_ids", ids)
        inst.set_input("token_type_ids", seg)
        inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
        for _ in range(4):   # the fourth forward replays the captured graph
            inst.forward()
        outs[fold] = inst.output("last_hidden").reshape(B * S, -1)
        inst.close()
    wr = r16w(w)
    ref = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids, seg, cfg.eps), B, S, mask)
    e0, e1, e01 = rel_err(outs["0"], ref), rel_err(outs["1"], ref), rel_err(outs["1"], outs["0"])
    ey, e1y = rel_err(outs["y"], ref), rel_err(outs["1"], outs["y"])
    es, e1s = rel_err(outs["s"], ref), rel_err(outs["1"], outs["s"])
    say("  un-folded %.3g  folded %.3g  folded, output kept %.3g  folded, own statistics %.3g  folded vs un-folded %.3g  "
        "vs output kept %.3g  vs own statistics %.3g" % (e0, e1, ey, es, e01, e1y, e1s))
    assert max(e0, e1, ey, es, e01, e1y, e1s) <= FP16_TOL


@pytest.mark.parametrize("hidden,heads,ffn,B,S,n_ln", [
    (1024, 16, 4096, 2, 64, 1),    # BERT-large widths: every LayerNorm but the last is folded
    (768, 12, 3072, 2, 100, 2),    # S is no multiple of 8: packed-QKV attention path, its LayerNorm stays a launch
    (256, 4, 1024, 3, 40, 1),      # small widths (single-slab K for the 256-byte-slab tiles)
    (192, 3, 768, 2, 48, 4),       # hidden is no multiple of 128: no LayerNorm is folded
])
def test_encoder_other_shapes_fp16(hidden, heads, ffn, B, S, n_ln):
    """Two encoder layers at other widths / sequence lengths through Instance::Forward (fp16, fused) against the
    checker; which LayerNorms the fusion pass may fold depends on the shape."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: 2-layer encoder hidden=%d heads=%d ffn=%d B=%d S=%d" % (hidden, heads, ffn, B, S))
    cfg = EncoderConfig(2, hidden, heads, ffn)
    w = make_weights(cfg, seed=hidden + S, bias_std=0.05)
    rng = np.random.default_rng(S)
    for lw in w["layers"]:
        for k in ("ln1_g", "ln2_g"):
            lw[k] = (1 + 0.2 * rng.standard_normal(hidden)).astype(np.float32)
        for k in ("ln1_b", "ln2_b"):
            lw[k] = (0.3 * rng.standard_normal(hidden)).astype(np.float32)
    ids, seg, lens, mask = make_inputs(cfg, B, S, S // 3, S, seed=S + 1)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "fp16")
    types = [t for t, _ in inst.layers()]
    say("  layers: " + " ".join("%s x%d" % (t, types.count(t)) for t in sorted(set(types))))
    assert types.count("RocmFusedAttention") == 2 and types.count("LayerNorm") == n_ln, types
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    for _ in range(4):
        inst.forward()
    got = inst.output("last_hidden").reshape(B * S, -1)
    inst.close()
    wr = r16w(w)
    ref = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids, seg, cfg.eps), B, S, mask)
    err = rel_err(got, ref)
    say("  max rel err %.3g" % err)
    assert err <= FP16_TOL


def test_model_check_and_profile_report():
    """The per-blob check tool (fused fp16 graph against the un-fused fp32 graph on the device) on a 2-layer encoder:
    every surviving blob within the fp16 bar, the checked graph identical to the production graph; and the per-layer
    profile report lists every layer of the optimised graph with its dims."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    from tnn_amd import model_check
    say("host: model_check on a 2-layer encoder, fp16")
    cfg = EncoderConfig.bert_base(2)
    w = make_weights(cfg, seed=21, bias_std=0.02)
    B, S = 2, 128
    ids, seg, lens, mask = make_inputs(cfg, B, S, 40, S, seed=22)
    graph = tnnmodel.encoder_graph(cfg, w, B, S)
    inputs = {"input_ids": ids, "token_type_ids": seg, "attention_bias": mask.reshape(B, 1, 1, S)}
    rows, same = model_check.check(graph, inputs, "fp16")
    say(model_check.report(rows))
    assert same and len(rows) >= 10
    assert all(r["ok"] for r in rows), [r for r in rows if not r["ok"]]
    assert {"RocmFusedAttention", "RocmFusedLinear", "RocmFusedEmbedding", "LayerNorm"} <= {r["type"] for r in rows}
    inst = host.RocmInstance.from_graph(graph, "fp16")
    for k, v in inputs.items():
        inst.set_input(k, v)
    for _ in range(3):
        inst.forward()
    text = inst.profile_table(3)
    inst.close()
    say(text)
    assert "Profiling Data Sort by Cost time" in text and "kernel runtime total" in text and "[2,128,3072] [2,128,768]" in text
    assert text.count("RocmFusedLinear") >= 12   # six layers in each of the two per-layer tables


@pytest.mark.parametrize("keep_ln_outputs", [False, True])
def test_model_check_device_against_cpu_checker_blob_by_blob(keep_ln_outputs, monkeypatch):
    """tools/model_check's comparison proper: every blob of the fused fp16 graph that survives the optimiser passes
    against the same blob as the CPU evaluates the decomposed graph (tests/encoder_ref.encoder_blobs, the CPU checker
    layer by layer), plus the engine's own element-wise pass rule.  By default the LayerNorm outputs inside a layer are
    rebuilt by their readers and never exist; TNN_ROCM_LN_STATS=0 keeps them as blobs, and they are checked as well."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    from tnn_amd import model_check
    say("host: model_check, device vs CPU checker, 3-layer encoder fp16, LayerNorm outputs %s"
        % ("kept" if keep_ln_outputs else "rebuilt by their readers"))
    monkeypatch.setenv("TNN_ROCM_LN_STATS", "0" if keep_ln_outputs else "1")
    cfg = EncoderConfig.bert_base(3)
    w = make_weights(cfg, seed=31, bias_std=0.02)
    B, S = 2, 96
    ids, seg, lens, mask = make_inputs(cfg, B, S, 30, S, seed=32)
    graph = tnnmodel.encoder_graph(cfg, w, B, S)
    inputs = {"input_ids": ids, "token_type_ids": seg, "attention_bias": mask.reshape(B, 1, 1, S)}
    reference = encoder_ref.encoder_blobs(r16w(w), cfg, ids, seg, B, S, mask)
    rows, same, skipped = model_check.check_against(graph, inputs, reference, "fp16")
    say(model_check.report(rows))
    assert same and not skipped, skipped
    names = {r["blob"] for r in rows}
    # what survives per layer: the attention context, the three sums the LayerNorms read (outputs of the projections
    # with the residual folded in), the FFN activation, and (when kept) the LayerNorm outputs needed as residuals
    assert {"x0", "l0_ctx", "l0_sum1", "l0_act", "l0_sum2", "l2_ctx", "last_hidden"} <= names, sorted(names)
    assert ({"l0_x1", "l0_x2", "l1_x1"} <= names) == keep_ln_outputs, sorted(names)
    assert all(r["ok"] for r in rows), [r for r in rows if not r["ok"]]
    # the engine's element rule (|d|/(|a|+|b|) > 0.005 and |d| > 1e-3) is written for an fp32 device; in fp16 a value of
    # size 1 carries an ulp of 1e-3, so a few small elements trip it as the layers stack up: they are reported per blob
    # and bounded here (observed: none in the first layer, 0.3 % of the last hidden state after three layers)
    T = B * S
    for r in rows:
        n = T * (cfg.ffn if r["blob"].endswith("_act") else cfg.hidden)
        assert r["engine_rule_failures"] <= 0.01 * n, (r["blob"], r["engine_rule_failures"], n)
    assert all(r["engine_rule_failures"] == 0 for r in rows if r["blob"] in ("x0", "l0_ctx", "l0_sum1", "l0_act", "l0_x1"))


def test_instance_reshape_matches_fresh_instances():
    """Instance::Reshape (default_network.cc:456-500): one instance moved through several (B, S) gives, at each shape and
    on each of four forwards (eager, eager, record + launch, replay), exactly what an instance created at that shape
    gives; weights are uploaded once; a shape beyond the planned blob memory re-plans it; a shape seen before replays
    its recording.  One shape is also held against the checker."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: Instance::Reshape through several shapes, 2-layer encoder fp16")
    cfg = EncoderConfig(2, 256, 4, 512)
    S_MAX = 96
    w = make_weights(cfg, seed=21, bias_std=0.05)
    w["pos_emb"] = w["pos_emb"][:S_MAX]

    def shapes(B, S):
        return {"input_ids": [B, S], "token_type_ids": [B, S], "attention_bias": [B, 1, 1, S]}

    def feed(inst, B, S, seed):
        ids, seg, lens, mask = make_inputs(cfg, B, S, max(S // 3, 1), S, seed=seed)
        inst.set_input("input_ids", ids)
        inst.set_input("token_type_ids", seg)
        inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
        return ids, seg, mask

    g = tnnmodel.encoder_graph(cfg, w, 4, S_MAX, dynamic=True)
    inst = host.RocmInstance.from_graph(g, "fp16", input_shapes=shapes(4, 64))
    types = [t for t, _ in inst.layers()]
    assert types.count("RocmFusedAttention") == 2 and types.count("RocmFusedEmbedding") == 1, types
    assert types.count("LayerNorm") == 1, types     # folding also happens when S is only known at reshape time
    # (4,64) created; shrink twice; S not a multiple of 8; beyond the planned memory; back to shapes seen before
    walk = [(4, 64), (2, 40), (3, 24), (2, 36), (5, 96), (2, 40), (4, 64), (1, 8)]
    for step, (B, S) in enumerate(walk):
        say("  shape B=%d S=%d" % (B, S))
        if step:
            inst.reshape(shapes(B, S))
        io = {l["name"]: l for l in inst.layer_io()}
        assert any(d == [B, S, cfg.hidden] for l in io.values() for d in l["output_dims"])
        ids, seg, mask = feed(inst, B, S, 100 + step)
        fresh = host.RocmInstance.from_graph(g, "fp16", input_shapes=shapes(B, S))
        feed(fresh, B, S, 100 + step)
        fresh.forward()
        want = fresh.output("last_hidden")
        fresh.close()
        assert want.shape == (B, S, cfg.hidden)
        for it in range(4):
            inst.forward()
            got = inst.output("last_hidden")
            assert got.shape == want.shape
            assert np.array_equal(got, want), "shape %s forward %d differs from a fresh instance" % ((B, S), it)
        if (B, S) == (2, 36):
            wr = r16w(w)
            ref = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids, seg, cfg.eps), B, S, mask)
            err = rel_err(got.reshape(B * S, -1), ref)
            say("  S=36 against the checker: max rel err %.3g" % err)
            assert err <= FP16_TOL
    # error behaviour of default_network.cc:470-475 (unknown blob) plus the rank check
    with pytest.raises(host.HostError, match="blob name is wrong"):
        inst.reshape({"no_such_input": [1, 8]})
    with pytest.raises(host.HostError, match="number of dimensions"):
        inst.reshape({"input_ids": [8]})
    # inputs that no longer agree with each other fail in the layer that notices, with its name
    with pytest.raises(host.HostError):
        inst.reshape({"input_ids": [2, 16]})
    inst.close()


@pytest.mark.parametrize("B,S", [(1, 2), (2, 33), (3, 128), (1, 200)])
def test_fp32_attention_group_equals_its_layers(B, S):
    """A plain fp32 forward runs every attention core as one group; ForwardWithCallback runs the same instance's layers one
    by one.  Same answer at fp32 accuracy, before and after Instance::Reshape, and against the checker."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: fp32 attention group, B=%d S=%d" % (B, S))
    cfg = EncoderConfig(2, 128, 2, 256)
    w = make_weights(cfg, seed=31, bias_std=0.05)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, 2, 200, dynamic=True), "fp32")
    for b, s in ((2, 200), (B, S)):
        if (b, s) != (2, 200):
            inst.reshape({"input_ids": [b, s], "token_type_ids": [b, s], "attention_bias": [b, 1, 1, s]})
        ids, seg, lens, mask = make_inputs(cfg, b, s, max(1, s // 3), s, seed=50 + s)
        for n, v in (("input_ids", ids), ("token_type_ids", seg), ("attention_bias", mask.reshape(b, 1, 1, s))):
            inst.set_input(n, v)
        inst.forward()
        got = inst.output("last_hidden").reshape(b * s, -1).copy()
        seen = []
        inst.forward_with_callback(after=lambda name, typ, blobs: seen.append(typ))
        assert seen.count("Softmax") == 2
        alone = inst.output("last_hidden").reshape(b * s, -1)
        ref = encoder_ref.encoder(w, cfg, encoder_ref.embed(w, ids, seg, cfg.eps), b, s, mask)
        assert rel_err(got, alone) <= 3e-6 and rel_err(got, ref) <= FP32_ASSERT
    inst.close()


def test_fp32_attention_group_equals_its_layers_where_a_mask_hides_every_key():
    """An additive mask of -inf throughout leaves a sequence without an answer: NaN from the softmax layer, and from the group;
    the other sequence is not concerned."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: fp32 attention group, a mask of -inf")
    cfg, B, S = EncoderConfig(2, 128, 2, 256), 2, 40
    w = make_weights(cfg, seed=31, bias_std=0.05)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), "fp32")
    ids, seg, lens, mask = make_inputs(cfg, B, S, 20, S, seed=51)
    mask[1] = -np.inf
    for n, v in (("input_ids", ids), ("token_type_ids", seg), ("attention_bias", mask.reshape(B, 1, 1, S))):
        inst.set_input(n, v)
    inst.forward()
    got = inst.output("last_hidden").reshape(B, S, -1).copy()
    inst.forward_with_callback(after=lambda name, typ, blobs: None)
    alone = inst.output("last_hidden").reshape(B, S, -1)
    assert np.isnan(alone[1]).all() and np.isnan(got[1]).all()
    assert rel_err(got[0], alone[0]) <= 3e-6
    inst.close()


@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16"])
def test_two_attention_masks_in_one_net(precision):
    """Two layers, each with a padding mask of its own, made in the graph as Sub(1 - m) -> Mul(-10000) right in front of the
    layer: the memory plan gives the second mask the buffer of the first one, whose last reader has passed by then.  Each
    layer has to see its own mask: in Forward, layer by layer (ForwardWithCallback), and against the checker."""
    host, tnnmodel, EncoderConfig, make_weights, _ = _mods()
    say("host: two attention masks, " + precision)
    cfg = EncoderConfig(2, 128, 2, 256)
    B, S = 2, 48
    w = make_weights(cfg, seed=61, bias_std=0.05, with_embeddings=False)
    for lw in w["layers"]:  # an attention output that weighs as much as the residual beside it
        lw["wv"], lw["wo"] = lw["wv"] * 4, lw["wo"] * 8
    g = tnnmodel.encoder_graph(cfg, w, B, S, with_embeddings=False)
    g.inputs = [i for i in g.inputs if i[0] != "attention_bias"]
    layers = []
    for t, n, i, o, pr in g.layers:
        if n in ("l0_q_mm", "l1_q_mm"):
            mk = "m" + n[1]
            g.add_input(mk, [B, 1, 1, S])
            g.res_eltwise(mk + "_inv", "Sub", np.array([1.0], np.float32))      # constant first: 1 - m
            g.res_eltwise(mk + "_scale", "Mul", np.array([-10000.0], np.float32))
            for b in ("_pad", "_bias"):
                g._blob(mk + b)
            layers += [("Sub", mk + "_inv", [mk], [mk + "_pad"], ["0"]), ("Mul", mk + "_scale", [mk + "_pad"], [mk + "_bias"], ["1"])]
        layers.append((t, n, ["m" + n[1] + "_bias" if b == "attention_bias" else b for b in i], o, pr))
    g.layers = layers
    rng = np.random.default_rng(62)
    x = rng.standard_normal((B, S, cfg.hidden)).astype(np.float32)
    lens = [np.array([40, 9]), np.array([17, 48])]
    keep = [(np.arange(S)[None, :] < n[:, None]).astype(np.float32) for n in lens]
    inst = host.RocmInstance.from_graph(g, precision)
    inst.set_input("hidden", x)
    for k in (0, 1):
        inst.set_input("m%d" % k, keep[k].reshape(B, 1, 1, S))
    inst.forward()
    got = inst.output("last_hidden").reshape(B * S, -1).copy()
    inst.forward_with_callback(after=lambda name, typ, blobs: None)
    alone = inst.output("last_hidden").reshape(B * S, -1)

    def checker(masks):
        y = x.reshape(B * S, -1)
        for lw, m in zip(w["layers"], masks):
            y = encoder_ref.encoder_layer(y, lw, B, S, cfg.heads, (1 - m) * np.float32(-10000.0), cfg.eps)
        return y

    ref = checker(keep)
    tol = {"fp32": FP32_ASSERT, "fp16": FP16_TOL, "bf16": BF16_TOL}[precision]
    err, err_alone = rel_err(got, ref), rel_err(got, alone)
    say("  to the checker %.3g, to the layers one by one %.3g" % (err, err_alone))
    assert rel_err(checker([keep[0], keep[0]]), ref) > 4 * tol  # the first mask twice would be seen
    assert err <= tol and err_alone <= (3e-6 if precision == "fp32" else 0)
    inst.close()


def test_instance_reshape_fp32_batch_only_with_static_head_split():
    """A graph whose head split names B and S cannot change them (the element count check of reshape_layer.cc:41-63
    fails, as in the engine); the error names the layer.  The un-fused fp32 path reshapes through the dynamic graph."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: Instance::Reshape on fp32 graphs")
    cfg = EncoderConfig(1, 128, 2, 256)
    w = make_weights(cfg, seed=31, bias_std=0.05)
    w["pos_emb"] = w["pos_emb"][:32]
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, 2, 32), "fp32")
    with pytest.raises(host.HostError, match="reshape of layer"):
        inst.reshape({"input_ids": [2, 16], "token_type_ids": [2, 16], "attention_bias": [2, 1, 1, 16]})
    inst.close()
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, 2, 32, dynamic=True), "fp32")
    for B, S in ((2, 32), (3, 16), (1, 24)):
        if (B, S) != (2, 32):
            inst.reshape({"input_ids": [B, S], "token_type_ids": [B, S], "attention_bias": [B, 1, 1, S]})
        ids, seg, lens, mask = make_inputs(cfg, B, S, S // 2, S, seed=40 + S)
        inst.set_input("input_ids", ids)
        inst.set_input("token_type_ids", seg)
        inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
        inst.forward()
        got = inst.output("last_hidden").reshape(B * S, -1)
        ref = encoder_ref.encoder(w, cfg, encoder_ref.embed(w, ids, seg, cfg.eps), B, S, mask)
        err = rel_err(got, ref)
        say("  fp32 B=%d S=%d max rel err %.3g" % (B, S, err))
        assert err <= FP32_ASSERT <= FP32_TOL
    inst.close()


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_encoder_int32_mask_input_builds_the_additive_mask_in_the_graph(precision):
    """Inputs as the tokenizer hands them over (ids, segment ids and a 0/1 mask, all NC_INT32): the graph builds the
    additive mask itself (Cast -> Unsqueeze -> Sub -> Mul, the layers an exported BERT carries).  The result is bit for
    bit that of the same weights fed with the additive mask as a float input."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: int32 mask input, " + precision)
    cfg = EncoderConfig(2, 256, 4, 512)
    w = make_weights(cfg, seed=51, bias_std=0.05)
    B, S = 3, 72
    w["pos_emb"] = w["pos_emb"][:S]
    ids, seg, lens, mask = make_inputs(cfg, B, S, 9, S, seed=52)
    outs = []
    for int_mask in (False, True):
        inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S, int_mask=int_mask), precision)
        types = [t for t, _ in inst.layers()]
        inst.set_input("input_ids", ids)
        inst.set_input("token_type_ids", seg)
        if int_mask:
            assert all(t in types for t in ("Cast", "Unsqueeze", "Sub", "Mul")), types
            inst.set_input("input_mask", (mask == 0).astype(np.int32))
        else:
            inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
        for _ in range(4):   # the fourth forward replays the recorded graph
            inst.forward()
        outs.append(inst.output("last_hidden"))
        inst.close()
    assert outs[0].shape == (B, S, cfg.hidden)
    assert np.array_equal(outs[0], outs[1])
    wr = r16w(w) if precision == "fp16" else w
    ref = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids, seg, cfg.eps), B, S, mask)
    err = rel_err(outs[1].reshape(B * S, -1), ref)
    say("  against the checker: max rel err %.3g" % err)
    assert err <= (FP16_TOL if precision == "fp16" else FP32_ASSERT)


@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16"])
def test_mask_made_of_integers_in_one_launch(precision):
    """The layers that make the additive mask out of integers run as one launch in a plain forward and one by one under
    ForwardWithCallback, or where a blob between them is a model output: the answer and the mask are bit for bit the same, for
    every mask that an instance is given in turn and after a reshape."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: mask of integers as a group, " + precision)
    cfg = EncoderConfig(2, 256, 4, 512)
    w = make_weights(cfg, seed=53, bias_std=0.05)
    B, S = 3, 40
    graphs = [tnnmodel.encoder_graph(cfg, w, B, S, int_mask=True, dynamic=True, position_ids=True, extra_outputs=extra)
              for extra in (("attention_bias",), ("attention_bias", "mask_pad"))]
    group, single = (host.RocmInstance.from_graph(g, precision) for g in graphs)
    rng = np.random.default_rng(54)
    for b, n in ((B, S), (1, 56), (2, 33)):
        ids, seg, lens, _ = make_inputs(cfg, b, n, 1, n, seed=b)
        masks = [np.ones((b, n)), np.arange(n)[None, :] < lens[:, None], rng.integers(0, 2, (b, n)), np.zeros((b, n))]
        shapes = {k: [b, n] for k in ("input_ids", "token_type_ids", "input_mask", "position_ids")}
        for inst in (group, single):
            inst.reshape(shapes)
            for name, value in (("input_ids", ids), ("token_type_ids", seg), ("position_ids", np.tile(np.arange(n), (b, 1)))):
                inst.set_input(name, value.astype(np.int32))
        for m in masks:
            got = []
            for inst, run in ((group, "forward"), (group, "callback"), (single, "forward")):
                inst.set_input("input_mask", m.astype(np.int32))
                inst.forward() if run == "forward" else inst.forward_with_callback()
                got.append((inst.output("last_hidden"), inst.output("attention_bias")))
            assert np.isfinite(got[0][0]).all()
            assert np.array_equal(got[0][1].reshape(b, n) == 0, m.astype(bool))
            if precision != "fp32":  # with a callback an fp32 net runs the attention's layers one by one as well
                assert np.array_equal(got[0][0], got[1][0])
            assert np.array_equal(got[0][0], got[2][0])
            assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][1], got[2][1])
    group.close()
    single.close()


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_reading_comprehension_demo_shape(precision):
    """The shape the reference's BERT demo feeds (examples/linux/src/BertReadingComprehension/BertReadingComprehension.cc:
    43, 73 and examples/base/bert_tokenizer.cc:351-355): one sequence of 256 tokens, ids / 0-1 mask / segment ids as
    NC_INT32 Mats of dims [1, 256], BERT-base width.  A padded question + paragraph: 141 valid tokens, segment 1 after
    the first 17."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: demo shape [1, 256], " + precision)
    cfg = EncoderConfig(2, 768, 12, 3072)
    w = make_weights(cfg, seed=91, bias_std=0.05)
    B, S, valid = 1, 256, 141
    w["pos_emb"] = w["pos_emb"][:S]
    rng = np.random.default_rng(92)
    ids = np.zeros((B, S), np.int32)
    ids[0, :valid] = rng.integers(1, cfg.vocab, size=valid)
    seg = np.zeros((B, S), np.int32)
    seg[0, 17:valid] = 1
    m01 = np.zeros((B, S), np.int32)
    m01[0, :valid] = 1
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S, int_mask=True), precision)
    types = [t for t, _ in inst.layers()]
    if precision == "fp16":
        assert types.count("RocmFusedAttention") == cfg.layers, types
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("input_mask", m01)
    for _ in range(4):   # the fourth forward replays the recorded graph
        inst.forward()
    out = inst.output("last_hidden")
    inst.close()
    assert out.shape == (B, S, cfg.hidden)
    mask = ((1 - m01) * -10000.0).astype(np.float32)
    wr = r16w(w) if precision == "fp16" else w
    ref = encoder_ref.encoder(wr, cfg, encoder_ref.embed(wr, ids, seg, cfg.eps), B, S, mask)
    err = rel_err(out.reshape(B * S, -1)[:valid], ref[:valid])
    say("  valid rows against the checker: max rel err %.3g" % err)
    assert err <= (FP16_TOL if precision == "fp16" else FP32_ASSERT)


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_encoder_position_ids_input_third_gather(precision):
    """Exports that keep the position ids a model input look the positions up with a third Gather.  Same result as the
    graph that adds the first S rows of the table; permuted position ids give the permuted table rows."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: position ids as an input (Gather x3), " + precision)
    cfg = EncoderConfig(1, 256, 4, 512)
    w = make_weights(cfg, seed=61, bias_std=0.05)
    B, S = 2, 40
    ids, seg, lens, mask = make_inputs(cfg, B, S, 9, S, seed=62)
    base = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, dict(w, pos_emb=w["pos_emb"][:S]), B, S), precision)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S, position_ids=True), precision)
    types = [t for t, _ in inst.layers()]
    assert types.count("RocmFusedEmbedding") == 1 and "Gather" not in types, types   # the third Gather is folded too
    pos = np.tile(np.arange(S, dtype=np.int32), (B, 1))
    for i in (base, inst):
        i.set_input("input_ids", ids)
        i.set_input("token_type_ids", seg)
        i.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    inst.set_input("position_ids", pos)
    base.forward()
    inst.forward()
    a, b = base.output("last_hidden"), inst.output("last_hidden")
    assert np.array_equal(a, b)
    # other positions: row s of sequence 1 takes table row S-1-s
    pos2 = pos.copy()
    pos2[1] = pos2[1][::-1]
    inst.set_input("position_ids", pos2)
    inst.forward()
    c = inst.output("last_hidden")
    wr = r16w(w) if precision == "fp16" else w
    H = cfg.hidden
    we = orc.gather(wr["word_emb"], ids.reshape(-1))[0].reshape(B, S, H)
    pe = orc.gather(wr["pos_emb"], pos2.reshape(-1))[0].reshape(B, S, H)
    te = orc.gather(wr["type_emb"], seg.reshape(-1))[0].reshape(B, S, H)
    tok = orc.binary("add", orc.binary("add", we, pe), te)
    x0 = orc.layernorm(tok.reshape(B * S, H), wr["emb_ln_g"], wr["emb_ln_b"], cfg.eps)
    ref = encoder_ref.encoder(wr, cfg, x0, B, S, mask)
    err = rel_err(c.reshape(B * S, -1), ref)
    say("  permuted positions against the checker: max rel err %.3g" % err)
    assert err <= (FP16_TOL if precision == "fp16" else FP32_ASSERT)
    assert np.array_equal(c[0], a[0]) and not np.array_equal(c[1], a[1])
    base.close()
    inst.close()


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_encoder_pooler_head(precision):
    """The pooler after the encoder (Gather of the first token with a constant index, Squeeze, dense, Tanh) runs on the
    device and gives tanh(W h[:, 0] + b) of the hidden states the same instance returns."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: pooler head, " + precision)
    cfg = EncoderConfig(1, 256, 4, 512)
    w = make_weights(cfg, seed=71, bias_std=0.05)
    rng = np.random.default_rng(72)
    w["pool_w"] = (rng.standard_normal((cfg.hidden, cfg.hidden)) * 0.05).astype(np.float32)
    w["pool_b"] = (rng.standard_normal(cfg.hidden) * 0.05).astype(np.float32)
    B, S = 3, 24
    w["pos_emb"] = w["pos_emb"][:S]
    ids, seg, lens, mask = make_inputs(cfg, B, S, 5, S, seed=73)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), precision)
    types = [t for t, _ in inst.layers()]
    assert "Tanh" in types and "Squeeze" in types and "Gather" in types, types
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    inst.forward()
    hidden = inst.output("last_hidden")
    pooled = inst.output("pooled")
    inst.close()
    assert pooled.shape == (B, cfg.hidden)
    pw = w["pool_w"].astype(np.float16).astype(np.float32) if precision == "fp16" else w["pool_w"]
    ref = np.tanh(orc.inner_product(np.ascontiguousarray(hidden[:, 0, :]), pw, w["pool_b"]))
    err = rel_err(pooled, ref)
    say("  pooled against tanh(W h0 + b): max rel err %.3g" % err)
    assert err <= (FP16_TOL if precision == "fp16" else 1e-5)


def test_plan_without_device_matches_the_instance():
    """tnn_host_plan (no device context) and a live instance agree on the optimised graph: layer types, blob names and
    every inferred shape."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: plan vs instance")
    cfg = EncoderConfig(2, 256, 4, 512)
    w = make_weights(cfg, seed=81)
    w["pos_emb"] = w["pos_emb"][:40]
    g = tnnmodel.encoder_graph(cfg, w, 2, 40, int_mask=True)
    for precision in ("fp32", "fp16"):
        plan = host.plan(g, precision=precision)
        inst = host.RocmInstance.from_graph(g, precision)
        live = inst.layer_io()
        types = [t for t, _ in inst.layers()]
        inst.close()
        assert [l["type"] for l in plan] == types
        for a, b in zip(plan, live):
            assert {k: a[k] for k in b} == b


def test_int8_mats_in_and_out_with_per_channel_blob_scales():
    """The int8 I/O contract of the blob converter (blob_converter_default.cc:190-193, 347-350, 396-403): an int8 Mat
    (RESERVED_INT8_TEST) is copied as it is into an int8 input blob and out of an int8 output blob; a float Mat goes
    through the blob's scales, one per channel when the blob has that many.  One quantised InnerProduct over
    [2, 8, 5, 5] -> [2, 16] with per-channel input and output blob scales, as the reference's int8 layer test builds
    it; int8 results against the checker bit for bit."""
    host, tnnmodel, *_ = _mods()
    say("host: int8 Mats in and out, per-channel blob scales")
    rng = np.random.default_rng(31)
    dims, N = [2, 8, 5, 5], 16
    K = 8 * 5 * 5
    g = tnnmodel.Graph()
    g.add_input("input0", dims)
    g.add_layer("QuantizedInnerProduct", "fc", ["input0"], ["output0"], [N, 1, 0, 1])
    w = rng.integers(-127, 128, size=(N, K)).astype(np.int8)
    b = rng.integers(-2000, 2000, size=N).astype(np.int32)
    w_scale = rng.uniform(0.001, 0.01, size=N).astype(np.float32)
    s_in = rng.uniform(0.02, 0.05, size=8).astype(np.float32)
    s_out = rng.uniform(0.5, 1.5, size=N).astype(np.float32)
    g.res_inner_product("fc", w, b, quant_scale=w_scale)
    g.res_blob_scale("input0", s_in)
    g.res_blob_scale("output0", s_out)
    g.add_output("output0")
    xq = rng.integers(-128, 128, size=dims).astype(np.int8)
    want, _ = orc.fc_int8(xq.reshape(2, K), w, b, orc.fc_int8_scale(w_scale, s_out, N))
    inst = host.RocmInstance.from_graph(g, "fp16")
    # int8 Mat in, int8 Mat out
    inst.set_input("input0", xq)
    inst.forward()
    got = inst.output_as("output0", np.int8)
    assert got.shape == (2, N) and np.array_equal(got, want)
    # the same int8 output through a float Mat: value * its channel's scale
    assert np.array_equal(inst.output("output0"), want.astype(np.float32) * s_out[None, :])
    # float Mat in: quantised with the input blob's per-channel scales
    xf = (xq.astype(np.float32) * s_in[None, :, None, None]).astype(np.float32)
    inst.set_input("input0", xf)
    inst.forward()
    inv = (1.0 / s_in.astype(np.float64)).astype(np.float32)
    xq2 = orc.float2int8(xf * inv[None, :, None, None])
    want2, _ = orc.fc_int8(xq2.reshape(2, K), w, b, orc.fc_int8_scale(w_scale, s_out, N))
    assert np.array_equal(inst.output_as("output0", np.int8), want2)
    inst.close()


@pytest.mark.parametrize("precision", ["fp16", "fp32"])
def test_instances_come_and_go_without_leaving_memory_behind(precision):
    """A serving process creates, reshapes and destroys instances for as long as it lives: after a few cycles of
    Init + Forward (eager, eager, record, replay) + Reshape + Forward + destroy, neither the device memory in use (blob
    pool, weights, workspace, converter buffers, recorded graphs) nor the process's resident host memory may keep
    growing.  Device memory is read from the driver (hipMemGetInfo through torch), so allocations of this library count
    whoever made them."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: create / reshape / forward / destroy cycles, %s: memory in use" % precision)
    cfg = EncoderConfig(2, 256, 4, 512)
    w = make_weights(cfg, seed=11, bias_std=0.02)
    g = tnnmodel.encoder_graph(cfg, w, 2, 64, dynamic=True)
    proto, model = g.proto(), g.model()

    def resident():
        with open("/proc/self/statm") as f:
            return int(f.read().split()[1]) * 4096

    def cycle():
        inst = host.RocmInstance(proto, model, precision)
        for rep, (b, s) in enumerate([(2, 64), (1, 32), (2, 64)]):
            if rep:
                inst.reshape({"input_ids": [b, s], "token_type_ids": [b, s], "attention_bias": [b, 1, 1, s]})
            ids, seg, lens, mask = make_inputs(cfg, b, s, 10, s, seed=rep)
            inst.set_input("input_ids", ids)
            inst.set_input("token_type_ids", seg)
            inst.set_input("attention_bias", mask.reshape(b, 1, 1, s))
            for _ in range(4):
                inst.forward()
            inst.output("last_hidden")
        inst.close()
        torch.cuda.synchronize()

    def device_in_use():
        free, total = torch.cuda.mem_get_info()
        return total - free

    before = device_in_use()
    held = [host.RocmInstance(proto, model, precision) for _ in range(8)]   # the probe sees what instances hold
    dev_held = device_in_use()
    for inst in held:
        inst.close()
    assert dev_held - before >= 8 << 20, (before, dev_held)
    for _ in range(4):   # the runtime's own pools (streams, kernel arguments, signals) have grown to their size after these
        cycle()
    dev0, host0 = device_in_use(), resident()
    for _ in range(16):
        cycle()
    dev1, host1 = device_in_use(), resident()
    say("  device in use %.1f -> %.1f MiB, host resident %.1f -> %.1f MiB over 16 cycles"
        % (dev0 / 2**20, dev1 / 2**20, host0 / 2**20, host1 / 2**20))
    assert dev1 - dev0 <= 2 << 20, (dev0, dev1)       # the driver hands memory out in 2 MiB pieces
    assert host1 - host0 <= 4 << 20, (host0, host1)   # one instance of this model holds far more than that


def test_an_fp32_net_holds_its_weights_once():
    """The attention groups of an fp32 net and the layers they stand for (which ForwardWithCallback still runs) share one set of
    projection weights on the device; projections without a bias among them."""
    host, tnnmodel, EncoderConfig, make_weights, _ = _mods()
    say("host: device memory of an fp32 net")
    cfg = EncoderConfig(4, 1024, 16, 1024)
    w = make_weights(cfg, seed=11, with_embeddings=False)
    g = tnnmodel.encoder_graph(cfg, w, 1, 32, with_embeddings=False)
    weights = sum(a.nbytes for lw in w["layers"] for a in lw.values())
    host.RocmInstance.from_graph(g, "fp32").close()  # what the runtime keeps for itself
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    inst = host.RocmInstance.from_graph(g, "fp32")
    held = free - torch.cuda.mem_get_info()[0]
    say("  weights %.1f MiB, instance %.1f MiB" % (weights / 2 ** 20, held / 2 ** 20))
    # twice the Q, K and V weights would be half as much again; blobs of 32 tokens are small, and every matrix is whole 2 MiB pieces
    assert weights <= held <= 1.25 * weights
    x = np.random.default_rng(3).standard_normal((1, 32, 1024)).astype(np.float32)
    inst.set_input("hidden", x)
    inst.set_input("attention_bias", np.zeros((1, 1, 1, 32), np.float32))
    inst.forward()
    got = inst.output("last_hidden").copy()
    inst.forward_with_callback(after=lambda name, typ, blobs: None)
    assert rel_err(got, inst.output("last_hidden")) <= 3e-6
    inst.close()


def _bf16_bits(x32):
    """float32 -> bfloat16 bit patterns, round to nearest even (finite values)"""
    u = np.ascontiguousarray(x32, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _bf16_to_f32(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16"])
def test_half_and_bfloat16_mats_in_and_out(precision):
    """RESERVED_FP16_TEST / RESERVED_BFP16_TEST Mats, the host types the engine's layer test feeds half-precision blobs
    with (layer_test.cc:266-275, blob_converter_default.cc:205-208, 323-330).  In: values that the half type holds exactly
    give, fed as a half Mat, the bits they give fed as an fp32 Mat, whatever the blob's type.  Out: the half Mat of an
    output is the fp32 Mat of that output rounded to the half type (to nearest even), exactly."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: half / bfloat16 Mats in and out, blobs %s" % precision)
    cfg = EncoderConfig(1, 256, 4, 512)
    lw = make_weights(cfg, seed=5, bias_std=0.05)["layers"][0]
    B, S, H = 2, 40, 256
    rng = np.random.default_rng(77)
    x = rng.standard_normal((B, S, H)).astype(np.float32)
    mask = np.zeros((B, 1, 1, S), np.float32)
    mask[1, 0, 0, 29:] = -10000.0
    g = tnnmodel.attention_block_graph(lw, B, S, H, 4)
    inst = host.RocmInstance.from_graph(g, precision)

    def run(hidden, bias):
        inst.set_input("hidden", hidden)
        inst.set_input("attention_bias", bias)
        inst.forward()
        return inst.output("y")

    x16 = x.astype(np.float16)
    xb = _bf16_bits(x)
    as_f32_of_half = run(x16.astype(np.float32), mask)
    as_half = run(x16, mask.astype(np.float16))            # -10000 is a half value
    assert np.array_equal(as_half, as_f32_of_half)
    as_f32_of_bf16 = run(_bf16_to_f32(xb), mask)
    as_bf16 = run(xb, mask)
    assert np.array_equal(as_bf16, as_f32_of_bf16)
    assert not np.array_equal(as_bf16, as_half)            # the two roundings of x are different inputs

    y32 = inst.output("y")
    y16 = inst.output_as("y", np.float16)
    yb = inst.output_as("y", np.uint16)
    assert y16.shape == y32.shape and yb.shape == y32.shape
    assert np.array_equal(y16, y32.astype(np.float16))
    assert np.array_equal(yb, _bf16_bits(y32))
    # int32 blobs take no half Mat
    inst.close()
    cfg2 = EncoderConfig(1, 128, 2, 256)
    w2 = make_weights(cfg2, seed=6)
    w2["pos_emb"] = w2["pos_emb"][:16]
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg2, w2, 1, 16), precision)
    with pytest.raises(host.HostError):
        inst.set_input("input_ids", np.zeros((1, 16), np.float16))
    inst.close()


def test_int32_output_blob_read_as_a_float_mat():
    """An int32 blob fetched as an NCHW_FLOAT Mat comes out converted to float (blob_converter_default.cc:213-221), and
    as an NC_INT32 Mat as it is: a Cast to int32 as the model's last layer."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: int32 output blob as float and as int32 Mat")
    g = tnnmodel.Graph()
    g.add_input("x", [2, 3, 5])
    g.add_layer("Cast", "to_int", ["x"], ["xi"], [tnnmodel.DT_INT32])
    g.add_output("xi")
    inst = host.RocmInstance.from_graph(g, "fp32")
    x = (np.random.default_rng(3).standard_normal((2, 3, 5)) * 50).astype(np.float32)
    inst.set_input("x", x)
    inst.forward()
    as_int = inst.output_as("xi", np.int32)
    as_float = inst.output("xi")
    inst.close()
    assert np.array_equal(as_int, x.astype(np.int32))          # Cast truncates toward zero (cpu_cast_layer_acc.cc)
    assert as_float.dtype == np.float32 and np.array_equal(as_float, as_int.astype(np.float32))


def converter_grid():
    """the parameter grid of the engine's BlobConverterTest for NCHW_FLOAT Mats (test/unit_test/blob_converter_test.cc:
    154-172): batch, channel, input size, scale, bias; per-channel values scale * (c + 1), bias * (c + 1) (:287-293)"""
    import itertools
    return list(itertools.product((1, 2), (1, 3, 4, 16), (1, 15, 16), (0.5, 1.0), (0.0, 1.0)))


def converter_round_trip_expected(x, scale, bias, half_blob):
    n, c = x.shape[:2]
    s = np.asarray(scale, np.float32).reshape(1, c, 1, 1)
    b = np.asarray(bias, np.float32).reshape(1, c, 1, 1)
    blob = (x * s + b).astype(np.float32)
    if half_blob:
        blob = blob.astype(np.float16).astype(np.float32)
    return (blob * s + b).astype(np.float32)


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_blob_converter_scale_and_bias_grid(precision):
    """The engine's blob-converter unit test restated for this device's Mat type: an fp32 NCHW Mat goes into the blob with
    per-channel scale and bias and comes back out with them applied again, over the test's whole grid (96 cases).  fp32
    blobs give exactly what fp32 arithmetic gives; half blobs that with one rounding of the blob."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: blob converter with scale and bias, 96 cases, blobs " + precision)
    rng = np.random.default_rng(9)
    worst = 0.0
    for batch, channel, size, scale, bias in converter_grid():
        g = tnnmodel.Graph()
        g.add_input("x", [batch, channel, size, size])
        g.add_layer("GELU", "act", ["x"], ["y"])
        g.add_output("y")
        inst = host.RocmInstance.from_graph(g, precision)
        x = rng.random((batch, channel, size, size), dtype=np.float32)      # InitRandom(0, 1): blob_converter_test.cc:213
        sc = [scale * (c + 1) for c in range(channel)]
        bi = [bias * (c + 1) for c in range(channel)]
        got = inst.input_blob_round_trip("x", x, sc, bi)
        inst.close()
        want = converter_round_trip_expected(x, sc, bi, precision == "fp16")
        if precision == "fp32":
            assert np.array_equal(got, want), (batch, channel, size, scale, bias)
        else:
            assert np.all(np.abs(got - want) <= 1e-6 + 1e-6 * np.abs(want)), (batch, channel, size, scale, bias)
        worst = max(worst, float(np.abs(got - want).max()))
    say("  largest difference to the expected Mat %.3g" % worst)


def _device_to_numpy(ptr, shape, np_dtype):
    """the bytes at a device address as a numpy array (one device-to-device copy into a tensor, then torch's own download)"""
    from tnn_amd import capi
    tdt = {np.dtype(np.float32): torch.float32, np.dtype(np.float16): torch.float16, np.dtype(np.int32): torch.int32,
           np.dtype(np.int8): torch.int8, np.dtype(np.uint16): torch.int16}[np.dtype(np_dtype)]
    t = torch.empty(shape, dtype=tdt, device="cuda")
    torch.cuda.synchronize()
    capi.call("tnn_rocm_memcpy_d2d", t.data_ptr(), ptr, t.numel() * t.element_size(), None)
    torch.cuda.synchronize()
    return t.cpu().numpy().view(np_dtype)


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_mats_in_device_memory(precision):
    """Mats whose memory is on the device (Mat(DEVICE_ROCM, ...), what cuda_blob_converter.cc:62-81, 141-161 does for
    DEVICE_CUDA Mats): token ids, segment ids and mask given as device arrays, the output taken as fp32, half and
    bfloat16 device Mats.  Every result is bit for bit that of the same call with host Mats."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: Mats in device memory, " + precision)
    cfg = EncoderConfig(2, 256, 4, 512)
    w = make_weights(cfg, seed=81, bias_std=0.05)
    B, S = 3, 48
    w["pos_emb"] = w["pos_emb"][:S]
    ids, seg, lens, mask = make_inputs(cfg, B, S, 11, S, seed=82)
    inst = host.RocmInstance.from_graph(tnnmodel.encoder_graph(cfg, w, B, S), precision)
    inst.set_input("input_ids", ids)
    inst.set_input("token_type_ids", seg)
    inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
    inst.forward()
    want32 = inst.output("last_hidden")
    want16 = inst.output_as("last_hidden", np.float16)
    wantb = inst.output_as("last_hidden", np.uint16)

    # other values first, so that the blobs cannot still hold the right ones
    inst.set_input("input_ids", np.zeros_like(ids))
    inst.forward()
    d_ids = torch.from_numpy(ids.astype(np.int32)).cuda()
    d_seg = torch.from_numpy(seg.astype(np.int32)).cuda()
    d_mask = torch.from_numpy(mask.reshape(B, 1, 1, S).astype(np.float32)).cuda()
    torch.cuda.synchronize()
    inst.set_input_device("input_ids", d_ids.data_ptr(), np.int32, [B, S])
    inst.set_input_device("token_type_ids", d_seg.data_ptr(), np.int32, [B, S])
    inst.set_input_device("attention_bias", d_mask.data_ptr(), np.float32, [B, 1, 1, S])
    inst.forward()
    for np_dtype, want in ((np.float32, want32), (np.float16, want16), (np.uint16, wantb)):
        ptr, shape = inst.output_device("last_hidden", np_dtype)
        assert shape == list(want.shape)
        got = _device_to_numpy(ptr, shape, np_dtype)
        assert np.array_equal(got, want), np_dtype
    assert np.array_equal(inst.output("last_hidden"), want32)          # and host Mats after device Mats
    # a half Mat on the device into the float mask input
    d_mask16 = d_mask.half()
    torch.cuda.synchronize()
    inst.set_input_device("attention_bias", d_mask16.data_ptr(), np.float16, [B, 1, 1, S])
    inst.forward()
    assert np.array_equal(inst.output("last_hidden"), want32)          # 0 and -10000 are half values
    with pytest.raises(host.HostError):                                # an int32 Mat needs an int32 blob, on the device too
        inst.set_input_device("attention_bias", d_ids.data_ptr(), np.int32, [B, 1, 1, S])
    inst.close()


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_blob_converter_scale_and_bias_grid_with_device_mats(precision):
    """the converter grid again with the Mats in device memory: scale and bias are applied by two broadcast kernels, and
    the result is bit for bit what the host-Mat form gives"""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: blob converter with scale and bias on device Mats, 96 cases, blobs " + precision)
    rng = np.random.default_rng(19)
    for batch, channel, size, scale, bias in converter_grid():
        g = tnnmodel.Graph()
        g.add_input("x", [batch, channel, size, size])
        g.add_layer("GELU", "act", ["x"], ["y"])
        g.add_output("y")
        inst = host.RocmInstance.from_graph(g, precision)
        x = rng.random((batch, channel, size, size), dtype=np.float32)
        sc = [scale * (c + 1) for c in range(channel)]
        bi = [bias * (c + 1) for c in range(channel)]
        want = inst.input_blob_round_trip("x", x, sc, bi)
        d_in = torch.from_numpy(x).cuda()
        d_out = torch.full_like(d_in, -7.0)
        torch.cuda.synchronize()
        inst.input_blob_round_trip("x", None, sc, bi, device_ptrs=(d_in.data_ptr(), d_out.data_ptr()))
        torch.cuda.synchronize()
        inst.close()
        assert np.array_equal(d_out.cpu().numpy(), want), (batch, channel, size, scale, bias)
        assert np.array_equal(d_in.cpu().numpy(), x)                   # the caller's Mat is left as it was


@pytest.mark.parametrize("np_dtype", [np.float32, np.int32, np.int8, np.float16, np.uint16])
def test_mat_utils_copy_to_the_device_and_back(np_dtype):
    """MatUtils::Copy (mat_utils.cc:73-100) with the device's Mat converter: host Mat -> DEVICE_ROCM Mat -> a second
    DEVICE_ROCM Mat that the copy allocates -> host Mat gives the bytes it was given, for every Mat type of the path"""
    host, *_ = _mods()
    say("host: MatUtils::Copy host -> device -> device -> host, %s" % np.dtype(np_dtype).name)
    rng = np.random.default_rng(4)
    for shape in ((1,), (3, 5), (2, 3, 7, 5), (8, 384, 768)):
        if np.dtype(np_dtype).kind == "f":
            a = (rng.standard_normal(shape) * 100).astype(np_dtype)
        else:
            a = rng.integers(-120, 120, shape).astype(np_dtype)
        assert np.array_equal(host.mat_copy_round_trip(a).view(np.uint8), a.view(np.uint8)), shape


def _grid_weights(cfg, S, seed):
    """encoder weights that are int8 multiples of 2^-9 with the largest magnitude (127 * 2^-9) present in every matrix
    and in every table row: quantising them by max|w| / 127 gives them back exactly"""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    w = make_weights(cfg, seed=seed, bias_std=0.05)
    w["pos_emb"] = w["pos_emb"][:S]
    step = np.float32(2.0 ** -9)

    def snap(a, per_row):
        q = np.clip(np.rint(a / step), -127, 127).astype(np.float32)
        if per_row:
            q[:, 0] = 127.0
        else:
            q.flat[0] = 127.0
        return (q * step).astype(np.float32)

    for key in ("word_emb", "type_emb"):
        w[key] = snap(w[key], True)
    for lw in w["layers"]:
        for key, a in lw.items():
            if a.ndim == 2:
                lw[key] = snap(a, False)
    return w


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_weight_only_int8_model_runs_as_its_dequantised_float_form(precision):
    """Dynamic range quantisation (int8 MatMul weights and embedding tables with fp32 scales in the model file, float
    arithmetic at run time: net_optimizer_dynamic_range_dequant.cc): the model gives bit for bit what the float model
    with the weights scale * int8 gives, through the fused layers."""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: weight-only int8 model against its dequantised float form, " + precision)
    cfg = EncoderConfig(2, 256, 4, 512)
    B, S = 2, 48
    w = _grid_weights(cfg, S, seed=91)
    ids, seg, lens, mask = make_inputs(cfg, B, S, 13, S, seed=92)
    outs = []
    for quantised in (False, True):
        g = tnnmodel.encoder_graph(cfg, w, B, S)
        if quantised:
            deq = g.weight_only_int8()
            assert np.array_equal(deq["emb_word"], w["word_emb"]) and np.array_equal(deq["l0_q_mm"], w["layers"][0]["wq"].T)
        inst = host.RocmInstance.from_graph(g, precision)
        if precision == "fp16":
            assert any(t == "RocmFusedAttention" for t, _ in inst.layers())
        inst.set_input("input_ids", ids)
        inst.set_input("token_type_ids", seg)
        inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
        inst.forward()
        outs.append(inst.output("last_hidden"))
        inst.close()
    assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0.1
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_weight_only_int8_inner_product_form(precision):
    """the InnerProduct spelling of the projections with weight-only int8 weights (DynamicRangeQuantizedInnerProduct: int8
    weight, float bias, one scale): bit for bit the float model with the weights scale * int8"""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: weight-only int8 InnerProduct projections, " + precision)
    cfg = EncoderConfig(1, 256, 4, 512)
    B, S, H = 2, 40, 256
    lw = _grid_weights(cfg, S, seed=95)["layers"][0]
    rng = np.random.default_rng(96)
    x = rng.standard_normal((B * S, H)).astype(np.float32)
    mask = np.zeros((B, 1, 1, S), np.float32)
    mask[0, 0, 0, 31:] = -10000.0
    outs = []
    for quantised in (False, True):
        g = tnnmodel.attention_block_graph(lw, B, S, H, 4, proj="inner_product")
        if quantised:
            deq = g.weight_only_int8()
            assert len(deq) == 4 and "DynamicRangeQuantizedInnerProduct" in g.proto()
        inst = host.RocmInstance.from_graph(g, precision)
        inst.set_input("hidden", x)
        inst.set_input("attention_bias", mask)
        inst.forward()
        outs.append(inst.output("y"))
        inst.close()
    assert np.abs(outs[0]).max() > 0.1 and np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_half_precision_weight_file_runs_as_its_float_form(precision):
    """a model file whose weights, biases, tables and constants are stored as IEEE half gives bit for bit what the fp32 file
    holding the same (half-representable) values gives: the records are widened exactly, ahead of the rewrites"""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: half-precision weight file against the fp32 file of the same values, " + precision)
    cfg = EncoderConfig(2, 256, 4, 512)
    B, S = 2, 48
    w = make_weights(cfg, seed=97, bias_std=0.05)
    w["pos_emb"] = w["pos_emb"][:S]

    def r16(a):
        return a.astype(np.float16).astype(np.float32)
    w = {k: ([{n: r16(a) for n, a in lw.items()} for lw in v] if k == "layers" else r16(v)) for k, v in w.items()}
    ids, seg, lens, mask = make_inputs(cfg, B, S, 13, S, seed=98)
    outs = []
    for half_file in (False, True):
        g = tnnmodel.encoder_graph(cfg, w, B, S)
        if half_file:
            g.half_weights()
        inst = host.RocmInstance.from_graph(g, precision)
        if precision == "fp16":
            types = [t for t, _ in inst.layers()]
            assert "RocmFusedAttention" in types and "RocmFusedEmbedding" in types, types
        inst.set_input("input_ids", ids)
        inst.set_input("token_type_ids", seg)
        inst.set_input("attention_bias", mask.reshape(B, 1, 1, S))
        inst.forward()
        outs.append(inst.output("last_hidden"))
        inst.close()
    assert np.abs(outs[0]).max() > 0.1 and np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_first_version_of_the_file_format_runs_like_the_current_one(precision):
    """an attention block stored in the first version of the file format gives the bits the current format gives"""
    host, tnnmodel, EncoderConfig, make_weights, make_inputs = _mods()
    say("host: first version of the file format, " + precision)
    cfg = EncoderConfig(1, 256, 4, 512)
    lw = make_weights(cfg, seed=5, bias_std=0.05)["layers"][0]
    B, S, H = 2, 40, 256
    x = np.random.default_rng(6).standard_normal((B * S, H)).astype(np.float32)
    mask = np.zeros((B, 1, 1, S), np.float32)
    mask[1, 0, 0, 25:] = -10000.0
    outs = []
    for legacy in (False, True):
        if legacy:
            with tnnmodel.legacy_format():
                g = tnnmodel.attention_block_graph(lw, B, S, H, 4, proj="inner_product")
                proto, model = g.proto(), g.model()
        else:
            g = tnnmodel.attention_block_graph(lw, B, S, H, 4, proj="inner_product")
            proto, model = g.proto(), g.model()
        inst = host.RocmInstance(proto, model, precision)
        inst.set_input("hidden", x)
        inst.set_input("attention_bias", mask)
        inst.forward()
        outs.append(inst.output("y"))
        inst.close()
    assert np.abs(outs[0]).max() > 0.1 and np.array_equal(outs[0], outs[1])
