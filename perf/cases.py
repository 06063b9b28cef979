"""What a user has this framework do, as timed cases: whole forward passes through `Model.predict_dev`, `Model.predict` and
the decode session entry points (`fdx_session_*`), on the architectures that `modelgen` builds.

A case names a path and its sizes.  The paths:

  cnn        a convolutional network on images that lie in device memory
  cnn_host   the same on numpy arrays, copies to and from the GPU included
  encoder    the transformer encoder stack on device memory
  prefill    a prompt through a decode session: last logits and next ids
  generate   a prompt, then greedy tokens one by one with the key / value cache

Models and sessions are loaded once and kept, as a serving program keeps them (weights are those of `modelgen`'s default
seeds); `prepare` makes the inputs and the output buffers.
"""
import collections
import ctypes
import importlib
import math

import numpy as np
import torch

fdx = importlib.import_module("frugally-deep_amd")
modelgen = importlib.import_module("frugally-deep_amd.modelgen")

VOCAB, LAYERS, D_MODEL, MAX_POS = 50257, 12, 768, 1024   # the decoder's sizes
ENC_LAYERS, ENC_D, ENC_FFN = 6, 512, 2048                # the encoder's sizes
CLASSES = 1000


def listed():
    return [
        # one small image: what a control loop or a camera frame costs, all latency and launches
        dict(name="small_cnn_b1", path="cnn", net="small_cnn", size=32, batch=1),
        # many small images at once (predict_multi over a list of samples)
        dict(name="small_cnn_b256", path="cnn", net="small_cnn", size=32, batch=256),
        # one photo through a deep network: interactive classification, few rows in every layer
        dict(name="resnet50_b1", path="cnn", net="resnet50", size=224, batch=1),
        # the benchmark's configuration: throughput of large batches
        dict(name="resnet50_b64", path="cnn", net="resnet50", size=224, batch=64),
        # a caller with host arrays, a modest batch: copies count
        dict(name="resnet50_host_b16", path="cnn_host", net="resnet50", size=224, batch=16),
        # the memory-bound network at its benchmark batch
        dict(name="mobilenet_v2_b128", path="cnn", net="mobilenet_v2", size=224, batch=128),
        # an odd batch of images of an odd size
        dict(name="mobilenet_v2_b7_s161", path="cnn", net="mobilenet_v2", size=161, batch=7),
        # sentence embeddings, the benchmark's batch of full sequences
        dict(name="encoder_b32_t256", path="encoder", seq=256, batch=32),
        # a few short sequences of a ragged length
        dict(name="encoder_b3_t77", path="encoder", seq=77, batch=3),
        # prompts on their way into the cache
        dict(name="prefill_b16_t128", path="prefill", batch=16, prompt=128),
        # serving: a batch of prompts, then tokens
        dict(name="generate_b16_p128_n32", path="generate", batch=16, prompt=128, new=32),
        # one user's prompt of an odd length, then tokens
        dict(name="generate_b1_p37_n24", path="generate", batch=1, prompt=37, new=24),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["small_cnn", "resnet50", "resnet50", "cnn_host", "mobilenet_v2", "mobilenet_v2", "encoder", "encoder",
                       "prefill", "prefill", "generate"])
    if path == "small_cnn":
        return dict(path="cnn", net="small_cnn", size=32, batch=_log_int(rng, 1, 256))
    if path in ("resnet50", "mobilenet_v2"):
        size = rng.choice([128, 160, 192, 224, rng.randint(129, 255)])
        most = int((64 if path == "resnet50" else 128) * min(1.0, (224 / size) ** 2))
        return dict(path="cnn", net=path, size=size, batch=_log_int(rng, 1, most))
    if path == "cnn_host":
        return dict(path="cnn_host", net=rng.choice(["resnet50", "mobilenet_v2"]), size=224, batch=_log_int(rng, 1, 32))
    if path == "encoder":
        seq = _log_int(rng, 16, 512)
        return dict(path="encoder", seq=seq, batch=_log_int(rng, 1, max(1, min(64, 8192 // seq))))
    if path == "prefill":
        prompt = _log_int(rng, 8, 512)
        return dict(path="prefill", batch=_log_int(rng, 1, max(1, min(16, 2048 // prompt))), prompt=prompt)
    return dict(path="generate", batch=_log_int(rng, 1, 16), prompt=_log_int(rng, 8, 128), new=rng.randint(8, 32))


# ---------------------------------------------------------------- models and sessions, loaded once

class _Kept:
    """The last few objects made, by their description; an older one lives on while a state uses it."""

    def __init__(self, most):
        self.most, self.items = most, collections.OrderedDict()

    def get(self, key, make):
        if key not in self.items:
            while len(self.items) >= self.most:
                self.items.popitem(last=False)
            self.items[key] = make()
        self.items.move_to_end(key)
        return self.items[key]


_models, _sessions, _facts = _Kept(4), _Kept(3), {}


def _spec(case):
    if case["path"] in ("cnn", "cnn_host"):
        if case["net"] == "small_cnn":
            return modelgen.small_cnn()
        spec = getattr(modelgen, case["net"])(input_size=case["size"])
        if case["net"] == "resnet50":   # random weights without trained BatchNormalization: logits of 600; these are of about 3
            spec["trainable_params"]["predictions"]["weights"] *= np.float32(1 / 200)
        return spec
    if case["path"] == "encoder":
        return modelgen.encoder(layers=ENC_LAYERS, seq=case["seq"], d_model=ENC_D, ffn=ENC_FFN)
    return modelgen.gpt2(layers=LAYERS, d_model=D_MODEL, vocab=VOCAB, max_pos=MAX_POS)


def _model_key(case):
    if case["path"] in ("cnn", "cnn_host"):
        return (case["net"], case["size"])
    return ("encoder", case["seq"]) if case["path"] == "encoder" else ("gpt2",)


def _model(case):
    return _models.get(_model_key(case), lambda: fdx.Model(modelgen.dumps(_spec(case)), verify=False))


class _Session:
    """A session with the model that it reads its weights from."""

    def __init__(self, model, batch, max_len):
        self.model = model
        self.handle = fdx.Session(model, batch, max_len)


def _session(case):
    model = _model(case)
    max_len = case["prompt"] + case.get("new", 0)
    return _sessions.get((case["batch"], max_len), lambda: _Session(model, case["batch"], max_len))


class _Buf:
    """A torch tensor's memory in the form that the framework's calls take."""

    def __init__(self, t):
        self.tensor, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _out(*shape):
    return _Buf(torch.empty(shape, dtype=torch.float32, device="cuda"))


# ---------------------------------------------------------------- one pass

def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    path, batch = case["path"], case["batch"]
    st = dict(path=path, batch=batch)
    if path in ("cnn", "cnn_host"):
        shape = (case["size"], case["size"], 3)
        # pixels in [0, 1]: patches of colour of each image's own, and noise
        coarse = torch.rand((batch, 3, 8, 8), generator=gen, device="cuda")
        x = torch.nn.functional.interpolate(coarse, size=shape[:2], mode="bilinear").permute(0, 2, 3, 1)
        x = (0.9 * x + 0.1 * torch.rand((batch,) + shape, generator=gen, device="cuda")).contiguous()
        if case["net"] == "small_cnn":
            x = 2 * x - 1                                                # this network takes [-1, 1]
        st.update(model=_model(case), shapes=[shape])
        if path == "cnn_host":
            st.update(x=x.cpu().numpy())
        else:
            st.update(inputs=[_Buf(x)], outputs=[_out(batch, *st["model"].output_shapes[0])])
    elif path == "encoder":
        shape = (case["seq"], ENC_D)
        x = torch.randn((batch,) + shape, generator=gen, device="cuda")
        st.update(model=_model(case), shapes=[shape], inputs=[_Buf(x)], outputs=[_out(batch, *shape)])
    else:
        ids = torch.randint(0, VOCAB, (batch, case["prompt"]), generator=gen, device="cuda").float()
        st.update(session=_session(case), ids=_Buf(ids), prompt=case["prompt"], new=case.get("new", 0),
                  logits=_out(batch, VOCAB), first=_out(batch))
        if path == "generate":
            st.update(tokens=_out(case["new"], batch))
    torch.cuda.synchronize()   # the framework works on a stream of its own
    return st


def run(state):
    path = state["path"]
    if path == "cnn_host":
        return state["model"].predict([state["x"]])[0]
    if path in ("cnn", "encoder"):
        state["model"].predict_dev(state["batch"], state["inputs"], state["shapes"], state["outputs"])
        return state["outputs"][0].tensor
    s = state["session"].handle
    s.reset()
    if path == "prefill":
        fdx.check(fdx.lib.fdx_session_prefill(s._h, fdx._dp(state["ids"]), state["prompt"], fdx._dp(state["logits"]), fdx._dp(state["first"])))
        return dict(logits=state["logits"].tensor, next_ids=state["first"].tensor)
    fdx.check(fdx.lib.fdx_session_prefill(s._h, fdx._dp(state["ids"]), state["prompt"], None, fdx._dp(state["first"])))
    fdx.check(fdx.lib.fdx_session_decode_greedy(s._h, fdx._dp(state["first"]), state["new"], fdx._dp(state["tokens"]), fdx._dp(state["logits"])))
    return dict(first=state["first"].tensor, tokens=state["tokens"].tensor, last_logits=state["logits"].tensor)


# ---------------------------------------------------------------- what a pass cannot do without

def _cnn_facts(case):
    """(multiply-add operations of one sample, parameters) of a network, from its layer list."""
    key = _model_key(case)
    if key not in _facts:
        spec = _spec(case)
        flops = modelgen.model_flops(spec)
        params = sum(v.size for p in spec["trainable_params"].values() for v in p.values() if isinstance(v, np.ndarray))
        _facts[key] = (flops, params)
    return _facts[key]


def work(case):
    path, b = case["path"], case["batch"]
    if path in ("cnn", "cnn_host"):
        flops, params = _cnn_facts(case)
        classes = 10 if case["net"] == "small_cnn" else CLASSES
        return {"bytes": 4 * (params + b * (3 * case["size"] ** 2 + classes)), "flops": b * flops}
    if path == "encoder":
        t, d = case["seq"], ENC_D
        params = ENC_LAYERS * (4 * d * d + 2 * d * ENC_FFN)
        return {"bytes": 4 * (params + 2 * b * t * d), "flops": 2 * b * t * params + ENC_LAYERS * 4 * b * t * t * d}
    t, n = case["prompt"], case.get("new", 0)
    block, head = LAYERS * 12 * D_MODEL * D_MODEL, VOCAB * D_MODEL
    # prompt: every position through the blocks (query t sees t + 1 keys), the head on the last one; its keys and values stay
    flops = 2 * b * (t * block + head) + LAYERS * 4 * b * D_MODEL * t * (t + 1) / 2
    nbytes = 4 * (block + head + b * VOCAB + 2 * LAYERS * b * t * D_MODEL)
    for i in range(n):   # a token: all weights again, the cache so far, the logits
        flops += 2 * b * (block + head) + LAYERS * 4 * b * D_MODEL * (t + i + 1)
        nbytes += 4 * (block + head + 2 * LAYERS * b * (t + i + 1) * D_MODEL + b * VOCAB)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # four times what the outputs move by when the sums take another order (other tiles, K ranges, direct for Winograd form):
    # measured 1.1e-7 small network, 4.5e-6 the deep ones (2-norm, on probabilities), 5.4e-7 encoder, 1.8e-6 decoder logits;
    # largest single value 5e-7, 1.6e-5, 3e-6, 8.7e-6.  Token ids: whole numbers in float buffers, the same in all of these.
    if case["path"] in ("cnn", "cnn_host"):
        return {"rel": 1e-6, "max": 4e-6} if case["net"] == "small_cnn" else {"rel": 2e-5, "max": 8e-5}
    return {"rel": 2.5e-6, "max": 1.5e-5} if case["path"] == "encoder" else {"rel": 8e-6, "max": 4e-5}
