"""The workloads this library's speed is judged by: what a program that speaks text through it has it do.

Every case goes through the package's public classes (the C ABI underneath) on the random-init
Qwen3-TTS-0.6B weights the benchmark uses: 28 talker layers, 5 code-predictor layers, f16 weights
N(0, 0.02), norms 1, biases 0; the codec decoder and the speaker encoder with the package's own
fan-in-scaled initialisation. A program loads its model once, so the weights are the same for every
case and seed; prompts, rows, caches, codes and audio come from the seed.

`exact` restates each path in plain torch in 64 bits, with the points at which the model's state is
stored in f16 (the K/V cache) and the f32 rotary angles kept, since they are part of what is computed.
"""
import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "navi-tts_amd"))
from navi_amd import abi, blob  # noqa: E402

H, QD, KVD, FF, HD, NQ, NKV = 1024, 2048, 1024, 3072, 128, 16, 8
TALKER_LAYERS, CP_LAYERS, GROUPS, TALKER_VOCAB, CP_VOCAB, EOS = 28, 5, 16, 3072, 2048, 2050
LAYER_WEIGHTS = H * (QD + 2 * KVD) + QD * H + 3 * H * FF
SAMPLES_PER_FRAME = 1920
MAX_PROMPT, MAX_POS, MAX_STREAMS, MAX_SECONDS = 1024, 2048, 64, 30.0


def listed():
    return [
        # One frame in the middle of an utterance: the talker step, 15 code-predictor steps and the
        # sampling, at the benchmark's context and the server's default sampling.
        {"name": "frame_ctx256", "kind": "frame", "n_past": 256},
        # One frame near the end of a long utterance (the cache holds 2048 positions).
        {"name": "frame_ctx1500", "kind": "frame", "n_past": 1500},
        # The frames of the first audio batch: the on-device loop from the prefill's hidden and logits,
        # greedy (the option whose codes are compared bit for bit).
        {"name": "loop4_ctx130", "kind": "loop", "n_past": 130, "frames": 4},
        # A request's start with a short text (32 ids): the prompt rows are built and prefilled.
        {"name": "prompt_32ids", "kind": "prompt", "ids": 32},
        # A text of 128 ids prefilled whole (130 rows), and a long one near the prompt limit.
        {"name": "prefill_130", "kind": "prefill", "rows": 130},
        {"name": "prefill_1001", "kind": "prefill", "rows": 1001},
        # The vocoder: the first batch of a streamed utterance (time to first audio), a streamed
        # utterance in the server's batches (4, then 16 at a time), and one 240-frame block.
        {"name": "vocoder_first4", "kind": "vocoder", "frames": 4, "first": 4, "batch": 16},
        {"name": "vocoder_stream52", "kind": "vocoder", "frames": 52, "first": 4, "batch": 16},
        {"name": "vocoder_block240", "kind": "vocoder", "frames": 240, "first": 240, "batch": 240},
        # A server's batched decode: one step of 32 full streams, and of a few ragged young ones.
        {"name": "streams32_ctx1024", "kind": "streams", "streams": 32, "ctx": 1024, "ragged": False},
        {"name": "streams7_ragged", "kind": "streams", "streams": 7, "ctx": 300, "ragged": True},
        # A voice clone from ten seconds of audio.
        {"name": "speaker_10s", "kind": "speaker", "samples": 240000},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["frame", "loop", "prompt", "prefill", "prefill", "vocoder", "block", "streams", "streams", "speaker"])
    if kind == "frame":
        return {"kind": "frame", "n_past": _log_int(rng, 1, 1800)}
    if kind == "loop":
        return {"kind": "loop", "n_past": _log_int(rng, 8, 1000), "frames": rng.randint(2, 5)}
    if kind == "prompt":
        return {"kind": "prompt", "ids": _log_int(rng, 9, 400)}
    if kind == "prefill":
        return {"kind": "prefill", "rows": _log_int(rng, 1, 1000)}
    if kind == "vocoder":
        return {"kind": "vocoder", "frames": _log_int(rng, 1, 80), "first": rng.randint(1, 8), "batch": 16}
    if kind == "block":
        n = _log_int(rng, 17, 239)
        return {"kind": "vocoder", "frames": n, "first": n, "batch": 240}
    if kind == "streams":
        n = _log_int(rng, 1, 48)
        return {"kind": "streams", "streams": n, "ctx": _log_int(rng, 4, min(1600, 32 * 1024 // n)), "ragged": rng.random() < 0.5}
    return {"kind": "speaker", "samples": _log_int(rng, 12000, 480000)}


# ---- the model and the handles a program keeps ----------------------------------------------

class _Weights:
    """Device tensors by name, as the package's create() calls take them (`kv` and `refs`)."""

    def __init__(self, parts, seed):
        self.kv = blob.qwen3tts_0p6b_kv()
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.t, self._specs = {}, blob.tensor_table(self.kv, parts)
        for s in self._specs:
            kind, val = s.init
            t = (torch.full(s.shape, val, device="cuda") if kind == "const" else
                 torch.randn(s.shape, generator=g, device="cuda").mul_(float(val)))
            self.t[s.name] = t.half() if s.dtype == blob.DT_F16 else t.float()

    def refs(self):
        arr, keep = (abi.TensorRef * len(self._specs))(), []
        for r, s in zip(arr, self._specs):
            keep.append(s.name.encode())
            r.name, r.ptr, r.dtype, r.ndim = keep[-1], self.t[s.name].data_ptr(), s.dtype, len(s.shape)
            for k, d in enumerate(s.shape):
                r.dims[k] = d
        return arr, keep


_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
        torch.cuda.synchronize()
    return _kept[key]


def _weights(part):
    return _keep("weights " + part, lambda: _Weights(("talker", "cp") if part == "talker" else (part,),
                                                     {"talker": 1, "codec": 2, "speaker": 3}[part]))


def _handle(name):
    def make():
        abi.device_open()
        part = "codec" if name.startswith("vocoder") else "speaker" if name == "speaker" else "talker"
        w = _weights(part)
        torch.cuda.synchronize()
        if name == "frame":
            h = abi.Frame(w)
            h.set_taps(True)               # the logits beside the codes
            return h
        if name == "talker":
            return abi.Talker(w, MAX_PROMPT, MAX_POS)
        if name == "streams":
            return abi.Streams(w, MAX_STREAMS, MAX_POS)
        if name == "speaker":
            return abi.Speaker(w, MAX_SECONDS)
        return abi.Vocoder(w, int(name.split()[1]))
    return _keep("handle " + name, make)


class _Span:
    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "strides": None,
                                         "version": 2}


def _view(ptr, shape, typestr="<f4"):
    """A device buffer of the library as a tensor."""
    return torch.as_tensor(_Span(ptr, shape, typestr), device="cuda")


class _Kv:
    """A stream's K/V cache as the view the library takes: the rows that tensors k and v
    [layer][position][kv_dim] hold from position `first` on."""

    def __init__(self, k, v, first, rows):
        self.k, self.v, self.n_used = k[:, first:], v[:, first:], rows
        p = [(ctypes.c_void_p * TALKER_LAYERS)(*[c[i].data_ptr() for i in range(TALKER_LAYERS)]) for c in (self.k, self.v)]
        self._p = p
        self.view = abi.KvView(TALKER_LAYERS, self.k.shape[1], KVD, *[ctypes.cast(x, ctypes.POINTER(ctypes.c_void_p)) for x in p])


def _cache(g, streams, positions):
    """The caches' tensors [stream][layer][position][kv_dim], from N(0, 1)."""
    return [torch.stack([torch.randn(TALKER_LAYERS, positions, KVD, generator=g, device="cuda").half() for _ in range(streams)])
            for _ in "kv"]


def _set(dst, src):
    """Device rows into a buffer that the library or the program reads its next call's rows from."""
    if abi.lib().navi_mem_d2d(dst, src.data_ptr(), src.numel() * src.element_size()) != abi.NAVI_OK:
        raise RuntimeError("navi_mem_d2d failed")


# ---- inputs -----------------------------------------------------------------------------------

def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _inputs(case, seed):
    """What of the state exact() needs too: from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    kind, s = case["kind"], {"kind": case["kind"], "case": dict(case)}
    s["seed"], s["g"] = int(rng.integers(1, 1 << 40)), g
    if kind in ("frame", "loop"):
        n, frames = case["n_past"], case.get("frames", 1)
        k, v = _cache(g, 1, n + frames)
        s["kv"] = _Kv(k[0], v[0], 0, n)
        s["trailing"] = _normal(g, frames + 1, H)                        # the text rows, then tts_pad
        if kind == "frame":
            s["step_in"] = _normal(g, H)
        else:                                                            # what a prefill leaves
            s["hidden"] = _normal(g, H)
            s["logits"] = 0.64 * _normal(g, TALKER_VOCAB)
    elif kind == "prompt":
        kv = blob.qwen3tts_0p6b_kv()
        im, an = kv["text.im_start_id"], kv["text.assistant_id"]
        text = rng.integers(0, 151643, case["ids"] - 8).tolist()
        s["ids"] = np.array([im, an, 198] + text + [kv["text.im_end_id"], 198, im, an, 198], np.int32)
        s["speaker"] = rng.standard_normal(H).astype(np.float32)
    elif kind == "prefill":
        s["rows"] = _normal(g, case["rows"], H)
    elif kind == "vocoder":
        s["codes"] = rng.integers(0, CP_VOCAB, (case["frames"], GROUPS)).astype(np.int32)
    elif kind == "streams":
        n, ctx = case["streams"], case["ctx"]
        s["n_past"] = [int(x) for x in (rng.integers(1, ctx + 1, n) if case["ragged"] else np.full(n, ctx))]
        s["n_past"][-1] = ctx
        s["cache"] = k, v = _cache(g, n, ctx + 1)          # each stream's new row is the last one
        s["kvs"] = [_Kv(k[i], v[i], ctx - p, p) for i, p in enumerate(s["n_past"])]
        s["step_in"], s["trailing"] = _normal(g, n, H), _normal(g, n, H)
        s["seeds"] = [s["seed"] + i for i in range(n)]
    else:                                                                # speech-like level, wide band
        s["wav"] = (0.1 * rng.standard_normal(case["samples"])).astype(np.float32)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    # the server's: top-k 50, T 0.9, penalty 1.05; the loop greedy
    s["sampling"] = abi.Sampling.greedy() if kind == "loop" else abi.Sampling.make()
    if kind in ("frame", "loop"):
        f = s["frame"] = _handle("frame")
        L, kv, n = abi.lib(), s["kv"], case["n_past"]
        new = slice(n, n + case.get("frames", 1) - (kind == "loop"))
        s["out"] = {"hidden": _view(L.navi_frame_tap_hidden(f.h), (H,)), "logits": _view(L.navi_frame_tap_logits(f.h), (TALKER_VOCAB,)),
                    "cp_logits": _view(L.navi_frame_tap_cp_logits(f.h), (GROUPS - 1, CP_VOCAB)), "step": _view(f.d_step_out, (H,)),
                    "k": kv.k[:, new], "v": kv.v[:, new]}
    elif kind in ("prompt", "prefill"):
        t = s["talker"] = _handle("talker")
        n = case["rows"] if kind == "prefill" else 10
        s["out"] = {"hidden": _view(t.d_hidden, (H,)), "logits": _view(t.d_logits, (TALKER_VOCAB,)),
                    "k": [_view(p, (n, KVD), "<f2") for p in t.kv.k], "v": [_view(p, (n, KVD), "<f2") for p in t.kv.v]}
    elif kind == "vocoder":
        s["vocoder"] = _handle("vocoder %d" % case["batch"])
        n, first, batch = case["frames"], case["first"], case["batch"]
        cuts = [0] + list(range(first, n, batch)) + [n] if first < n else [0, n]
        s["batches"] = [s["codes"][a:b] for a, b in zip(cuts, cuts[1:])]
    elif kind == "streams":
        s["streams"] = _handle("streams")
        s["text"] = _keep("streams' trailing rows", lambda: torch.empty(MAX_STREAMS, H, device="cuda"))
        s["frame_index"] = [3] * case["streams"]
        n = case["streams"]
        s["out"] = {"step": _view(s["streams"].d_step_out, (n, H)), "k": s["cache"][0][:, :, -1], "v": s["cache"][1][:, :, -1]}
    else:
        s["encoder"] = _handle("speaker")
    torch.cuda.synchronize()
    return s


# ---- one pass -----------------------------------------------------------------------------------

def run(s):
    return globals()["_run_" + s["kind"]](s)


def _run_frame(s):
    f = s["frame"]
    f.reset()
    _set(f.d_step_out, s["step_in"])
    r = f.run(s["kv"], s["case"]["n_past"], s["trailing"].data_ptr(), s["sampling"], s["seed"], 3)
    if not r.ok:
        raise RuntimeError(r.error.decode())
    return {"codes": np.array(list(r.codes)), **s["out"]}


def _run_loop(s):
    f, c, t = s["frame"], s["case"], s["trailing"]
    f.reset()
    codes, _, _ = f.run_many(s["kv"], c["n_past"] - 1, t.data_ptr(), c["frames"], t[c["frames"]].data_ptr(), s["sampling"], s["seed"],
                             0, c["frames"], skip_first=True, d_hidden=s["hidden"].data_ptr(), d_logits=s["logits"].data_ptr())
    return {"codes": codes, **s["out"]}


def _run_prompt(s):
    t = s["talker"]
    p = t.build_prompt(s["ids"], "english", s["speaker"])
    t.prefill(p.prefill, p.n_prefill)
    if "trailing" not in s["out"]:                 # the talker's own rows: the same buffers on every call
        s["out"]["trailing"] = _view(p.trailing, (p.n_trailing, H))
        s["out"]["tts_pad"] = _view(p.tts_pad, (H,))
    return s["out"]


def _run_prefill(s):
    s["talker"].prefill(s["rows"].data_ptr(), s["case"]["rows"])
    return s["out"]


def _run_vocoder(s):
    v = s["vocoder"]
    v.reset()
    return [v.decode(b) for b in s["batches"]]


def _run_streams(s):
    h = s["streams"]
    h.reset()
    _set(h.d_step_out, s["step_in"])
    _set(s["text"].data_ptr(), s["trailing"])
    codes = h.run(s["kvs"], s["n_past"], s["text"].data_ptr(), s["sampling"], s["seeds"], s["frame_index"])
    return {"codes": codes, **s["out"]}


def _run_speaker(s):
    return s["encoder"].embed(s["wav"])


# ---- what a pass cannot do without ----------------------------------------------------------------

def _layer_flops(rows, keys):
    """Multiply-adds x 2 of one decoder layer over `rows` rows that see `keys` keys in all."""
    return 2.0 * rows * LAYER_WEIGHTS + 4.0 * keys * QD


def _frame_work(streams, keys):
    """Bytes and flops of one frame of `streams` streams that see `keys` cached keys in all. The code
    predictor's 5 layers have to be read for each of its 15 dependent passes."""
    cp_pass = CP_LAYERS * LAYER_WEIGHTS
    talker = TALKER_LAYERS * LAYER_WEIGHTS + TALKER_VOCAB * H
    heads = (GROUPS - 1) * CP_VOCAB * H
    b = 2.0 * (talker + 15 * cp_pass + heads) + 4.0 * KVD * TALKER_LAYERS * (keys + streams)
    f = streams * 2.0 * (talker + GROUPS * cp_pass + heads) + TALKER_LAYERS * 4.0 * QD * (keys + streams)
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "frame":
        b, f = _frame_work(1, case["n_past"])
    elif kind == "loop":
        b = f = 0.0
        talker = 2.0 * (TALKER_LAYERS * LAYER_WEIGHTS + TALKER_VOCAB * H)
        for i in range(case["frames"]):
            x = _frame_work(1, case["n_past"] - 1 + i)
            # the first frame's talker step is the prefill's
            b, f = b + x[0] - (talker if i == 0 else 0.0), f + x[1] - (talker if i == 0 else 0.0)
    elif kind in ("prompt", "prefill"):
        n = case["rows"] if kind == "prefill" else 10
        b = 2.0 * (TALKER_LAYERS * LAYER_WEIGHTS + TALKER_VOCAB * H) + 4.0 * n * H + 4.0 * n * KVD * TALKER_LAYERS
        f = TALKER_LAYERS * _layer_flops(n, n * (n + 1) / 2) + 2.0 * TALKER_VOCAB * H
        if kind == "prompt":
            m = case["ids"] - 2                                          # header, text, bos, eos and pad rows
            b, f = b + 2.0 * (2048 * 2048 + 2048 * H) + 4.0 * m * 2048, f + 2.0 * m * (2048 * 2048 + 2048 * H)
    elif kind == "vocoder":
        per, weights = _codec_macs()
        calls = len(range(case["first"], case["frames"], case["batch"])) + 1 if case["first"] < case["frames"] else 1
        b = 2.0 * weights * calls + case["frames"] * (4.0 * SAMPLES_PER_FRAME + 4 * GROUPS)
        f = 2.0 * per * case["frames"]
    elif kind == "streams":
        n, mean = case["streams"], case["ctx"] if not case["ragged"] else (case["ctx"] + 1) / 2
        b, f = _frame_work(n, int(n * mean))
    else:
        frames = case["samples"] // 256
        conv = 512 * 128 * 5 + 3 * (2 * 512 * 512 + 7 * 64 * 64 * 3) + 1536 * 1536 + 128 * 1536 + 1536 * 128
        b = 4.0 * case["samples"] + 2.0 * (conv + 3 * 2 * 512 * 128 + 2 * 128 * 1536 + 1024 * 3072) + 4.0 * H
        f = 2.0 * conv * frames
    return {"bytes": b, "flops": f}


def _codec_macs():
    """(multiply-adds per frame, weights) of the codec decoder, from the shapes of its tensors."""
    d, xl = 1536, 512 * 1024 * 3 + 1024 * 512 + 3 * 512 * 1024
    macs = 512 * 256 * 2 + 1024 * 512 * 3 + 512 * 1024 + 8 * xl + 1024 * 512
    weights, rate = macs, 1
    for r in (2, 2):
        macs += rate * r * 1024 * 1024
        rate *= r
        macs += rate * (7 * 1024 + 2 * 4096 * 1024)
        weights += r * 1024 * 1024 + 7 * 1024 + 2 * 4096 * 1024
    macs, weights = macs + rate * d * 1024 * 7, weights + d * 1024 * 7
    for r in (8, 5, 4, 3):
        macs += rate * 2 * r * d * (d // 2)
        weights += 2 * r * d * (d // 2)
        rate, d = rate * r, d // 2
        macs += rate * 3 * 8 * d * d
        weights += 3 * 8 * d * d
    return macs + rate * d * 7, weights + d * 7


def tolerance(case):
    """About four times the distance from `exact` that the first version of these cases measured."""
    if case["kind"] in ("vocoder", "speaker"):     # f32 sums throughout: 1.2e-6 and 2.3e-7
        return {"rel": 5e-6, "max": 2e-4} if case["kind"] == "vocoder" else {"rel": 1e-6, "max": 1e-5}
    # The K/V rows are stored in f16: sums in another order round some of them the other way, and that
    # travels on through the layers. 5e-5 to 3.5e-4 after a prefill's 28 layers, the fewer the rows the
    # more; up to 1.2e-4 in a frame. `differ`: a draw or an argmax that falls to a neighbour at a tie.
    return {"rel": 1.2e-3, "max": 1e-2, "differ": 0.01} if case["kind"] in ("prompt", "prefill") else \
        {"rel": 5e-4, "max": 5e-3, "differ": 0.01}


# ---- the same in 64 bits -------------------------------------------------------------------------

def exact(case, seed):
    with torch.no_grad():
        s = _inputs(case, seed)
        out = globals()["_exact_" + case["kind"]](case, s)
        torch.cuda.synchronize()
        return out


def _cached(part, name):
    t = _weights(part).t[name]
    return _keep("64 " + name, lambda: t.double()) if t.numel() < (1 << 24) else t.double()


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rotate(x, pos, theta):
    """x [..., rows, heads, dim]: rotate-half, the angle an f32 product as the model has it."""
    d = x.shape[-1]
    inv = torch.from_numpy((1.0 / theta ** (np.arange(0, d, 2, dtype=np.float64) / d)).astype(np.float32)).cuda()
    a = (pos.float()[..., None] * inv).double()[..., None, :]
    c, s, x0, x1 = a.cos(), a.sin(), x[..., : d // 2], x[..., d // 2:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


def _layer(prefix, x, k, v, pos):
    """One decoder layer over rows x [n][H] at consecutive positions pos.., with the f16 cache rows k, v
    of the positions before them. Returns the rows and the cache rows with theirs appended."""
    def w(name):
        return _cached("talker", prefix + name + ".weight")
    n = x.shape[0]
    at = torch.arange(pos, pos + n, device="cuda")
    y = _rms(x, w("input_layernorm"))
    q = _rotate(_rms((y @ w("self_attn.q_proj").T).view(n, NQ, HD), w("self_attn.q_norm")), at, 1e6)
    kn = _rotate(_rms((y @ w("self_attn.k_proj").T).view(n, NKV, HD), w("self_attn.k_norm")), at, 1e6)
    k = torch.cat([k, kn.reshape(n, KVD).half()])
    v = torch.cat([v, (y @ w("self_attn.v_proj").T).half()])
    kk = k.double().view(-1, NKV, 1, HD).expand(-1, NKV, NQ // NKV, HD).reshape(-1, NQ, HD).permute(1, 2, 0).contiguous()
    vv = v.double().view(-1, NKV, 1, HD).expand(-1, NKV, NQ // NKV, HD).reshape(-1, NQ, HD).permute(1, 0, 2).contiguous()
    a = torch.bmm(q.permute(1, 0, 2).contiguous(), kk) / math.sqrt(HD)
    a.masked_fill_(torch.arange(a.shape[2], device="cuda")[None, None, :] > at[None, :, None], float("-inf"))
    a = torch.bmm(torch.softmax(a, -1), vv).permute(1, 0, 2).reshape(n, QD)
    x = x + a @ w("self_attn.o_proj").T
    y = _rms(x, w("post_attention_layernorm"))
    return x + (torch.nn.functional.silu(y @ w("mlp.gate_proj").T) * (y @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T, k, v


def _talker(x, kv, pos):
    """The talker over rows x; kv: per layer the (k, v) rows before them. (hidden, logits) of the last row."""
    new = []
    for i in range(TALKER_LAYERS):
        x, k, v = _layer("talker.model.layers.%d." % i, x, *kv[i], pos)
        new.append((k, v))
    h = _rms(x[-1], _cached("talker", "talker.model.norm.weight"))
    return h, _cached("talker", "talker.codec_head.weight") @ h, new


def _mix(x):
    m = (1 << 64) - 1
    x = (x + 0x9E3779B97F4A7C15) & m
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & m
    return x ^ (x >> 31)


def _uniform(seed):
    """The model's draw: the fourth output of a PCG32 stream, its top 24 bits."""
    m = (1 << 64) - 1
    st = (seed * 0x9E3779B97F4A7C15 + 0xBF58476D1CE4E5B9 + 1) & m
    for _ in range(3):
        st = (st * 6364136223846793005 + 1442695040888963407) & m
    xs, rot = (((st >> 18) ^ st) >> 27) & 0xFFFFFFFF, st >> 59
    return ((((xs >> rot) | (xs << (-rot & 31))) & 0xFFFFFFFF) >> 8) / 16777216.0


def _pick(v, seed):
    """Top-k 50 at temperature 0.9: the first index whose running sum reaches the draw."""
    v = v / 0.9
    p = torch.where(v >= torch.topk(v, 50).values[-1], torch.exp(v - v.max()), torch.zeros_like(v))
    i = int(torch.searchsorted(torch.cumsum(p, 0) / p.sum(), _uniform(seed)))
    return min(i, v.numel() - 1)


def _frame(hidden, logits, trailing, seed, index, seen, pick=_pick):
    """codes, cp logits and the next step input of one frame from the talker's hidden and logits."""
    m = (1 << 64) - 1
    ts = _mix(seed ^ ((index * 0xA24BAED4963EE407) & m))
    cs = _mix(ts ^ 0x9FB21C651E98DF25)
    v = logits.clone()
    for c in seen:
        v[c] = v[c] / 1.05 if v[c] > 0 else v[c] * 1.05
    keep = v[EOS].clone()
    v[TALKER_VOCAB - 1024:] = float("-inf")
    if index >= 2:
        v[EOS] = keep
    codes, cp = [pick(v, ts)], []
    seen |= {codes[0]} - {EOS}
    emb = [_weights("talker").t["talker.model.codec_embedding.weight"]] + \
        [_weights("talker").t["talker.code_predictor.model.codec_embedding.%d.weight" % i] for i in range(GROUPS - 1)]
    none = torch.empty(0, KVD, dtype=torch.float16, device="cuda")
    kv, x = [(none, none)] * CP_LAYERS, torch.stack([hidden, emb[0][codes[0]].double()])
    for pos in range(1, GROUPS):
        if pos > 1:
            x = emb[pos - 1][codes[-1]].double()[None]
        for i in range(CP_LAYERS):
            x, k, v = _layer("talker.code_predictor.model.layers.%d." % i, x, *kv[i], 0 if pos == 1 else pos)
            kv[i] = (k, v)
        h = _rms(x[-1], _cached("talker", "talker.code_predictor.model.norm.weight"))
        cp.append(_cached("talker", "talker.code_predictor.lm_head.%d.weight" % (pos - 1)) @ h)
        codes.append(pick(cp[-1], (cs + pos * 0xD1B54A32D192ED03) & m))
    step = emb[0][codes[0]].double()
    for i in range(1, GROUPS):
        step = step + emb[i][codes[i]].double()
    return codes, torch.stack(cp), step + trailing.double()


def _rows(kv, n):
    return [(kv.k[i, :n], kv.v[i, :n]) for i in range(TALKER_LAYERS)]


def _exact_frame(case, s):
    n = case["n_past"]
    h, lg, new = _talker(s["step_in"].double()[None], _rows(s["kv"], n), n)
    _, cp, step = _frame(h, lg, s["trailing"][0], s["seed"], 3, set())
    return {"codes": None, "hidden": h, "logits": lg, "cp_logits": cp, "step": step,
            "k": torch.stack([k[n:] for k, _ in new]).double(), "v": torch.stack([v[n:] for _, v in new]).double()}


def _exact_loop(case, s):
    n, kv, seen = case["n_past"], None, set()
    kv = _rows(s["kv"], n)
    h, lg = s["hidden"].double(), s["logits"].double()
    for i in range(case["frames"]):
        if i:
            h, lg, kv = _talker(step[None], kv, n - 1 + i)
        _, cp, step = _frame(h, lg, s["trailing"][i], s["seed"], i, seen, lambda v, _: int(torch.argmax(v)))
    return {"codes": None, "hidden": h, "logits": lg, "cp_logits": cp, "step": step,
            "k": torch.stack([k[n:] for k, _ in kv]).double(), "v": torch.stack([v[n:] for _, v in kv]).double()}


def _prefilled(x):
    none = torch.empty(0, KVD, dtype=torch.float16, device="cuda")
    h, lg, new = _talker(x, [(none, none)] * TALKER_LAYERS, 0)
    return {"hidden": h, "logits": lg, "k": [k.double() for k, _ in new], "v": [v.double() for _, v in new]}


def _exact_prefill(case, s):
    return _prefilled(s["rows"].double())


def _exact_prompt(case, s):
    kv, w = blob.qwen3tts_0p6b_kv(), _weights("talker").t
    ids = s["ids"][:-5].tolist() + [kv["text.tts_bos_id"], kv["text.tts_eos_id"], kv["text.tts_pad_id"]]
    x, p = w["talker.model.text_embedding.weight"][ids].double(), "talker.text_projection.linear_fc"
    x = torch.nn.functional.silu(x @ _cached("talker", p + "1.weight").T + w[p + "1.bias"].double())
    x = x @ _cached("talker", p + "2.weight").T + w[p + "2.bias"].double()
    bos, eos, pad = x[-3], x[-2], x[-1]
    code = w["talker.model.codec_embedding.weight"].double()
    think = ["talker.codec_think_id", "talker.codec_think_bos_id", "talker.language.english", "talker.codec_think_eos_id"]
    rows = [x[0], x[1], x[2]] + [pad + code[kv[k]] for k in think] + [pad + torch.from_numpy(s["speaker"]).cuda().double()]
    rows += [bos + code[kv["talker.codec_pad_id"]], x[3] + code[kv["talker.codec_bos_id"]]]
    return {**_prefilled(torch.stack(rows)), "trailing": torch.cat([x[4:-3], eos[None]]), "tts_pad": pad}


def _exact_streams(case, s):
    """The talker's step. What hangs on the draws has no value here: among the many of a batch, 64 bits
    may resolve one at the edge of two codes the other way."""
    new = [_talker(s["step_in"][i].double()[None], _rows(s["kvs"][i], p), p)[2] for i, p in enumerate(s["n_past"])]
    return {"codes": None, "step": None, "k": torch.stack([torch.stack([k[-1] for k, _ in n]) for n in new]).double(),
            "v": torch.stack([torch.stack([v[-1] for _, v in n]) for n in new]).double()}


def _conv(x, w, b, dil=1):
    """Causal: x [T][Cin], w [Cout][Cin][K] -> [T][Cout]."""
    K, T = w.shape[2], x.shape[0]
    x = torch.cat([x.new_zeros((K - 1) * dil, x.shape[1]), x])
    return sum(x[j * dil:j * dil + T] @ w[:, :, j].T for j in range(K)) + b


def _up(x, w, b, s):
    """Transposed, stride s, kernel s or 2 s, trimmed on the right: x [T][Cin] -> [T s][Cout]."""
    T, k = x.shape[0], w.shape[2]
    y = torch.stack([x @ w[:, :, j] for j in range(k)], 1)                # [T][k][Cout]
    out = x.new_zeros(T + 1, s, w.shape[1])
    out[:T] += y[:, :s]
    if k > s:
        out[1:] += y[:, s:]
    return out[:T].reshape(T * s, -1) + b


def _snake(x, a, b):
    return x + torch.sin(x * torch.exp(a)) ** 2 / (torch.exp(b) + 1e-9)


def _exact_vocoder(case, s):
    D = "codec.decoder."

    def w(name):
        return _cached("codec", D + name)

    def cb(name):
        return (w(name + ".weight"), w(name + ".bias"))
    codes, q = torch.from_numpy(s["codes"]).cuda().long(), "quantizer."
    first = w(q + "rvq_first.vq.layers.0._codebook.codebook")[codes[:, 0]]
    rest = sum(w(q + "rvq_rest.vq.layers.%d._codebook.codebook" % i)[codes[:, i + 1]] for i in range(GROUPS - 1))
    x = first @ w(q + "rvq_first.output_proj.weight")[:, :, 0].T + rest @ w(q + "rvq_rest.output_proj.weight")[:, :, 0].T
    x = _conv(x, *cb("pre_conv.conv"))
    p = "pre_transformer."
    x = x @ w(p + "input_proj.weight").T + w(p + "input_proj.bias")
    T = x.shape[0]
    at = torch.arange(T, device="cuda")
    far = (at[None, :] > at[:, None]) | (at[:, None] - at[None, :] >= 72)
    for i in range(8):
        n = p + "layers.%d." % i
        y = _rms(x, w(n + "input_layernorm.weight"), 1e-5)
        qq, kk, vv = ((y @ w(n + "self_attn.%s_proj.weight" % c).T).view(T, 16, 64) for c in "qkv")
        qq, kk = _rotate(qq, at, 1e4), _rotate(kk, at, 1e4)
        a = torch.bmm(qq.permute(1, 0, 2).contiguous(), kk.permute(1, 2, 0).contiguous()) / 8.0
        a = torch.softmax(a.masked_fill(far[None], float("-inf")), -1)
        a = torch.bmm(a, vv.permute(1, 0, 2).contiguous()).permute(1, 0, 2).reshape(T, 1024)
        x = x + a @ w(n + "self_attn.o_proj.weight").T * w(n + "self_attn_layer_scale.scale")
        y = _rms(x, w(n + "post_attention_layernorm.weight"), 1e-5)
        y = torch.nn.functional.silu(y @ w(n + "mlp.gate_proj.weight").T) * (y @ w(n + "mlp.up_proj.weight").T)
        x = x + y @ w(n + "mlp.down_proj.weight").T * w(n + "mlp_layer_scale.scale")
    x = _rms(x, w(p + "norm.weight"), 1e-5) @ w(p + "output_proj.weight").T + w(p + "output_proj.bias")
    for j in range(2):
        u = "upsample.%d." % j
        x = _up(x, *cb(u + "0.conv"), 2)
        y, k = torch.cat([x.new_zeros(6, 1024), x]), w(u + "1.dwconv.conv.weight")
        y = sum(y[i:i + x.shape[0]] * k[:, 0, i] for i in range(7)) + w(u + "1.dwconv.conv.bias")
        y = torch.nn.functional.layer_norm(y, (1024,), *cb(u + "1.norm"), eps=1e-6)
        y = torch.nn.functional.gelu(y @ w(u + "1.pwconv1.weight").T + w(u + "1.pwconv1.bias"))
        x = x + (y @ w(u + "1.pwconv2.weight").T + w(u + "1.pwconv2.bias")) * w(u + "1.gamma")
    x = _conv(x, *cb("decoder.0.conv"))
    for i, r in enumerate((8, 5, 4, 3)):
        b = "decoder.%d.block." % (i + 1)
        x = _up(_snake(x, w(b + "0.alpha"), w(b + "0.beta")), *cb(b + "1.conv"), r)
        for j, dil in enumerate((1, 3, 9)):
            u = b + "%d." % (j + 2)
            y = _conv(_snake(x, w(u + "act1.alpha"), w(u + "act1.beta")), *cb(u + "conv1.conv"), dil)
            x = x + _conv(_snake(y, w(u + "act2.alpha"), w(u + "act2.beta")), *cb(u + "conv2.conv"))
    x = _conv(_snake(x, w("decoder.5.alpha"), w("decoder.5.beta")), *cb("decoder.6.conv"))[:, 0].clamp(-1.0, 1.0)
    cuts = [0] + list(range(case["first"], case["frames"], case["batch"])) + [case["frames"]]
    if case["first"] >= case["frames"]:
        cuts = [0, case["frames"]]
    return [x[a * SAMPLES_PER_FRAME:b * SAMPLES_PER_FRAME] for a, b in zip(cuts, cuts[1:])]


def _mel_filters():
    """Slaney mel scale and norm over 513 bins of 24 kHz, 0 to 12 kHz, rounded to f32 as the model holds them."""
    hz = np.arange(513) * 12000.0 / 512
    top = 15.0 + math.log(12.0) / (math.log(6.4) / 27.0)
    m = np.arange(130) * top / 129
    f = np.where(m >= 15.0, 1000.0 * np.exp(math.log(6.4) / 27.0 * (m - 15.0)), 200.0 / 3.0 * m)
    lo, up = (hz[None] - f[:128, None]) / (f[1:129] - f[:128])[:, None], (f[2:, None] - hz[None]) / (f[2:] - f[1:129])[:, None]
    return (np.maximum(0.0, np.minimum(lo, up)) * (2.0 / (f[2:] - f[:128]))[:, None]).astype(np.float32).astype(np.float64)


def _exact_speaker(case, s):
    y = np.pad(s["wav"].astype(np.float64), (384, 384), mode="reflect")
    at = np.arange((len(y) - 1024) // 256 + 1)[:, None] * 256 + np.arange(1024)[None]
    spec = np.fft.rfft(y[at] * (0.5 - 0.5 * np.cos(2.0 * np.pi * np.arange(1024) / 1024)), axis=1)
    mel = np.log(np.maximum(np.sqrt(np.abs(spec) ** 2 + 1e-9) @ _mel_filters().T, 1e-5))
    P = "speaker_encoder."

    def conv(name, x, dil=1):
        """"same" with reflected ends: x [T][Cin] -> [T][Cout]."""
        w, b, T = _cached("speaker", P + name + ".weight"), _cached("speaker", P + name + ".bias"), x.shape[0]
        pad = (w.shape[2] - 1) * dil // 2
        if pad:
            x = torch.cat([x[1:pad + 1].flip(0), x, x[-pad - 1:-1].flip(0)])
        return sum(x[j * dil:j * dil + T] @ w[:, :, j].T for j in range(w.shape[2])) + b
    h, outs = torch.relu(conv("blocks.0.conv", torch.from_numpy(mel).cuda())), []
    for b, dil in ((1, 2), (2, 3), (3, 4)):
        n = "blocks.%d." % b
        parts = list(torch.relu(conv(n + "tdnn1.conv", h)).split(64, 1))
        c = [parts[0]]
        for i in range(1, 8):
            c.append(torch.relu(conv(n + "res2net_block.blocks.%d.conv" % (i - 1), parts[i] + (c[-1] if i > 1 else 0.0), dil)))
        y = torch.relu(conv(n + "tdnn2.conv", torch.cat(c, 1)))
        g = torch.relu(conv(n + "se_block.conv1", y.mean(0, keepdim=True)))
        h = y * torch.sigmoid(conv(n + "se_block.conv2", g)) + h
        outs.append(h)
    x = torch.relu(conv("mfa.conv", torch.cat(outs, 1)))
    T = x.shape[0]
    mean, std = x.mean(0), torch.sqrt(x.var(0, unbiased=False).clamp_min(1e-12))
    a = conv("asp.tdnn.conv", torch.cat([x, mean.expand(T, -1), std.expand(T, -1)], 1))
    a = torch.softmax(conv("asp.conv", torch.tanh(torch.relu(a))), 0)
    m = (a * x).sum(0)
    v = torch.sqrt((a * (x - m) ** 2).sum(0).clamp_min(1e-12))
    return conv("fc", torch.cat([m, v])[None])[0]
