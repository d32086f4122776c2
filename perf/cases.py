"""Timed cases of the framework's public entry points: what a program that
serves text-to-speech with it calls.

* ``fast``      -- Engine.fast_logits: the Fast-AR logits after a prefix of codes
                   (a caller with its own sampler); the smallest call.
* ``steps``     -- Engine.eval of a short prompt, then Engine.step token by
                   token, each with full-vocabulary logits (a caller that owns
                   the decode loop).
* ``prefill``   -- Engine.eval of a whole prompt: plain text, or a voice-clone
                   prompt with reference frames.
* ``generate``  -- Engine.generate_codes, then the next turn's first text token
                   through Engine.step on the state the generation left.
* ``batch``     -- Engine.generate_codes_batch, then the same on request 0.
* ``codec``     -- Codec.decode_waveform (host arrays) or decode_waveform_device
                   (codes and samples on the GPU): codes to audio.
* ``latents``   -- Codec.decode_latents: post-module transformer and upsampling.
* ``decoder``   -- Codec.decoder: the convolutional decoder alone.

Models are the seeded synthetic S2-Pro-shaped GGUFs of ``s2hip.synth`` (f16,
Q8_0 or Q4_0 linears); prompts, codes and latents are drawn from the seed.
A program keeps its opened engine or codec over many inputs, so they are
opened once per process here as well.
"""

import math
import mmap
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("fish-s2pro_amd"))

from s2hip import Codec, Engine, synth  # noqa: E402

MODELS = {"f16": synth.FULL, "q8": synth.FULL_Q8, "q4": synth.FULL_Q4}
CODEC_MAX_FRAMES = 512
NEVER = 1 << 30  # min_tokens_before_end: the frame count is the caller's


def listed():
    return [
        # one Fast-AR evaluation with three codes known: launch latency
        {"name": "fast_f16_3", "kind": "fast", "model": "f16", "prefix": 3, "kv": 768},
        # a caller's own decode loop after a short prompt
        {"name": "steps_f16", "kind": "steps", "model": "f16", "prompt": 40, "steps": 8, "kv": 768, "kv_f16": False},
        # the same on 4-bit weights with a half-precision KV cache and a longer context
        {"name": "steps_q4_kvf16", "kind": "steps", "model": "q4", "prompt": 331, "steps": 5, "kv": 2560, "kv_f16": True},
        # a plain text prompt of the benchmark's length
        {"name": "prefill_f16_256", "kind": "prefill", "model": "f16", "prompt": 256, "voice": 0, "kv": 768, "kv_f16": False},
        # a voice-clone prompt: 250 + 1000 reference frames + 250
        {"name": "prefill_f16_1500", "kind": "prefill", "model": "f16", "prompt": 1500, "voice": 1000, "kv": 2560, "kv_f16": False},
        # a ragged mid-size prompt on 8-bit weights
        {"name": "prefill_q8_389", "kind": "prefill", "model": "q8", "prompt": 389, "voice": 200, "kv": 768, "kv_f16": False},
        # the headline loop: 256-token prompt, greedy, batch 1
        {"name": "generate_f16", "kind": "generate", "model": "f16", "prompt": 256, "frames": 32, "temperature": 0.0, "top_p": 1.0, "top_k": 0, "kv": 768},
        # sampled speech on 8-bit weights with the default sampler settings
        {"name": "generate_q8_sampled", "kind": "generate", "model": "q8", "prompt": 117, "frames": 24, "temperature": 0.7, "top_p": 0.7, "top_k": 30, "kv": 768},
        # eight concurrent voice-clone requests
        {"name": "batch8_f16", "kind": "batch", "model": "f16", "requests": 8, "prompt": 300, "voice": 200, "frames": 16, "kv": 2560},
        # five concurrent requests on 4-bit weights
        {"name": "batch5_q4", "kind": "batch", "model": "q4", "requests": 5, "prompt": 150, "voice": 0, "frames": 16, "kv": 768},
        # a whole utterance: 512 code frames, 24 s of audio, on the GPU
        {"name": "codec_512", "kind": "codec", "frames": 512, "device": True},
        # a streaming-sized piece through host arrays
        {"name": "codec_37_host", "kind": "codec", "frames": 37, "device": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fast", "steps", "prefill", "prefill", "generate", "batch", "codec", "codec", "latents", "decoder"])
    model = rng.choice(["f16", "f16", "q8", "q4"])
    if kind == "fast":
        return {"kind": kind, "model": model, "prefix": rng.randint(0, 9), "kv": 768}
    if kind == "steps":
        return {"kind": kind, "model": model, "prompt": _log_int(rng, 1, 500), "steps": rng.randint(3, 10), "kv": 768,
                "kv_f16": rng.random() < 0.3}
    if kind == "prefill":
        n = _log_int(rng, 3, 1500)
        return {"kind": kind, "model": model, "prompt": n, "voice": rng.choice([0, n // 2]), "kv": 2560 if n > 700 else 768,
                "kv_f16": rng.random() < 0.3}
    if kind == "generate":
        # greedy, or the default sampler; top-p over the whole codebook is left out:
        # thousands of the synthetic model's flat probabilities share its draw, which
        # then hangs on the last bits of the logits
        t, p, k = rng.choice([(0.0, 1.0, 0), (0.7, 0.7, 30)])
        return {"kind": kind, "model": model, "prompt": _log_int(rng, 12, 400), "frames": rng.randint(6, 30),
                "temperature": t, "top_p": p, "top_k": k, "kv": 768}
    if kind == "batch":
        n = _log_int(rng, 20, 300)
        return {"kind": kind, "model": model, "requests": rng.randint(2, 8), "prompt": n, "voice": rng.choice([0, n // 2]),
                "frames": rng.randint(6, 12), "kv": 768}
    if kind == "codec":
        return {"kind": kind, "frames": _log_int(rng, 1, 500), "device": rng.random() < 0.5}
    if kind == "latents":
        return {"kind": kind, "frames": _log_int(rng, 1, 400)}
    return {"kind": "decoder", "frames": _log_int(rng, 2, 1200)}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
_opened = {}


def _dir():
    d = os.environ.get("S2HIP_MODEL_DIR") or os.path.join(tempfile.gettempdir(), "s2hip_models_%d" % os.getuid())
    os.makedirs(d, exist_ok=True)
    return d


def _model_path(model):
    return synth.ensure_gguf(MODELS[model], _dir(), threads=min(16, os.cpu_count() or 1))


def _codec_path():
    return synth.ensure_codec_gguf(_dir(), threads=min(16, os.cpu_count() or 1))


def _engine(model, kv, kv_f16=False):
    key = (model, kv, kv_f16)
    if key not in _opened:
        _opened[key] = Engine(_model_path(model), kv, MODELS[model].im_end_id, kv_f16=kv_f16)
    return _opened[key]


def _codec():
    if "codec" not in _opened:
        _opened["codec"] = Codec(_codec_path(), CODEC_MAX_FRAMES)
    return _opened["codec"]


def _prompt(shape, n, voice, seed):
    if voice:
        return synth.voice_clone_prompt(shape, n - voice, voice, seed)
    return synth.synthetic_prompt(shape, n, seed)


def _inputs(case, seed):
    """The host arrays of a case, from its seed alone."""
    kind = case["kind"]
    rng = np.random.default_rng([seed, 11])
    if kind == "codec":
        n = case["frames"]
        return {"codes": np.concatenate([rng.integers(0, 4096, (1, n)), rng.integers(0, 1024, (9, n))]).astype(np.int32)}
    if kind == "latents":  # sums of ten projected code vectors: spread of about 3
        return {"x": (3.0 * rng.standard_normal((case["frames"], 1024))).astype(np.float32)}
    if kind == "decoder":
        return {"x": rng.standard_normal((case["frames"], 1024)).astype(np.float32)}
    shape = MODELS[case["model"]]
    if kind == "fast":  # a post-norm hidden row has a root mean square of one
        return {"hidden": rng.standard_normal(shape.dim).astype(np.float32),
                "prefix": rng.integers(0, shape.codebook_size, case["prefix"]).astype(np.uint32)}
    if kind == "steps":
        return {"prompt": _prompt(shape, case["prompt"], 0, seed),
                "rows": _prompt(shape, case["steps"] + 2, case["steps"], seed + 1).reshape(-1, shape.num_codebooks + 1)[1:-1]}
    if kind == "prefill":
        return {"prompt": _prompt(shape, case["prompt"], case["voice"], seed)}
    requests = case["requests"] if kind == "batch" else 1
    return {"prompts": [_prompt(shape, case["prompt"], case.get("voice", 0), seed + 1009 * b) for b in range(requests)],
            "next": synth.synthetic_prompt(shape, 1, seed + 5), "rng": [int(seed) + 77 * b for b in range(requests)]}


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case)
    if case["kind"] in ("codec", "latents", "decoder"):
        state["codec"] = _codec()
        if case.get("device"):
            state["codes_dev"] = torch.from_numpy(state["codes"]).cuda()
            state["samples"] = torch.empty(case["frames"] * 2048, device="cuda")
            torch.cuda.synchronize()
    else:
        state["engine"] = _engine(case["model"], case["kv"], case.get("kv_f16", False))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "codec":
        c, n = state["codec"], case["frames"]
        if case["device"]:
            c.decode_waveform_device(state["codes_dev"].data_ptr(), 10, n, state["samples"].data_ptr())
            return state["samples"]
        return c.decode_waveform(state["codes"], 10, n).samples
    if kind == "latents":
        return state["codec"].decode_latents(state["x"])
    if kind == "decoder":
        return state["codec"].decoder(state["x"])
    eng = state["engine"]
    if kind == "fast":
        return eng.fast_logits(state["hidden"], state["prefix"])
    if kind == "prefill":
        eng.reset()
        return eng.eval(state["prompt"])
    if kind == "steps":
        eng.reset()
        out = [eng.eval(state["prompt"])]
        for row in state["rows"]:
            out.append(eng.step(row))
        return out
    if kind == "generate":
        g = eng.generate_codes(state["prompts"][0], case["frames"], case["temperature"], case["top_p"], case["top_k"],
                               NEVER, state["rng"][0])
        codes = g["codes"]
    else:
        g = eng.generate_codes_batch(state["prompts"], case["frames"], min_tokens_before_end=NEVER, rng_states=state["rng"])
        codes = [r["codes"] for r in g["requests"]]
    hidden, logits = eng.step(state["next"])
    return {"codes": codes, "hidden": hidden, "logits": logits}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _conv_macs():
    """Multiply-adds per code frame of the codec's products: (post-module and
    upsampling, decoder) and their f16 weight counts."""
    post = 8 * (1024 * 3072 + 1024 * 1024 + 3 * 1024 * 3072)
    up1 = 2 * 1024 * 1024 + 2 * (2 * 1024 * 4096)
    up2 = 2 * up1
    front_w = post + 2 * (2 * 1024 * 1024 + 2 * 1024 * 4096)
    ch, rate = (1536, 768, 384, 192, 96), (8, 8, 4, 2)
    macs, w, f = 7 * 1024 * 1536, 7 * 1024 * 1536, 1  # per latent frame
    for b in range(4):
        macs += f * rate[b] * 2 * ch[b] * ch[b + 1]
        w += 2 * rate[b] * ch[b] * ch[b + 1]
        f *= rate[b]
        macs += 3 * f * 8 * ch[b + 1] ** 2
        w += 3 * 8 * ch[b + 1] ** 2
    return (post + up1 + up2, front_w), (macs + f * 7 * 96, w)


def _lm_work(case):
    shape = MODELS[case["model"]]
    per = {"f16": 2.0, "q8": 34 / 32, "q4": 18 / 32}[case["model"]]
    slow = shape.slow_layers * shape.linear_params_per_slow_layer()
    fast = shape.fast_layers * shape.linear_params_per_fast_layer()
    d, kvd = shape.dim, shape.kv_heads * shape.head_dim
    kvb = 2 if case.get("kv_f16") else 4
    head = shape.vocab * d
    cand = (shape.codebook_size + 1) * d
    out = shape.codebook_size * d
    nbytes = flops = 0.0

    def evaluate(n, past, logits=True):
        nonlocal nbytes, flops
        nbytes += slow * per + n * 2 * kvd * shape.slow_layers * kvb + past * 2 * kvd * shape.slow_layers * kvb
        flops += 2.0 * slow * n + 4.0 * shape.slow_layers * shape.heads * shape.head_dim * (n * past + n * (n + 1) / 2)
        if logits:
            nbytes += 2 * head + 4 * shape.vocab
            flops += 2.0 * head

    kind = case["kind"]
    if kind == "fast":  # positions 0 .. prefix in one pass over the weights
        n = case["prefix"] + 1
        return {"bytes": fast * per + out * per + 4 * (d + shape.codebook_size), "flops": 2.0 * (fast * n + out)}
    if kind == "prefill":
        evaluate(case["prompt"], 0)
    elif kind == "steps":
        evaluate(case["prompt"], 0)
        for i in range(case["steps"]):
            evaluate(1, case["prompt"] + i)
    else:
        r = case.get("requests", 1)
        frames = case["frames"]
        nbytes += slow * per  # every request's prompt in one pass over the weights
        for _ in range(r):
            b0 = nbytes
            evaluate(case["prompt"], 0, logits=False)
            nbytes = b0 + case["prompt"] * 2 * kvd * shape.slow_layers * kvb
        for i in range(frames):
            past = case["prompt"] + i
            nbytes += slow * per + cand * 2 + 9 * (fast + out) * per + r * (past + 1) * 2 * kvd * shape.slow_layers * kvb
            flops += r * (2.0 * slow + 2.0 * cand + 2.0 * 10 * fast + 9 * 2.0 * out
                          + 4.0 * shape.slow_layers * shape.heads * shape.head_dim * (past + 1))
        evaluate(1, case["prompt"] + frames)
    return {"bytes": nbytes, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind not in ("codec", "latents", "decoder"):
        return _lm_work(case)
    (front, front_w), (dec, dec_w) = _conv_macs()
    n = case["frames"]
    if kind == "codec":
        return {"bytes": n * (40 + 2048 * 4) + 2 * (front_w + dec_w), "flops": 2.0 * n * (front + 4 * dec)}
    if kind == "latents":
        return {"bytes": n * 5 * 4096 + 2 * front_w, "flops": 2.0 * n * front}
    return {"bytes": n * (4096 + 512 * 4) + 2 * dec_w, "flops": 2.0 * n * dec}


def tolerance(case):
    kind = case["kind"]
    if kind in ("codec", "decoder"):
        # convolution inputs are f16: a sum in another order moves some of them
        # by one rounding, and thirteen convolutions carry that on
        return {"rel": 6e-3, "max": 0.2}
    if kind == "latents":
        return {"rel": 1e-5, "max": 1e-3}
    if case.get("kv_f16"):
        # cache entries rounded to 16 bits: another sum order moves some by one rounding
        return {"rel": 1e-3, "max": 4e-2}
    # f32 sums through 36 layers; "differ" is for a tie between two codes
    return {"rel": 2.5e-5, "max": 1e-3, "differ": 0.01}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------
class _Gguf:
    """The tensors of a GGUF file as 64-bit torch tensors on the GPU (their stored bytes stay there)."""

    SCALAR = {0: "B", 1: "b", 2: "H", 3: "h", 4: "I", 5: "i", 6: "f", 7: "?", 10: "Q", 11: "q", 12: "d"}
    BLOCK = {0: (1, 4), 1: (1, 2), 2: (32, 18), 8: (32, 34)}

    def __init__(self, path):
        with open(path, "rb") as f:
            self.map = mmap.mmap(f.fileno(), 0, access=mmap.ACCESS_READ)
        self.at = 4
        _, n, kv = self.take("<IQQ")
        self.meta = {}
        for _ in range(kv):
            key = self.text()
            self.meta[key] = self.value(self.take("<I")[0])
        infos = []
        for _ in range(n):
            name = self.text()
            dims = self.take("<%dQ" % self.take("<I")[0])
            infos.append((name, dims) + self.take("<IQ"))
        align = self.meta.get("general.alignment", 32)
        start = (self.at + align - 1) // align * align
        self.infos = {name: (dims, kind, start + off) for name, dims, kind, off in infos}
        self.held = {}

    def take(self, fmt):
        v = struct.unpack_from(fmt, self.map, self.at)
        self.at += struct.calcsize(fmt)
        return v

    def text(self):
        n = self.take("<Q")[0]
        s = bytes(self.map[self.at:self.at + n]).decode()
        self.at += n
        return s

    def value(self, kind):
        if kind == 8:
            return self.text()
        if kind == 9:
            k, n = self.take("<IQ")
            return [self.value(k) for _ in range(n)]
        return self.take("<" + self.SCALAR[kind])[0]

    def stored(self, name):
        if name not in self.held:
            dims, kind, off = self.infos[name]
            per, size = self.BLOCK[kind]
            raw = np.frombuffer(self.map, np.uint8, math.prod(dims) // per * size, off)
            self.held[name] = torch.from_numpy(raw.copy()).cuda()
        return self.held[name]

    def __call__(self, name, rows=None):
        """The tensor, outermost dimension first; of a matrix, `rows` alone if given."""
        dims, kind, _ = self.infos[name]
        t = self.stored(name)
        shape = tuple(reversed(dims))
        if kind in (0, 1):
            t = t.view(torch.float32 if kind == 0 else torch.float16).view(shape)
            return (t if rows is None else t[rows]).double()
        b = t.view(-1, 34 if kind == 8 else 18)
        d = b[:, :2].contiguous().view(torch.float16).double()
        if kind == 8:
            q = b[:, 2:].contiguous().view(torch.int8).double()
        else:
            q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8.0
        return (q * d).view(shape)


_files = {}


def _file(path):
    if path not in _files:
        _files.clear()
        _files[path] = _Gguf(path)
    return _files[path]


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, base):
    """x [n][heads][hd]: adjacent pairs turned by position / base^(2 i / hd), an angle that the model defines in 32 bits."""
    hd = x.shape[-1]
    div = np.power(np.float64(np.float32(base)), np.arange(0, hd, 2) / hd).astype(np.float32)
    ang = (pos.astype(np.float32)[:, None] / div[None, :]).astype(np.float64)
    c, s = (torch.from_numpy(f(ang)).cuda()[:, None, :] for f in (np.cos, np.sin))
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _attend(q, k, v, past, window=None):
    """q [n][H][hd] at positions past .., over k, v [T][Hkv][hd]; causal."""
    n, heads, hd = q.shape
    rep = heads // k.shape[1]
    kt = k.repeat_interleave(rep, 1).permute(1, 2, 0).contiguous()
    vt = v.repeat_interleave(rep, 1).permute(1, 0, 2).contiguous()
    s = torch.bmm(q.permute(1, 0, 2).contiguous(), kt) / math.sqrt(hd)
    i = torch.arange(past, past + n, device="cuda")[:, None]
    j = torch.arange(k.shape[0], device="cuda")[None, :]
    hide = j > i
    if window:
        hide = hide | (j <= i - window)
    s = s.masked_fill(hide, -math.inf).softmax(-1)
    return torch.bmm(s, vt).permute(1, 0, 2).reshape(n, heads * hd)


class _Lm:
    """The dual-AR transformer of a GGUF file in 64 bits."""

    def __init__(self, path, kv_f16=False):
        self.w = _file(path)
        self.kv_f16 = kv_f16
        m = self.w.meta
        self.eps, self.base = m["fish-speech.attention.layer_norm_rms_epsilon"], m["fish-speech.rope.freq_base"]
        self.feps, self.fbase = m["fish_speech.fast_layer_norm_rms_eps"], m["fish_speech.fast_rope_freq_base"]
        self.kv = {}

    def reset(self):
        self.kv = {}

    def embed(self, flat, shape):
        rows = torch.from_numpy(np.asarray(flat, np.int64).reshape(-1, shape.num_codebooks + 1)).cuda()
        x = self.w("embeddings.weight", rows[:, 0])
        sem = (rows[:, 0] >= shape.semantic_begin) & (rows[:, 0] <= shape.semantic_end)
        if bool(sem.any()):
            at = rows[sem, 1:] + torch.arange(shape.num_codebooks, device="cuda") * shape.codebook_size
            add = self.w("codebook_embeddings.weight", at.reshape(-1)).view(-1, shape.num_codebooks, shape.dim).sum(1)
            x[sem] = (x[sem] + add) / math.sqrt(shape.num_codebooks + 1)
        return x

    def layers(self, xs, seqs, prefix, count, heads, kvh, hd, eps, base, qk_norm, f16):
        """One pass of the rows xs[i] appended to the sequences seqs[i]."""
        sizes = [x.shape[0] for x in xs]
        x = torch.cat(xs)
        w = self.w
        nq, nk = heads * hd, kvh * hd
        for l in range(count):
            p = "%s.%d." % (prefix, l)
            qkv = (_rms(x, w(p + "attention_norm.weight"), eps) @ w(p + "attention.wqkv.weight").T).split(sizes)
            att = []
            for part, seq in zip(qkv, seqs):
                n = part.shape[0]
                q, k, v = (t.reshape(n, -1, hd) for t in part.split([nq, nk, nk], 1))
                if qk_norm:
                    q, k = _rms(q, w(p + "attention.q_norm.weight"), eps), _rms(k, w(p + "attention.k_norm.weight"), eps)
                old = self.kv.get((seq, p))
                past = old[0].shape[0] if old else 0
                pos = np.arange(past, past + n)
                q, k = _rope(q, pos, base), _rope(k, pos, base)
                if f16:
                    k, v = k.half().double(), v.half().double()
                if old:
                    k, v = torch.cat([old[0], k]), torch.cat([old[1], v])
                self.kv[(seq, p)] = (k, v)
                att.append(_attend(q, k, v, past))
            x = x + torch.cat(att) @ w(p + "attention.wo.weight").T
            h = _rms(x, w(p + "ffn_norm.weight"), eps)
            g = h @ w(p + "feed_forward.w1.weight").T
            x = x + (g * torch.sigmoid(g) * (h @ w(p + "feed_forward.w3.weight").T)) @ w(p + "feed_forward.w2.weight").T
        return x.split(sizes)

    def slow(self, flats, seqs, shape):
        """The post-norm hidden of the last token of each block of tokens."""
        xs = self.layers([self.embed(f, shape) for f in flats], seqs, "layers", shape.slow_layers, shape.heads,
                         shape.kv_heads, shape.head_dim, self.eps, self.base, True, self.kv_f16)
        return _rms(torch.stack([x[-1] for x in xs]), self.w("norm.weight"), self.eps)

    def logits(self, hidden, rows=None):
        return hidden @ self.w("embeddings.weight", rows).T

    def fast(self, rows, seqs, shape):
        """Fast-AR logits after each sequence's new rows."""
        xs = self.layers(rows, seqs, "fast_layers", shape.fast_layers, shape.fast_heads, shape.fast_kv_heads,
                         shape.fast_head_dim, self.feps, self.fbase, False, False)
        return _rms(torch.stack([x[-1] for x in xs]), self.w("fast_norm.weight"), self.feps) @ self.w("fast_output.weight").T


def _sample(logits, case, state):
    """(index, new generator state) of one draw over logits; the model defines
    the probabilities and their running sums in 32 bits, term after term."""
    x = logits.cpu().numpy()
    state = (state * 6364136223846793005 + 1) % (1 << 64)
    t = case.get("temperature", 0.0)
    if t <= 0.0:
        return int(x.argmax()), state
    order = np.argsort(-x, kind="stable")
    if case["top_k"]:
        order = order[: case["top_k"]]
    x = x[order].astype(np.float32)
    p = np.exp(((x - x[0]) / np.float32(t)).astype(np.float64)).astype(np.float32)
    p /= np.cumsum(p)[-1]
    reach = np.cumsum(p) >= np.float32(case["top_p"])
    p = p[: int(reach.argmax()) + 1] if reach.any() else p
    p = p / np.cumsum(p)[-1]
    u = np.float32((state >> 11) / float(1 << 53))
    over = np.cumsum(p) > min(max(u, np.float32(0.0)), np.float32(1.0) - np.float32(1e-7))
    return int(order[over.argmax() if over.any() else len(p) - 1]), state


def _exact_lm(case, seed):
    kind, shape = case["kind"], MODELS[case["model"]]
    x = _inputs(case, seed)
    lm = _Lm(_model_path(case["model"]), case.get("kv_f16", False))
    if kind == "fast":
        rows = torch.cat([torch.from_numpy(x["hidden"]).cuda().double()[None],
                          lm.w("fast_embeddings.weight", torch.from_numpy(x["prefix"].astype(np.int64)).cuda())])
        return lm.fast([rows], [0], shape)[0]
    if kind in ("prefill", "steps"):
        out = []
        for block in [x["prompt"]] + list(x.get("rows", [])):
            h = lm.slow([block], [0], shape)[0]
            out.append((h, lm.logits(h)))
        return out[0] if kind == "prefill" else out
    n = len(x["prompts"])
    seqs, rngs = list(range(n)), list(x["rng"])
    cand = torch.arange(shape.semantic_begin, shape.semantic_end + 1, device="cuda")
    hidden = torch.cat([lm.slow([x["prompts"][b]], [b], shape) for b in seqs])

    def sample(logits):
        got = []
        for b in seqs:
            i, rngs[b] = _sample(logits[b], case, rngs[b])
            got.append(i)
        return got

    sem = sample(lm.logits(hidden, cand))
    for _ in range(case["frames"]):
        rows, codes = [hidden[b][None] for b in seqs], [[c] for c in sem]
        for cb in range(1, shape.num_codebooks):
            emb = lm.w("fast_embeddings.weight", torch.tensor([c[-1] for c in codes], device="cuda"))
            new = [torch.cat([rows[b], emb[b][None]]) if cb == 1 else emb[b][None] for b in seqs]
            if cb == 1:
                for key in [k for k in lm.kv if k[1].startswith("fast")]:
                    del lm.kv[key]
            for b, c in enumerate(sample(lm.fast(new, seqs, shape))):
                codes[b].append(c)
        hidden = lm.slow([[shape.semantic_begin + c[0]] + c for c in codes], seqs, shape)
        sem = sample(lm.logits(hidden, cand))
    h = lm.slow([x["next"]], [0], shape)[0]
    return {"codes": None if kind == "generate" else [None] * n, "hidden": h, "logits": lm.logits(h)}


def _causal(x, w, bias, dilation=1):
    """x [F][C] rounded to f16 as the model defines it, w [M][C][k]: causal convolution."""
    x = x.half().double()
    k = w.shape[2]
    y = bias.expand(x.shape[0], -1).clone()
    for t in range(k):
        back = (k - 1 - t) * dilation
        if back < x.shape[0]:
            y[back:] += x[: x.shape[0] - back] @ w[:, :, t].T
    return y


def _transposed(x, w, bias, stride):
    """x [F][C], w [C][M][k]: transposed convolution cropped to F * stride frames."""
    f = x.shape[0]
    y = bias.expand(f * stride, -1).clone().view(f, stride, -1)
    for t in range(w.shape[2]):
        back, r = t // stride, t % stride
        if back < f:
            y[back:, r] += x[: f - back] @ w[:, :, t]
    return y.view(f * stride, -1)


def _snake(x, alpha):
    a = torch.where(alpha.abs() < 1e-8, torch.full_like(alpha, 1e-8), alpha)
    return x + torch.sin(x * a) ** 2 / a


def _codec_latents(w, x):
    for l in range(8):
        p = "quantizer.post_module.layers.%d." % l
        n = x.shape[0]
        q, k, v = (t.reshape(n, 16, 64) for t in
                   (_rms(x, w(p + "attention_norm.weight"), 1e-5) @ w(p + "attention.wqkv.weight").T).split(1024, 1))
        pos = np.arange(n)
        a = _attend(_rope(q, pos, 1e4), _rope(k, pos, 1e4), v, 0, window=128)
        x = x + a @ w(p + "attention.wo.weight").T * w(p + "attention_layer_scale.gamma")
        h = _rms(x, w(p + "ffn_norm.weight"), 1e-5)
        g = h @ w(p + "feed_forward.w1.weight").T
        f = (g * torch.sigmoid(g) * (h @ w(p + "feed_forward.w3.weight").T)) @ w(p + "feed_forward.w2.weight").T
        x = x + f * w(p + "ffn_layer_scale.gamma")
    x = _rms(x, w("quantizer.post_module.norm.weight"), 1e-5)
    for s in range(2):
        p = "quantizer.upsample.%d." % s
        x = _transposed(x, w(p + "0.conv.weight"), w(p + "0.conv.bias"), 2)
        dw = w(p + "1.dwconv.conv.weight")[:, 0]
        y = w(p + "1.dwconv.conv.bias").expand(x.shape[0], -1).clone()
        for t in range(7):
            back = 6 - t
            if back < x.shape[0]:
                y[back:] += x[: x.shape[0] - back] * dw[:, t]
        y = torch.nn.functional.layer_norm(y, (1024,), w(p + "1.norm.weight"), w(p + "1.norm.bias"), 1e-6)
        y = torch.nn.functional.gelu(y @ w(p + "1.pwconv1.weight").T + w(p + "1.pwconv1.bias"))
        x = x + (y @ w(p + "1.pwconv2.weight").T + w(p + "1.pwconv2.bias")) * w(p + "1.gamma")
    return x


def _codec_decoder(w, x):
    x = _causal(x, w("decoder.model.0.conv.weight"), w("decoder.model.0.conv.bias"))
    for b in range(4):
        p = "decoder.model.%d.block." % (b + 1)
        x = _snake(x, w(p + "0.alpha").view(-1))
        x = _transposed(x, w(p + "1.conv.weight"), w(p + "1.conv.bias"), (8, 8, 4, 2)[b])
        for r in range(3):
            q = p + "%d.block." % (r + 2)
            y = _causal(_snake(x, w(q + "0.alpha").view(-1)), w(q + "1.conv.weight"), w(q + "1.conv.bias"), (1, 3, 9)[r])
            x = x + _causal(_snake(y, w(q + "2.alpha").view(-1)), w(q + "3.conv.weight"), w(q + "3.conv.bias"))
    x = _snake(x, w("decoder.model.5.alpha").view(-1))
    return torch.tanh(_causal(x, w("decoder.model.6.conv.weight").view(1, 96, 7), w("decoder.model.6.conv.bias")))[:, 0]


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind not in ("codec", "latents", "decoder"):
            return _exact_lm(case, seed)
        w, x = _file(_codec_path()), _inputs(case, seed)
        if kind == "latents":
            return _codec_latents(w, torch.from_numpy(x["x"]).cuda().double())
        if kind == "decoder":
            return _codec_decoder(w, torch.from_numpy(x["x"]).cuda().double())
        lat = torch.zeros(case["frames"], 1024, dtype=torch.float64, device="cuda")
        codes = torch.from_numpy(x["codes"].astype(np.int64)).cuda()
        for i in range(10):
            p = "quantizer.semantic_quantizer.quantizers.0." if i == 0 else "quantizer.quantizer.quantizers.%d." % (i - 1)
            lat += w(p + "codebook.weight")[codes[i]] @ w(p + "out_proj.weight").T + w(p + "out_proj.bias")
        return _codec_decoder(w, _codec_latents(w, lat))
