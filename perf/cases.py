"""The work whose speed matters to a user of this framework, as cases that a timing program can run one by one.

Every case goes through the public Python entry points (ctypes over the tk_* ABI), from host inputs to host results, as a host application's calls do:

  vad      30 ms windows of microphone input -> speech probabilities; the smallest call, made all day
  detect   camera frames -> boxes: one frame at a time in a cycle, many at once where one device serves many cameras
  listen   utterances -> mel, encoder, decoder: one speaker, or the pending utterances of many
  chat     a decoder of the Mistral class, Q4_K_M or f16: prompts of equal length, then greedy steps, then one step whose logits come back
  prompt   a layer-list decoder (bf16) takes in prompts of given lengths, the logits of each one's last position come back
  step     a layer-list decoder (bf16) takes one position for each of its live sequences, the logits come back

Models are the repository's own geometries with its seeded synthetic weights; a seed draws frames, sound and token ids.
"""
import math

import numpy as np
import torch

import trackiellm_amd as tk

VOCAB = 32000
CONF, IOU = 0.5, 0.5
#: CLS_BIAS: lowers the synthetic network's class outputs to where some tens of boxes of a frame pass CONF
DET_SEED, CLS_BIAS, ASR_SEED, VAD_SEED, LLM_SEED = 5, -11.0, 6, 7, 4
RANK = 128  # inner width of the layer-list decoders' low-rank gates


# ---------------------------------------------------------------- cases

def listed():
    return [
        # one second of microphone input, window by window: what decides whether anything else runs
        {"name": "vad", "kind": "vad", "windows": 33},
        # one cycle of one user: a VGA frame (latency of a deep chain of small layers) ...
        {"name": "detect_1", "kind": "detect", "frames": 1, "width": 640, "height": 480},
        # ... and a device that serves many cameras
        {"name": "detect_32", "kind": "detect", "frames": 32, "width": 640, "height": 480},
        # a short spoken command: encoder of one window, sixteen decoder steps of one row
        {"name": "listen_1", "kind": "listen", "clips": 1, "samples": 20011, "steps": 16},
        # the pending utterances of many users at once
        {"name": "listen_32", "kind": "listen", "clips": 32, "samples": 16000, "steps": 16},
        # one user, a prompt with context and a short answer: prompt passes, then steps that stream all weights for one row
        {"name": "chat_1", "kind": "chat", "weights": "q4", "layers": 32, "rows": 1, "prompt": 437, "steps": 24},
        # sixteen users of one model
        {"name": "chat_16", "kind": "chat", "weights": "q4", "layers": 32, "rows": 16, "prompt": 64, "steps": 24},
        # a full pass: 256 concurrent cycles
        {"name": "chat_256", "kind": "chat", "weights": "q4", "layers": 32, "rows": 256, "prompt": 32, "steps": 8},
        # fp16 checkpoints (a few layers of the same width), several users
        {"name": "f16_24", "kind": "chat", "weights": "f16", "layers": 4, "rows": 24, "prompt": 48, "steps": 16},
        # a long prompt through attention beside a delta rule
        {"name": "prompt_delta", "kind": "prompt", "model": "dense-4096", "lengths": "2047"},
        # several prompts of uneven lengths in one pass, retention and chunked attention
        {"name": "prompt_retention", "kind": "prompt", "model": "kaparax-2048", "lengths": "777,64,1,301,512,130"},
        # a decode step of many sequences (grouped experts have no case: with random weights their routers' close calls fall with every
        # rounding, and outputs of two correct runs cannot be compared)
        {"name": "step_40", "kind": "step", "model": "dense-2048", "rows": 40, "context": 350},
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))
    kind = rng.choice(["vad", "detect", "listen", "chat", "chat", "prompt", "step"])
    if kind == "vad":
        return {"kind": kind, "windows": log(1, 400)}
    if kind == "detect":
        return {"kind": kind, "frames": log(1, 32), "width": rng.randint(160, 1280), "height": rng.randint(120, 720)}
    if kind == "listen":
        return {"kind": kind, "clips": log(1, 32), "samples": log(6400, 96000), "steps": rng.randint(4, 20)}
    if kind == "chat":
        f16 = rng.random() < 0.3
        rows = log(1, 64 if f16 else 256)
        return {"kind": kind, "weights": "f16" if f16 else "q4", "layers": 4 if f16 else 32, "rows": rows, "prompt": log(4, max(5, min(600, 8192 // rows))), "steps": rng.randint(4, 8 if rows > 64 else 24)}
    model = rng.choice(["dense-4096", "dense-2048", "kaparax-4096", "kaparax-2048"])
    if kind == "prompt":
        left, lengths = log(48, 2048), []
        while left > 0 and len(lengths) < 12:
            lengths.append(rng.randint(1, left) if rng.random() < 0.6 else left)
            left -= lengths[-1]
        return {"kind": kind, "model": model, "lengths": ",".join(map(str, lengths))}
    rows = log(1, 256)
    return {"kind": kind, "model": model, "rows": rows, "context": log(16, min(1500, 65536 // rows))}


# ---------------------------------------------------------------- models

def mistral(layers):
    return tk.LlmHParams(layers, 4096, 32, 8, 128, 14336, VOCAB, 1e-5, 10000.0, 0, 0, 0, 0, 1)


def layered(name):
    """configurations of the layer-list decoders, as the benchmark has them"""
    width = int(name.split("-")[1])
    heads = width // 128

    def attention(h, kv, mask, **more):
        return dict({"heads": h, "kv_heads": kv, "dim": 128, "vdim": 128, "rot": {"dims": 64, "base": 10000.0}, "scale": 128 ** -0.5, "mask": mask}, **more)
    if name.startswith("kaparax"):
        mlp = {"kind": "dense", "ff": 14336 if width == 4096 else 8192, "limit": 7.0}
        ret = {"type": "retention", "mlp": mlp, "mixer": {"heads": heads, "dim": 128, "vdim": 128, "rot": {"dims": 128, "base": 10000.0},
                                                         "decay": [1.0 - 2.0 ** (-5 - 4.0 * i / heads) for i in range(heads)]}}
        att = {"type": "attention", "mlp": mlp, "mixer": attention(heads, heads // 4, {"size": width // 4}, conv=4, softcap=30.0)}
        return {"architecture": "Kaparax", "embedding": {"scale": float(width) ** 0.5}, "width": width, "vocab": VOCAB, "norm": {"eps": 1e-5},
                "layers": [ret, att] * (2 if width == 4096 else 4)}
    mlp = {"kind": "dense", "ff": 14336 if width == 4096 else 8192}
    left = attention(heads // 2, heads // 8, {"size": width // 4, "keep_first": 4})
    right = {"heads": heads // 2, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "conv": 4}
    layer = {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0}, "mlp": mlp}
    return {"architecture": "Vuvulorn", "width": width, "vocab": VOCAB, "norm": {"eps": 1e-5}, "layers": [layer] * (4 if width == 4096 else 8)}


# ---------------------------------------------------------------- inputs

def picture(rng, h, w):
    """smooth patches with sensor noise"""
    patch = rng.integers(0, 256, (h // 24 + 2, w // 24 + 2, 3)).astype(np.float32).repeat(24, 0).repeat(24, 1)[:h, :w]
    return np.clip(patch + rng.normal(0.0, 10.0, (h, w, 3)).astype(np.float32), 0, 255).astype(np.uint8)


def speech(rng, n):
    """voiced sound: a few harmonics under a slow envelope, and noise"""
    t = np.arange(n) / 16000.0
    f0 = rng.uniform(90, 240)
    x = sum(rng.uniform(0.2, 1.0) / k * np.sin(2 * np.pi * (k * f0 * t + rng.uniform())) for k in range(1, 9))
    x = x * (0.6 + 0.4 * np.sin(2 * np.pi * (3.0 * t + rng.uniform()))) + rng.normal(0.0, 0.05, n)
    return np.clip(6000.0 * x, -32768, 32767).astype(np.int16)


def lengths_of(case):
    return [int(v) for v in case["lengths"].split(",")]


def tokens_of(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "chat":
        return rng.integers(3, VOCAB, (case["rows"], case["prompt"])).astype(np.int32)
    ls = lengths_of(case) if case["kind"] == "prompt" else [case["context"] + 1] * case["rows"]
    return [rng.integers(3, VOCAB, n).astype(np.int32) for n in ls]


def host_inputs(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "vad":
        x = np.stack([speech(rng, 480) for _ in range(case["windows"])]).astype(np.float32) / 32768.0
        return x * rng.uniform(0.0, 1.0, (case["windows"], 1)).astype(np.float32)
    if case["kind"] == "detect":
        return [picture(rng, case["height"], case["width"]) for _ in range(case["frames"])]
    return np.stack([speech(rng, case["samples"]) for _ in range(case["clips"])])


class State:
    """keeps what a program keeps; a session is closed before its model"""

    def __init__(self, case, **have):
        self.case = case
        self.__dict__.update(have)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "vad":
        return State(case, net=tk.Vad("synthetic://vad?seed=%d" % VAD_SEED), x=host_inputs(case, seed))
    if kind == "detect":
        net = tk.ObjectDetector(model="synthetic://yolov8n?seed=%d&cls_bias=%g" % (DET_SEED, CLS_BIAS), conf=CONF, iou=IOU, max_batch=case["frames"])
        return State(case, net=net, x=host_inputs(case, seed))
    if kind == "listen":
        return State(case, net=tk.Asr(hp=tk.WHISPER_TINY_EN(), seed=ASR_SEED, max_batch=case["clips"]), x=host_inputs(case, seed))
    toks = tokens_of(case, seed)
    if kind == "chat":
        model = tk.LlmModel(mistral(case["layers"])).fill_synthetic(LLM_SEED, f16=case["weights"] == "f16")
        sess = tk.LlmSession(model, case["rows"], case["prompt"] + case["steps"] + 2)
        rows = np.arange(case["rows"], dtype=np.int32)
        return State(case, sess=sess, x=toks, seq=rows, pos=np.full(case["rows"], case["prompt"] + case["steps"], np.int32))
    model = tk.LlmModel(config=layered(case["model"]), seed=LLM_SEED, gate_rank=RANK)
    sess = tk.LlmSession(model, len(toks), max(map(len, toks)) + 8)
    ls = [len(t) for t in toks]
    if kind == "prompt":
        seq = np.repeat(np.arange(len(ls), dtype=np.int32), ls)
        pos = np.concatenate([np.arange(n, dtype=np.int32) for n in ls])
        return State(case, sess=sess, x=np.concatenate(toks), seq=seq, pos=pos, out=np.cumsum(ls).astype(np.int32) - 1)
    n, rows = case["context"], np.arange(case["rows"], dtype=np.int32)  # the sequences so far; run() takes the next position of each
    sess.forward_rows(np.repeat(rows, n), np.tile(np.arange(n, dtype=np.int32), len(ls)), np.concatenate([t[:n] for t in toks]), rows[:0], want_logits=False)
    return State(case, sess=sess, x=np.array([t[n] for t in toks], np.int32), seq=rows, pos=np.full(case["rows"], n, np.int32), out=rows)


# ---------------------------------------------------------------- one pass

def boxes_of(found, kind=np.float32):
    """[(class, score, x, y, w, h)] of each frame -> tables of fixed size"""
    out = {"count": np.array([len(f) for f in found], np.int32), "class": np.zeros((len(found), 500), np.int32), "score": np.zeros((len(found), 500), kind),
           "box": np.zeros((len(found), 500, 4), np.int32)}
    for i, f in enumerate(found):
        if f:
            t = np.array(f)
            out["class"][i, :len(f)], out["score"][i, :len(f)], out["box"][i, :len(f)] = t[:, 0], t[:, 1], t[:, 2:]
    return out


def run(state):
    case, kind = state.case, state.case["kind"]
    if kind == "vad":
        return state.net.probabilities(state.x)
    if kind == "detect":
        found = state.net.detect_batch(state.x) if case["frames"] > 1 else [state.net.detect(state.x[0])]
        return boxes_of([[(d[0], d[2]) + d[3] for d in f] for f in found])
    if kind == "listen":
        if case["clips"] == 1:  # one speaker's program also takes the sound's embedding
            ids, mel, enc, logits = state.net.transcribe_tokens(state.x, case["steps"])
            return {"ids": ids, "mel": mel, "encoder": enc, "logits": logits}
        ids, logprob = state.net.transcribe_policy(state.x, case["steps"])
        return {"ids": ids, "logprob": logprob}
    if kind == "chat":
        first = state.sess.prefill(state.x)
        ids, _ = state.sess.decode(case["rows"], case["steps"])
        logits, last = state.sess.forward(state.seq, state.pos, ids[-1])
        return {"first": first, "ids": ids, "last": last, "logits": logits}
    return state.sess.forward_rows(state.seq, state.pos, state.x, state.out)[0]


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "vad":
        n = case["windows"]
        return {"bytes": 4 * (64 * 480 + n * 481), "flops": 2 * n * 64 * 481}
    if kind == "detect":
        macs = weights = 0
        for cin, cout, k, stride, h, w in yolo_layers():
            macs += cin * cout * k * k * h * w
            weights += cin * cout * k * k
        n = case["frames"]
        return {"bytes": n * 3 * case["width"] * case["height"] + 4 * weights, "flops": 2 * n * macs}
    if kind == "listen":
        n, s, d, t, v = case["clips"], case["steps"], 384, 1500, 51864
        enc = 3000 * 400 * 402 + 3000 * 201 * 80 + 3000 * 240 * d + t * 3 * d * d + 4 * (12 * t * d * d + 2 * t * t * d) + 4 * 2 * t * d * d
        dec = 4 * (14 * d * d + 2 * t * d) + d * v
        return {"bytes": 2 * n * case["samples"] + 4 * (4 * 12 * d * d + 4 * 16 * d * d + d * v), "flops": 2 * n * (enc + s * dec)}
    if kind == "chat":
        per = case["layers"] * (4096 * 6144 + 4096 * 4096 + 3 * 4096 * 14336)
        size = 2.0 if case["weights"] == "f16" else 4.293e9 / (32 * 218103808 + VOCAB * 4096)
        rows, n, s = case["rows"], case["prompt"], case["steps"] + 1
        kv = case["layers"] * 2 * 8 * 128 * 2
        flops = 2 * rows * ((n + s) * per + (1 + s) * VOCAB * 4096 + (n * n / 2 + s * (n + s / 2)) * case["layers"] * 2 * 4096)
        return {"bytes": (1 + s) * size * (per + VOCAB * 4096) + rows * kv * (n + s * (n + s / 2)) + 4 * rows * VOCAB, "flops": flops}
    c = layered(case["model"])
    ls = lengths_of(case) if kind == "prompt" else [1] * case["rows"]
    rows, w = sum(ls), c["width"]
    reads, macs = VOCAB * w, len(ls) * VOCAB * w
    state = 0.0
    for layer in c["layers"]:
        mixers = [layer["mixer"]["left"], layer["mixer"]["right"]] if layer["type"] == "parallel" else [layer["mixer"]]
        for m in mixers:
            h, kv = m["heads"], m.get("kv_heads", m["heads"])
            dense = w * 128 * ((h + 2 * kv) + h if "mask" in m else (2 * kv + 2 * h if "conv" in m else 4 * h))
            if "conv" in m and "mask" not in m:
                dense += (w + h * 128) * 2 * RANK
            reads += dense
            macs += dense * rows
            size = (m.get("mask") or {}).get("size", 0)
            if size:
                past = [min(n / 2, size) * n if kind == "prompt" else min(case["context"], size) for n in ls]
                macs += 2 * 128 * h * sum(past)
                state += 4 * 128 * kv * (sum(past) if kind == "step" else rows)
            else:
                macs += 3 * 128 * 128 * h * rows
                state += (8 if kind == "step" else 4) * 128 * 128 * h * len(ls)
        reads += 3 * w * layer["mlp"]["ff"]
        macs += 3 * w * layer["mlp"]["ff"] * rows
    return {"bytes": 2 * reads + state + 4 * len(ls) * VOCAB, "flops": 2 * macs}


def tolerance(case):
    kind = case["kind"]
    if kind in ("vad", "detect", "listen"):
        return {"rel": 2e-5, "max": 1e-3, "differ": 0.005}  # float32 sums of a few thousand products through up to 63 layers
    if kind == "chat":
        # int8 activations and exact integer sums: another order of the float sums moves a rounding to int8 here and there (2e-3 .. 5e-3 of the logits)
        return {"rel": 2e-2, "max": 0.3, "differ": 0.01}
    return {"rel": 2e-2, "max": 0.3}  # bf16 operands, 0.002 .. 0.005 off 64 bits; where a head's output is small its norm enlarges a rounding


# ---------------------------------------------------------------- the same in 64 bits, from the mathematics

def exact(case, seed):
    kind = case["kind"]
    if kind == "vad":
        return exact_vad(case, seed)
    if kind == "detect":
        return exact_detect(case, seed) if case["frames"] <= 32 else None
    if kind == "listen":
        return exact_listen(case, seed) if case["clips"] == 1 else None  # log-probabilities of ids that only the run itself knows
    if kind == "chat":
        return None  # what comes out is defined by its roundings to int8 (or f16) on the way: 64 bits give other numbers, not better ones
    return exact_layered(case, seed)


def device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def splitmix(z):
    """splitmix64 of int64 tensors (wrapping)"""
    def lsr(v, s):
        return (v >> s) & ((1 << (64 - s)) - 1)
    z = z + (0x9E3779B97F4A7C15 - (1 << 64))
    z = (z ^ lsr(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ lsr(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ lsr(z, 31)


def wrap(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def normals(seed, tensor, n):
    """the synthetic checkpoints' numbers: sum of four 16-bit uniforms, float32"""
    start = splitmix(torch.tensor(wrap(seed ^ (tensor * 0xD6E8FEB86659FD93)), device=device()))
    h = splitmix(start + torch.arange(n, device=device()))
    s = sum((h >> k) & 0xFFFF for k in (0, 16, 32, 48))
    return (s - 131070).float() * np.float32(2.64289216e-5).item()


def f32_root(a, b):
    return float(np.sqrt(np.float32(a) / np.float32(b)))


def exact_vad(case, seed):
    x = torch.from_numpy(host_inputs(case, seed)).double().to(device())
    w1 = f32_root(1, 480) * 8 * normals(VAD_SEED, 7001, 64 * 480)
    w2 = f32_root(1, 64) * 4 * normals(VAD_SEED, 7003, 64)
    h = torch.relu(x @ w1.double().view(64, 480).T + (0.1 * normals(VAD_SEED, 7002, 64)).double())
    return torch.sigmoid(h @ w2.double() - 1.0)


# -- detector: YOLOv8n, 640 x 640

def yolo_walk(conv, pool, up, x, cat):
    """the network against any backend; conv(x, cout, k, stride, act)"""
    def c2f(x, c2, n, shortcut):
        ys = list(cat.split(conv(x, c2, 1, 1, True)))
        for _ in range(n):
            t = conv(conv(ys[-1], c2 // 2, 3, 1, True), c2 // 2, 3, 1, True)
            ys.append(cat.add(ys[-1], t) if shortcut else t)
        return conv(cat(ys), c2, 1, 1, True)
    x = conv(conv(x, 16, 3, 2, True), 32, 3, 2, True)
    x = conv(c2f(x, 32, 1, True), 64, 3, 2, True)
    f4 = c2f(x, 64, 2, True)
    f6 = c2f(conv(f4, 128, 3, 2, True), 128, 2, True)
    x = c2f(conv(f6, 256, 3, 2, True), 256, 1, True)
    ys = [conv(x, 128, 1, 1, True)]
    for _ in range(3):
        ys.append(pool(ys[-1]))
    f9 = conv(cat(ys), 256, 1, 1, True)
    h12 = c2f(cat([up(f9), f6]), 128, 1, False)
    h15 = c2f(cat([up(h12), f4]), 64, 1, False)
    h18 = c2f(cat([conv(h15, 64, 3, 2, True), h12]), 128, 1, False)
    h21 = c2f(cat([conv(h18, 128, 3, 2, True), f9]), 256, 1, False)
    heads = []
    for f in (h15, h18, h21):
        b = conv(conv(conv(f, 64, 3, 1, True), 64, 3, 1, True), 64, 1, 1, False)
        c = conv(conv(conv(f, 80, 3, 1, True), 80, 3, 1, True), 80, 1, 1, False)
        heads.append((b, c))
    return heads


class Shapes:
    """cat / split / add on (channels, height, width)"""

    def __call__(self, xs):
        return (sum(x[0] for x in xs), xs[0][1], xs[0][2])

    def split(self, y):
        return (y[0] // 2, y[1], y[2]), (y[0] // 2, y[1], y[2])

    def add(self, a, b):
        return a


class Maps:
    def __call__(self, xs):
        return torch.cat(xs, 0)

    def split(self, y):
        return y.chunk(2, 0)

    def add(self, a, b):
        return a + b


def yolo_layers():
    """(cin, cout, k, stride, height, width of the output) of the 63 convolutions in order"""
    out = []

    def conv(x, cout, k, s, act):
        h, w = (x[1] + 2 * (k // 2) - k) // s + 1, (x[2] + 2 * (k // 2) - k) // s + 1
        out.append((x[0], cout, k, s, h, w))
        return (cout, h, w)
    yolo_walk(conv, lambda x: x, lambda x: (x[0], 2 * x[1], 2 * x[2]), (3, 640, 640), Shapes())
    return out


def exact_detect(case, seed):
    layers, ws = yolo_layers(), []
    for i, (cin, cout, k, _, _, _) in enumerate(layers):
        fan = cin * k * k
        w = np.float32(f32_root(2, fan)).item() * normals(DET_SEED, 1000 + i, cout * fan)
        b = 0.05 * normals(DET_SEED, 5000 + i, cout)
        if i in (len(layers) - 1, len(layers) - 7, len(layers) - 13):
            b = b + CLS_BIAS
        ws.append((w.view(cout, k * k, cin).transpose(1, 2).reshape(cout, -1).double(), b.double()))  # [cout][cin][ky kx]
    found = [exact_boxes(yolo_maps(frame, ws)) for frame in host_inputs(case, seed)]
    sx, sy = case["width"] / 640.0, case["height"] / 640.0
    return boxes_of([[(k, s, int(x1 * sx), int(y1 * sy), int((x2 - x1) * sx), int((y2 - y1) * sy)) for s, k, x1, y1, x2, y2 in f] for f in found], np.float64)


def yolo_maps(frame, ws):
    h, w = frame.shape[:2]
    img = torch.from_numpy(frame).double().to(device()).permute(2, 0, 1)
    axes = []
    for n in (h, w):  # the preprocessor's sampling positions
        g = np.float32(np.float32(n - 1) / np.float32(640)) * np.arange(640, dtype=np.float32)
        i = g.astype(np.int32)
        axes.append((torch.from_numpy(i).long().to(device()), torch.from_numpy(np.minimum(i + 1, n - 1)).long().to(device()), torch.from_numpy((g - i).astype(np.float64)).to(device())))
    (y0, y1, dy), (x0, x1, dx) = axes
    top = img[:, y0][:, :, x0] * (1 - dx) + img[:, y0][:, :, x1] * dx
    low = img[:, y1][:, :, x0] * (1 - dx) + img[:, y1][:, :, x1] * dx
    x = top * (1 - dy)[:, None] + low * dy[:, None]
    mean, dev = (torch.tensor(v, dtype=torch.float64, device=device())[:, None, None] for v in ((0.485, 0.456, 0.406), (0.229, 0.224, 0.225)))
    x = (x / 255.0 - mean) / dev
    it = iter(ws)

    def conv(x, cout, k, s, act):
        wt, b = next(it)
        cols = torch.nn.functional.unfold(x[None], k, padding=k // 2, stride=s)[0] if k > 1 else x.reshape(x.shape[0], -1)
        side = (x.shape[1] + 2 * (k // 2) - k) // s + 1
        y = (wt @ cols + b[:, None]).view(cout, side, -1)
        return y * torch.sigmoid(y) if act else y
    return yolo_walk(conv, lambda x: torch.nn.functional.max_pool2d(x[None], 5, 1, 2)[0], lambda x: x.repeat_interleave(2, 1).repeat_interleave(2, 2), x, Maps())


def exact_boxes(heads):
    """[(score, class, x1, y1, x2, y2)] after suppression within classes, best first"""
    cand = []
    for (b, c), stride in zip(heads, (8.0, 16.0, 32.0)):
        side = b.shape[1]
        d = (torch.softmax(b.reshape(4, 16, -1), 1) * torch.arange(16, dtype=torch.float64, device=b.device)[None, :, None]).sum(1)
        gx = (torch.arange(side, device=b.device) + 0.5).repeat(side)
        gy = (torch.arange(side, device=b.device) + 0.5).repeat_interleave(side)
        s, k = torch.sigmoid(c.reshape(80, -1)).max(0)
        cand.append(torch.stack([s, k.double(), (gx - d[0]) * stride, (gy - d[1]) * stride, (gx + d[2]) * stride, (gy + d[3]) * stride], 1))
    cand = torch.cat(cand).cpu().numpy()
    cand = cand[cand[:, 0] > CONF]
    cand = cand[np.argsort(-cand[:, 0], kind="stable")][:2048]
    kept = []
    for r in cand:
        for q in kept:
            if q[1] == r[1]:
                iw, ih = min(r[4], q[4]) - max(r[2], q[2]), min(r[5], q[5]) - max(r[3], q[3])
                inter = max(iw, 0.0) * max(ih, 0.0)
                if inter > IOU * ((r[4] - r[2]) * (r[5] - r[3]) + (q[4] - q[2]) * (q[5] - q[3]) - inter):
                    break
        else:
            kept.append(r)
    return kept[:500]


# -- speech: Whisper tiny.en

def exact_listen(case, seed):
    d, heads, frames = 384, 6, 3000
    count = [3]  # tensors 0 .. 2 are the front end's tables

    def tensor(rows, cols, scale, base=0.0):
        t = base + scale * normals(ASR_SEED, 9000 + count[0], rows * cols)
        count[0] += 1
        return t.double().view(rows, cols)

    def linear(n, k):
        return tensor(n, k, f32_root(1, k))

    def bias(n):
        return tensor(1, n, 0.02)[0]

    def norm(n):
        return tensor(1, n, 0.1, 1.0)[0], tensor(1, n, 0.02)[0]

    def block():
        return {"ln1": norm(d), "q": (linear(d, d), bias(d)), "k": (linear(d, d), None), "v": (linear(d, d), bias(d)), "o": (linear(d, d), bias(d))}

    def feed(p):
        p.update({"ln2": norm(d), "fc1": (linear(4 * d, d), bias(4 * d)), "fc2": (linear(d, 4 * d), bias(d))})
        return p

    def gelu(x):
        return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))

    def layer_norm(x, p):
        return torch.nn.functional.layer_norm(x, (d,), p[0], p[1], 1e-5)

    def lin(x, p):
        return x @ p[0].T if p[1] is None else x @ p[0].T + p[1]

    def attend(q, k, v, seen=None):
        out = torch.empty_like(q)
        for i in range(0, d, 64):
            s = q[:, i:i + 64] @ k[:, i:i + 64].T / 8.0
            out[:, i:i + 64] = torch.softmax(s if seen is None else s.masked_fill(~seen, -math.inf), -1) @ v[:, i:i + 64]
        return out

    conv1, conv2 = (linear(d, 240), bias(d)), (linear(d, 3 * d), bias(d))
    count[0] += 1  # sinusoids
    enc = [feed(block()) for _ in range(4)]
    enc_ln = norm(d)
    emb = tensor(51864, d, 0.05)
    pos = tensor(448, d, 0.01)
    dec = []
    for _ in range(4):
        p = block()
        p.update({"lnx": norm(d), "xq": (linear(d, d), bias(d)), "xk": (linear(d, d), None), "xv": (linear(d, d), bias(d)), "xo": (linear(d, d), bias(d))})
        dec.append(feed(p))
    dec_ln = norm(d)

    # log-mel of the 30 s window
    pcm = np.zeros(480000)
    pcm[:case["samples"]] = host_inputs(case, seed)[0] / 32768.0
    x = np.pad(pcm, 200, mode="reflect")
    window = 0.5 - 0.5 * np.cos(2 * np.pi * np.arange(400) / 400)
    power = np.abs(np.fft.rfft(np.lib.stride_tricks.sliding_window_view(x, 400)[::160][:frames] * window, axis=1)) ** 2
    mel = np.log10(np.maximum(power @ mel_filters().T, 1e-10))
    mel = (np.maximum(mel, mel.max() - 8.0) + 4.0) / 4.0
    ml = torch.from_numpy(mel).to(device())

    def taps(x, stride):  # [T][C] -> [T / stride][3 C]
        z = torch.nn.functional.pad(x, (0, 0, 1, 1))
        return torch.cat([z[k:k + x.shape[0]:stride] for k in range(3)], 1)
    x = gelu(lin(taps(gelu(lin(taps(ml, 1), conv1)), 2), conv2))
    ang = torch.arange(1500, dtype=torch.float64)[:, None] * torch.exp(-math.log(10000.0) / 191 * torch.arange(192, dtype=torch.float64))[None]
    x = x + torch.cat([torch.sin(ang), torch.cos(ang)], 1).to(device())
    for p in enc:
        h = layer_norm(x, p["ln1"])
        x = x + lin(attend(lin(h, p["q"]), lin(h, p["k"]), lin(h, p["v"])), p["o"])
        x = x + lin(gelu(lin(layer_norm(x, p["ln2"]), p["fc1"])), p["fc2"])
    states = layer_norm(x, enc_ln)
    x = emb[[50257, 50362]] + pos[:2]  # <|startoftranscript|><|notimestamps|>: the logits after the second are the first that count
    past = torch.ones(2, 2, dtype=torch.bool, device=x.device).tril()
    for p in dec:
        h = layer_norm(x, p["ln1"])
        x = x + lin(attend(lin(h, p["q"]), lin(h, p["k"]), lin(h, p["v"]), past), p["o"])
        h = layer_norm(x, p["lnx"])
        x = x + lin(attend(lin(h, p["xq"]), lin(states, p["xk"]), lin(states, p["xv"])), p["xo"])
        x = x + lin(gelu(lin(layer_norm(x, p["ln2"]), p["fc1"])), p["fc2"])
    return {"ids": None, "mel": ml[None], "encoder": states[None], "logits": layer_norm(x[1:], dec_ln) @ emb.T}


def mel_filters():
    """80 triangles on the Slaney scale up to 8 kHz, each of unit area"""
    hz = np.fft.rfftfreq(400, 1 / 16000.0)
    top = 15.0 + math.log(8.0) / (math.log(6.4) / 27.0)
    m = np.linspace(0.0, top, 82)
    pts = np.where(m < 15.0, m * 200.0 / 3.0, 1000.0 * np.exp(math.log(6.4) / 27.0 * (m - 15.0)))
    up = (hz[None] - pts[:80, None]) / (pts[1:81] - pts[:80])[:, None]
    down = (pts[2:, None] - hz[None]) / (pts[2:] - pts[1:81])[:, None]
    return np.maximum(np.minimum(up, down), 0.0) * (2.0 / (pts[2:] - pts[:80]))[:, None]


# -- layer-list decoders

class Weights:
    """the random weights of a configuration, tensor by tensor in the order in which the model makes them"""

    def __init__(self, seed):
        self.seed, self.count = seed, 0

    def matrix(self, rows, cols):
        self.count += 1
        z = wrap(self.seed + 0x1000003 * self.count) + (0x9E3779B97F4A7C15 - (1 << 64)) * torch.arange(1, rows * cols + 1, device=device())
        z = splitmix(z - (0x9E3779B97F4A7C15 - (1 << 64)))
        u = ((z >> 40) & 0xFFFFFF).float() * (2.0 / 16777216.0) - 1.0
        return (u * f32_root(3, cols)).bfloat16().double().view(rows, cols)

    def values(self, n, lo, hi):
        """a linear congruential run, by its closed form over the indices"""
        self.count += 1
        idx = torch.arange(1, n + 1, device=device())
        z = torch.full((n,), wrap(self.seed + 0x1000003 * self.count), device=device())
        a, c = 6364136223846793005, 1442695040888963407
        for bit in range(max(1, n).bit_length()):
            z = torch.where((idx >> bit) & 1 == 1, z * wrap(a) + wrap(c), z)
            a, c = a * a & ((1 << 64) - 1), (a + 1) * c & ((1 << 64) - 1)
        return float(np.float32(lo)) + float(np.float32(hi) - np.float32(lo)) * ((z >> 40) & 0xFFFFFF).float() / 16777216.0

    def vector(self, n, lo, hi):
        return self.values(n, lo, hi).double()


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def rotate(x, dims, base):
    """[T][heads][dim]"""
    half = dims // 2
    ang = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * base ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dims)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def conv_past(x, taps):
    """[T][C] with [C][n]: every position and the n - 1 before it"""
    n = taps.shape[1]
    z = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
    return sum(taps[:, j] * z[j:j + x.shape[0]] for j in range(n))


def attend_masked(q, k, v, scale, mask, cap):
    per = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=torch.float64, device=q.device)
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // per].T * scale
        s = cap * torch.tanh(s / cap) if cap else s
        out[:, h] = torch.softmax(s.masked_fill(~mask, -math.inf), -1) @ v[:, h // per]
    return out


def exact_layered(case, seed):
    c, toks = layered(case["model"]), tokens_of(case, seed)
    if sum(len(t) for t in toks) > 15000:
        return None  # a token-by-token recurrence of that many steps takes too long here
    w, W, eps = c["width"], Weights(LLM_SEED), c["norm"]["eps"]
    kap = c["architecture"] == "Kaparax"
    table = W.values(VOCAB * w, -1.7, 1.7).bfloat16().view(VOCAB, w)
    xs = [table[torch.from_numpy(t).long().to(device())].double() * (c["embedding"]["scale"] if kap else 1.0) for t in toks]
    del table

    def norm_params():
        return (W.vector(w, 0.8, 1.2), W.vector(w, -0.1, 0.1)) if kap else (W.vector(w, 0.8, 1.2), None)

    def norm(x, p):
        if kap:
            return torch.nn.functional.layer_norm(x, (w,), p[0], p[1], eps)
        return rms(x, eps) * p[0]

    for layer in c["layers"]:
        mixers = [layer["mixer"]] if kap else [layer["mixer"]["left"], layer["mixer"]["right"]]
        made = [(attention_of if "mask" in m else retention_of if "decay" in m else delta_of)(W, m, w, eps, kap) for m in mixers]
        pre1 = norm_params() if kap else None
        norm1 = norm_params()
        pre2 = norm_params() if kap else None
        norm2 = norm_params()
        f = layer["mlp"]
        gate, up, down = W.matrix(f["ff"], w), W.matrix(f["ff"], w), W.matrix(w, f["ff"])
        for i, x in enumerate(xs):
            h = norm(x, pre1) if kap else x
            x = x + norm(sum(m(h) for m in made), norm1)
            h = norm(x, pre2) if kap else x
            g, u = h @ gate.T, h @ up.T
            if kap:
                g, u = g.clamp(max=f["limit"]), u.clamp(-f["limit"], f["limit"])
                y = (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ down.T
            else:
                y = (g * torch.sigmoid(g) * u) @ down.T
            xs[i] = x + norm(y, norm2)
        del gate, up, down, made
    final = norm_params()
    head = W.matrix(VOCAB, w)
    return torch.stack([norm(x[-1:], final)[0] @ head.T for x in xs])


def attention_of(W, m, w, eps, kap):
    hq, hk = m["heads"], m["kv_heads"]
    wq, wk, wv, wo = W.matrix(hq * 128, w), W.matrix(hk * 128, w), W.matrix(hk * 128, w), W.matrix(w, hq * 128)
    if kap:
        extra = [W.vector(n * 4, -0.9, 0.9).view(n, 4) for n in (hq * 128, hk * 128, hk * 128)]
    else:
        extra = [W.vector(n, -0.1, 0.1) for n in (hq * 128, hk * 128, hk * 128, w)] + [W.vector(128, 0.8, 1.2), W.vector(128, 0.8, 1.2)]

    def go(h):
        t, size = h.shape[0], m["mask"]["size"]
        q, k, v = h @ wq.T, h @ wk.T, h @ wv.T
        if kap:
            q, k, v = (conv_past(z, e) for z, e in zip((q, k, v), extra))
        else:
            q, k, v = q + extra[0], k + extra[1], v + extra[2]
        q, k, v = q.view(t, hq, 128), k.view(t, hk, 128), v.view(t, hk, 128)
        if not kap:
            q, k = rms(q, eps) * extra[4], rms(k, eps) * extra[5]
        q, k = (rotate(z, m["rot"]["dims"], m["rot"]["base"]) for z in (q, k))
        i = torch.arange(t, device=h.device)
        i, j = i[:, None], i[None]
        mask = (j <= i) & (i // size == j // size) if kap else (j <= i) & ((i - j < size) | (j < m["mask"]["keep_first"]))
        y = attend_masked(q, k, v, m["scale"], mask, m.get("softcap")).reshape(t, -1) @ wo.T
        return y if kap else y + extra[3]
    return go


def retention_of(W, m, w, eps, kap):
    n = m["heads"]
    wq, wk, wv, wg = (W.matrix(n * 128, w) for _ in range(4))
    wo = W.matrix(w, n * 128)

    def go(h):
        t = h.shape[0]
        q, k, v = ((h @ z.T).view(t, n, 128) for z in (wq, wk, wv))
        q, k = (rotate(z, m["rot"]["dims"], m["rot"]["base"]) for z in (q, k))
        gap = torch.arange(t, device=h.device)[:, None] - torch.arange(t, device=h.device)[None]
        out = torch.empty_like(v)
        for i in range(n):
            fade = torch.where(gap >= 0, m["decay"][i] ** gap.clamp(min=0).double(), torch.zeros((), dtype=torch.float64, device=h.device))
            out[:, i] = (q[:, i] @ k[:, i].T * 128 ** -0.5 * fade) @ v[:, i]
        g = h @ wg.T
        return (rms(out, eps).reshape(t, -1) * g * torch.sigmoid(g)) @ wo.T
    return go


def delta_of(W, m, w, eps, kap):
    n, kv = m["heads"], m["kv_heads"]
    wq, wk, wv, wb = W.matrix(kv * 128, w), W.matrix(kv * 128, w), W.matrix(n * 128, w), W.matrix(n, w)
    a1, g1, a2, g2, wo = W.matrix(RANK, w), W.matrix(RANK, w), W.matrix(n * 128, RANK), W.matrix(n * 128, RANK), W.matrix(w, n * 128)
    cq, ck, cv = (W.vector(r * 4, -0.9, 0.9).view(r, 4) for r in (kv * 128, kv * 128, n * 128))
    a_log, dt, gain = W.vector(n, 0.0, 2.7), W.vector(n * 128, -6.0, -2.0), W.vector(128, 0.8, 1.2)

    def go(h):
        t = h.shape[0]

        def mixed(z, taps, heads):
            z = conv_past(h @ z.T, taps)
            return (z * torch.sigmoid(z)).view(t, heads, 128)

        def unit(z):
            return z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
        q, k, v = unit(mixed(wq, cq, kv)) * 128 ** -0.5, unit(mixed(wk, ck, kv)), mixed(wv, cv, n)
        q, k = q.repeat_interleave(n // kv, 1), k.repeat_interleave(n // kv, 1)
        beta = torch.sigmoid(h @ wb.T)
        fade = torch.exp(-torch.exp(a_log)[None, :, None] * torch.nn.functional.softplus((h @ a1.T) @ a2.T + dt).view(t, n, 128))
        S = torch.zeros(n, 128, 128, dtype=torch.float64, device=h.device)
        out = torch.empty_like(v)
        for i in range(t):
            S = S * fade[i][:, :, None]
            u = beta[i][:, None] * (v[i] - (S * k[i][:, :, None]).sum(1))
            S = S + k[i][:, :, None] * u[:, None]
            out[i] = (S * q[i][:, :, None]).sum(1)
        gate = torch.sigmoid((h @ g1.T) @ g2.T).view(t, n, 128)
        return (rms(out, eps) * gain * gate).reshape(t, -1) @ wo.T
    return go
