"""What a user of this framework has it do, as cases that can be timed: the byte model's streaming step and its
teacher-forced scoring, compression and decompression of chunks (the path under BOA files and the codec API), the range
coder on precomputed tables, and the per-step batch coder.  Models are random-init (fixed seed) in the shapes that the
configurations, tests and benchmark of this repository use: d_model 256 with 1 to 8 layers, d_model 512 with 16 layers
and bfloat16 weights.  The data are the benchmark's kinds: float32 records, mixed int16 / float32 records, and symbols
drawn from tables.

Inputs come from the seed alone.  A loaded model (weights on the GPU, engine) is kept between preparations of the same
case, as a program keeps the model it has loaded; nothing that depends on the inputs is kept.
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (REPO, os.path.join(REPO, "boa-constrictor_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import codec  # noqa: E402
import gpu_range_coder  # noqa: E402
import model as boa_model  # noqa: E402
from boa_amd import _native as nat  # noqa: E402

VOCAB, D_STATE = 256, 16


def listed():
    return [
        # one byte at a time for one stream: the streaming predictor (default model of the constructor, 4 layers)
        {"name": "step_1x4L", "kind": "step", "d": 256, "layers": 4, "precision": "f32", "lanes": 1},
        # scoring a batch of texts: next-byte logits of every position (the teacher-forced forward)
        {"name": "forward_8x500_bf16x3", "kind": "forward", "d": 256, "layers": 8, "precision": "bf16x3", "lanes": 8,
         "length": 500, "last": 500},
        # a single small message or file, one chunk
        {"name": "compress_1x1000", "kind": "compress", "d": 256, "layers": 8, "precision": "f32", "lanes": 1,
         "length": 1000, "last": 1000},
        # the chunk count of the CPU reference configuration, with a shorter last chunk
        {"name": "compress_64x1500", "kind": "compress", "d": 256, "layers": 8, "precision": "f32", "lanes": 64,
         "length": 1500, "last": 1111},
        # the headline's 4096 chunks (shorter ones: the rate does not depend on it)
        {"name": "compress_4096x512", "kind": "compress", "d": 256, "layers": 8, "precision": "f32", "lanes": 4096,
         "length": 512, "last": 400},
        # the larger model with bfloat16 weights
        {"name": "compress_d512_1000x257", "kind": "compress", "d": 512, "layers": 16, "precision": "bf16w",
         "lanes": 1000, "length": 257, "last": 99},
        # decompression: the CPU configuration's 64 chunks, the command line's default of 1000 chunks in the split
        # mode, the headline's 4096, and the larger model
        {"name": "decompress_64x500", "kind": "decompress", "d": 256, "layers": 8, "precision": "f32", "lanes": 64,
         "length": 500, "last": 345},
        {"name": "decompress_1000x300_bf16x3", "kind": "decompress", "d": 256, "layers": 8, "precision": "bf16x3",
         "lanes": 1000, "length": 300, "last": 150},
        {"name": "decompress_4096x257", "kind": "decompress", "d": 256, "layers": 8, "precision": "f32", "lanes": 4096,
         "length": 257, "last": 257},
        {"name": "decompress_d512_1000x65", "kind": "decompress", "d": 512, "layers": 16, "precision": "bf16w",
         "lanes": 1000, "length": 65, "last": 33},
        # the range coder alone on quantised tables: the coded bytes of 1024-byte chunks (the first byte is not coded)
        {"name": "tables_16384x1023", "kind": "tables", "lanes": 16384, "length": 1023, "bits": 16, "entry_bytes": 2},
        # the per-step batch coder: probabilities in, symbols out, as an external model drives it
        {"name": "batch_coder_1000x24", "kind": "batch_coder", "lanes": 1000, "length": 24, "symbols": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "forward", "compress", "compress", "decompress", "decompress", "tables", "batch_coder"])
    if kind == "tables":
        bits, entry = rng.choice([(16, 2), (16, 4), (24, 4)])
        lanes = _log(rng, 1, 16384)
        most = 8192 * 1023 * 2 // (lanes * entry)
        return {"kind": kind, "lanes": lanes, "length": _log(rng, 5, max(6, min(4096, most))), "bits": bits,
                "entry_bytes": entry}
    if kind == "batch_coder":
        return {"kind": kind, "lanes": _log(rng, 1, 4096), "length": _log(rng, 2, 24),
                "symbols": rng.choice([256, 256, rng.randint(2, 1024)])}
    if rng.random() < 0.2:
        c = {"kind": kind, "d": 512, "layers": rng.choice([2, 16]), "precision": "bf16w"}
    else:
        c = {"kind": kind, "d": 256, "layers": rng.randint(1, 8), "precision": rng.choice(["f32", "f32", "bf16x3"])}
    if kind == "step":
        c["lanes"] = _log(rng, 1, 1024)
        return c
    size = c["layers"] * c["d"] * c["d"]  # weights of the layers, in units of the tested model's 8 x 256 x 256
    share = min(1.0, 8 * 256 * 256 / size)
    if kind == "decompress":
        c["lanes"] = _log(rng, 1, 4096 if c["d"] == 256 else 1000)
        longest = 257 * share
    else:
        c["lanes"] = _log(rng, 1, 4096 if kind == "compress" else 256)
        longest = min(2000 * share, 4096 * 257 * share / c["lanes"])
    c["length"] = _log(rng, 17, max(18, int(longest)))
    c["last"] = rng.randint(1, c["length"]) if kind != "forward" else c["length"]
    return c


@functools.lru_cache(maxsize=1)
def _loaded(d, layers, precision, lanes, tile):
    """A model as a program holds it: weights loaded, engine ready for its batch size."""
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(layers)
        m = boa_model.BoaConstrictor(d_model=d, num_layers=layers, vocab_size=VOCAB)
    m.precision = precision
    m.eval()
    if tile:
        m.engine(lanes, tile)
    return m


def _model(case):
    kind, n = case["kind"], case.get("length", 1)
    tile = {"step": 0, "decompress": 1}.get(kind, min(boa_model.DEFAULT_TILE_LEN, max(n - 1 if kind == "compress" else n, 1)))
    if kind == "decompress":  # the payload to decompress is compressed first, with the same model
        tile = min(boa_model.DEFAULT_TILE_LEN, max(n - 1, 1))
    return _loaded(case["d"], case["layers"], case["precision"], case["lanes"], tile)


def _records(nbytes, rng, mixed):
    """Float32 records (four log-normal energies, three normal coordinates, one integer id), or int16 and float32
    records in turn."""
    n = nbytes // 32 + 1
    rec = np.empty((n, 8), dtype="<f4")
    rec[:, 0:4] = rng.lognormal(1.0, 1.5, (n, 4))
    rec[:, 4:7] = rng.standard_normal((n, 3))
    rec[:, 7] = rng.integers(-(1 << 31), 1 << 31, n, dtype=np.int64).astype(np.int32).view(np.float32)
    if mixed:
        half = np.clip(rng.normal(0.0, 300.0, (n, 8)), -32768, 32767).astype("<i2").view("<f4")
        rec[:, 4:8] = half
    return rec.reshape(-1).view(np.uint8)[:nbytes]


def _chunks(case, seed):
    n, length = case["lanes"], case["length"]
    data = _records((n - 1) * length + case["last"], np.random.default_rng([seed, 1]), case["d"] == 512)
    return [data[i * length:(i + 1) * length] for i in range(n)]


def _room(length):
    """Code words that a chunk of this length has room for in the program's file buffer: these models and tables code
    a byte in about 8 bits, a quarter of a word."""
    return length // 3 + 8


def prepare(case, seed):
    kind, n = case["kind"], case["lanes"]
    if kind == "tables":
        T, K = case["length"], VOCAB
        dt = torch.int16 if case["entry_bytes"] == 2 else torch.int32
        s = {"cdf": torch.empty((n, T, K), dtype=dt, device="cuda"),
             "syms": torch.empty((n, T), dtype=torch.uint8, device="cuda"),
             "words": torch.zeros((n, T + 8), dtype=torch.int32, device="cuda"),
             "nwords": torch.zeros(n, dtype=torch.int32, device="cuda"),
             "back": torch.zeros((n, T), dtype=torch.uint8, device="cuda")}
        nat.check(nat.lib().rc_synth_tables(ctypes.c_uint64(seed + 1), 3.0, case["bits"], case["entry_bytes"], K, n, T,
                                            nat.ptr(s["cdf"]), nat.ptr(s["syms"]), nat.stream_ptr()))
        return {"case": case, **s}
    if kind == "batch_coder":
        g = torch.Generator(device="cuda").manual_seed(seed)
        T, K = case["length"], case["symbols"]
        probs = torch.softmax(3.0 * torch.randn((T, n, K), generator=g, device="cuda"), dim=-1)
        syms = torch.multinomial(probs.view(T * n, K), 1, generator=g).view(T, n).to(torch.int32)
        return {"case": case, "probs": probs, "syms": syms, "file": np.zeros(n * _room(T), np.int32),
                "back": torch.zeros((T, n), dtype=torch.int32, device="cuda")}
    m = _model(case)
    if kind == "step":
        tok = torch.from_numpy(np.random.default_rng([seed, 2]).integers(0, VOCAB, n).astype(np.int32)).cuda()
        return {"case": case, "model": m, "stream": m.init_stream(max_len=1 << 30, batch_size=n), "tokens": tok}
    chunks = _chunks(case, seed)
    if kind == "forward":
        return {"case": case, "model": m, "tokens": torch.from_numpy(np.stack(chunks)).to(torch.int32).cuda()}
    if kind == "compress":
        return {"case": case, "model": m, "chunks": chunks, "file": np.zeros(n * _room(case["length"]), np.int32)}
    payload, nwords, first, lens = codec.compress_payload(m, chunks)
    return {"case": case, "model": m, "payload": payload, "nwords": nwords, "first": first, "lens": lens}


def run(state):
    case = state["case"]
    kind, n = case["kind"], case["lanes"]
    if kind == "step":
        return state["model"].step(state["tokens"], state["stream"])
    if kind == "forward":
        return state["model"].forward(state["tokens"])
    if kind == "compress":
        payload, nwords, first, _ = codec.compress_payload(state["model"], state["chunks"])
        state["file"][:payload.size] = payload.view(np.int32)
        return {"payload": state["file"], "nwords": nwords, "first": np.frombuffer(bytes(first), np.uint8)}
    if kind == "decompress":
        out = codec.decompress_payload(state["model"], state["payload"], state["nwords"], state["lens"], state["first"])
        # bytes past a chunk's end are not written: each chunk's own bytes, back to back, are the file
        return np.concatenate([out[:-1].reshape(-1), out[-1, :state["lens"][-1]]])
    if kind == "tables":
        lib, bits, eb, T, pitch = nat.lib(), case["bits"], case["entry_bytes"], case["length"], state["words"].shape[1]
        cdf, syms, words, nwords, back = (nat.ptr(state[k]) for k in ("cdf", "syms", "words", "nwords", "back"))
        nat.check(lib.rc_encode_tables(bits, eb, cdf, VOCAB, syms, n, T, words, pitch, nwords, nat.stream_ptr()))
        nat.check(lib.rc_decode_tables(bits, eb, cdf, VOCAB, words, pitch, nwords, n, T, back, nat.stream_ptr()))
        return {"words": state["words"], "nwords": state["nwords"], "back": state["back"]}
    T, K, coder = case["length"], case["symbols"], gpu_range_coder.gpu.queue.RangeCoderBatch
    enc = coder(n, K, T)
    for t in range(T):
        enc.encode_step(state["syms"][t], state["probs"][t])
    enc.finalize()
    streams = enc.get_compressed_list()
    dec = coder(n, K, T)
    dec.load_compressed_list(streams)
    dec.init_decoder()
    for t in range(T):
        dec.decode_step(state["probs"][t], state["back"][t])
    sizes = np.array([len(s) for s in streams])
    state["file"][:sizes.sum()] = np.concatenate(streams).view(np.int32)
    return {"words": state["file"], "sizes": sizes, "back": state["back"]}


def _shape(case):
    d = case["d"]
    return d, 2 * d, -(-d // 16), case["layers"]


def work(case):
    kind, n, T = case["kind"], case["lanes"], case.get("length", 1)
    if kind == "tables":  # every table row once in each direction, the symbols and (about 5.5 bits each) their code
        rows = n * T
        return {"bytes": 2 * rows * (VOCAB * case["entry_bytes"] + 1.7), "flops": 2 * rows * 8}
    if kind == "batch_coder":  # the probabilities once in each direction; their sum
        rows = n * T
        return {"bytes": 2 * rows * (4 * case["symbols"] + 4.7), "flops": 2 * rows * 2 * case["symbols"]}
    d, di, r, layers = _shape(case)
    params = layers * (2 * di * d + (r + 2 * D_STATE) * di + r * di + d * di + 8 * d * d) + d * d + VOCAB * d
    scan = layers * di * (6 * D_STATE + 8 + 8)
    weights = params * (2 if case["precision"] == "bf16w" else 4)
    if kind == "step":  # the state of every stream is read and written too
        state = 2 * n * layers * di * 4 * (D_STATE + 3)
        return {"bytes": weights + state + n * (4 + 4 * VOCAB), "flops": n * (2 * params + scan)}
    last = case["last"]
    if kind == "forward":
        return {"bytes": weights + n * T * (4 + 4 * VOCAB), "flops": n * T * (2 * params + scan)}
    # bytes in and code words out, or the reverse: about as many for these records; the model runs on every byte but
    # the last of its chunk
    total = (n - 1) * T + last
    return {"bytes": weights + 2 * total, "flops": max(1, total - n) * (2 * params + scan)}


def tolerance(case):
    # code words, symbols and bytes are whole numbers: the coder is exact, and files have to stay readable
    if case["kind"] not in ("step", "forward"):
        return "exact"
    # logits: float32 sums in another order, or products of operands of about 16 significant bits
    return {"rel": 2.5e-6} if case["precision"] == "f32" else {"rel": 3.2e-5}


def exact(case, seed):
    """The logits in 64 bits: the model written out in plain torch."""
    if case["kind"] not in ("step", "forward"):
        return None
    s = prepare(case, seed)
    # the matrices of bfloat16 weights are rounded when they are loaded, whatever the arithmetic
    mats = ("in_proj.weight", "x_proj.weight", "out_proj.weight", "ff.0.weight", "ff.2.weight", "head.0.weight",
            "head.2.weight")
    w = {k: (v.bfloat16() if case["precision"] == "bf16w" and k.endswith(mats) else v).cuda().double()
         for k, v in s["model"].state_dict().items()}
    tok = s["tokens"].long()
    tok = tok[:, None] if tok.ndim == 1 else tok
    B, T = tok.shape
    d, di, r, layers = _shape(case)
    x = w["embedding.weight"][tok]
    for i in range(layers):
        p = "blocks.%d." % i
        m = p + "mamba."
        xz = F.linear(F.layer_norm(x, (d,), w[p + "ln1.weight"], w[p + "ln1.bias"]), w[m + "in_proj.weight"])
        u, z = xz[..., :di], xz[..., di:]
        past = F.pad(u, (0, 0, 3, 0))
        taps = w[m + "conv1d.weight"][:, 0, :]
        u = F.silu(sum(past[:, k:k + T] * taps[:, k] for k in range(4)) + w[m + "conv1d.bias"])
        dbc = F.linear(u, w[m + "x_proj.weight"])
        dt = F.softplus(F.linear(dbc[..., :r], w[m + "dt_proj.weight"], w[m + "dt_proj.bias"]))
        A = -torch.exp(w[m + "A_log"])
        h = torch.zeros((B, di, D_STATE), dtype=torch.float64, device="cuda")
        ys = []
        for t in range(T):
            step = dt[:, t, :, None]
            h = torch.exp(step * A) * h + (step * u[:, t, :, None]) * dbc[:, t, None, r:r + D_STATE]
            ys.append((h * dbc[:, t, None, r + D_STATE:]).sum(-1))
        y = (torch.stack(ys, 1) + w[m + "D"] * u) * F.silu(z)
        y = F.linear(y, w[m + "out_proj.weight"])
        y = F.layer_norm(y, (d,), w[p + "ln2.weight"], w[p + "ln2.bias"])
        y = F.gelu(F.linear(y, w[p + "ff.0.weight"], w[p + "ff.0.bias"]))
        x = x + F.linear(y, w[p + "ff.2.weight"], w[p + "ff.2.bias"])
    x = F.linear(F.relu(F.linear(x, w["head.0.weight"], w["head.0.bias"])), w["head.2.weight"], w["head.2.bias"])
    return x[:, 0] if case["kind"] == "step" else x
