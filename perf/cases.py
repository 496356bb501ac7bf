"""Performance cases of the codec: what its users have it do, through the
public entry points (the C ABI by way of its Python binding), over the range
of models, lane counts and lengths that they run.

A case is one pass of one of five paths:

  compress    data in HBM -> one coded stream per chunk in HBM (teacher-forced
              forward, CDF, range coder, compaction)
  decompress  those streams -> the data (one model step per byte and lane)
  file_compress, file_decompress
              the same through host buffers and the container
  forward     teacher-forced scoring: tokens of every lane -> logits
  step        streaming: a few single-token steps of every lane -> logits

with a model (d_model, n_layers, d_state, precision), `chunks` chunks of
`chunk` bytes of which the last has `last`, and at most `lanes` of them in
flight.  Streams, containers and decoded bytes are exact: a container
written before a change has to decode after it.
"""
import importlib
import math

import numpy as np
import torch

boa = importlib.import_module("boa-constrictor_amd.boa_hip")

# (d_model, n_layers, d_state, precision), the repository's models: the small
# one, its one-layer sibling of an odd width, the headline model in both
# precisions, and the large one
MODELS = {
    "d64": (64, 2, 16, "fp32"),
    "d80": (80, 1, 16, "fp32"),
    "d256": (256, 8, 16, "fp32"),
    "d256b": (256, 8, 16, "bf16"),
    "d512b": (512, 12, 32, "bf16"),
}


def _case(name, path, model, chunks, chunk, last, lanes):
    c = {"path": path, "model": model, "chunks": chunks, "chunk": chunk, "last": last,
         "lanes": lanes}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a stream coded live, byte by byte, with the small model: latency of
        # a chain of short launches
        _case("step_d64", "step", "d64", 64, 8, 8, 64),
        # one mebibyte file in 16 KiB chunks, host buffer to container
        _case("file_compress_d64", "file_compress", "d64", 64, 16384, 16384, 64),
        # a small container read back
        _case("file_decompress_d64", "file_decompress", "d64", 61, 2048, 1777, 64),
        # files with the odd-width model, more chunks than lanes: two whole
        # batches and a short one
        _case("compress_d80", "compress", "d80", 1100, 3001, 700, 512),
        # scoring a few ragged texts with the headline model
        _case("forward_d256", "forward", "d256", 37, 219, 219, 37),
        # the headline: a thousand chunks, fp32, there and back (chunks cut
        # short of their 64 KiB; a forward tile is 1600 tokens)
        _case("compress_d256", "compress", "d256", 1000, 2085, 1999, 1000),
        _case("decompress_d256", "decompress", "d256", 1000, 257, 200, 1000),
        # decoding a large archive, fp32: four thousand lanes
        _case("decompress_d256_4k", "decompress", "d256", 4096, 97, 97, 4096),
        # the same model in bf16 at a large archive's lane count
        _case("compress_d256_bf16", "compress", "d256b", 8192, 512, 512, 8192),
        _case("decompress_d256_bf16", "decompress", "d256b", 8192, 97, 50, 8192),
        # the large bf16 model
        _case("compress_d512_bf16", "compress", "d512b", 4096, 256, 255, 4096),
        _case("decompress_d512_bf16", "decompress", "d512b", 4096, 49, 49, 4096),
    ]


# For draw(): the paths by how often they are run, and per model the lane
# counts it is run at, the most tokens of a forward or compress call and the
# most steps of a decode call (no drawn case costs more than a listed one).
_PATHS = ["compress"] * 5 + ["decompress"] * 5 + ["file_compress", "file_decompress"] + \
    ["forward"] * 2 + ["step"]
_RANGES = {
    "d64": (1, 1024, 2 << 20, 3000),
    "d80": (1, 1024, 2 << 20, 800),
    "d256": (8, 4096, 1 << 20, 256),
    "d256b": (64, 8192, 3 << 20, 128),
    "d512b": (64, 4096, 3 << 18, 40),
}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(_PATHS)
    model = rng.choice(["d64", "d80", "d256", "d256", "d256b", "d256b", "d512b"])
    lo, hi, tokens, steps = _RANGES[model]
    chunks = _log_int(rng, lo, hi)
    if path == "step":
        return _case(None, path, model, chunks, *(2 * [rng.randint(4, 12)]), chunks)
    if path == "forward":  # logits come back whole: 1 KB a token
        chunk = _log_int(rng, 1, max(1, min(4096, (tokens // 8) // chunks)))
        return _case(None, path, model, chunks, chunk, chunk, chunks)
    if path.endswith("decompress"):
        chunk = _log_int(rng, max(2, steps // 8), steps)
    else:
        chunk = _log_int(rng, 32, max(33, min(32768, tokens // chunks)))
    # now and then fewer lanes in flight than chunks
    lanes = max(1, (chunks + 2) // 3) if rng.random() < 0.2 and not path.endswith("decompress") \
        else chunks
    return _case(None, path, model, chunks, chunk, rng.randint(1, chunk), lanes)


# ------------------------------------------------------------------ inputs
def _dims(case):
    d, L, ds, prec = MODELS[case["model"]]
    r = (d + 15) // 16
    return d, L, ds, prec, 2 * d, r, r + 2 * ds


def _weights(case, seed):
    """Mamba-style random init in file order, {name: float32 tensor} on the GPU."""
    d, L, ds, _, di, r, R = _dims(case)
    g = torch.Generator("cuda").manual_seed(1000 + seed)
    t = {}

    def uni(name, shape, bound):
        t[name] = (torch.rand(shape, generator=g, device="cuda") * 2 - 1) * bound

    def full(name, shape, v):
        t[name] = torch.full(shape, float(v), device="cuda")

    t["emb"] = torch.randn((256, d), generator=g, device="cuda")
    for i in range(L):
        p = "%d." % i
        full(p + "ln1.w", (d,), 1)
        full(p + "ln1.b", (d,), 0)
        uni(p + "in.w", (2 * di, d), d ** -0.5)
        full(p + "in.b", (2 * di,), 0)
        uni(p + "conv.w", (di, 4), 0.5)
        uni(p + "conv.b", (di,), 0.5)
        uni(p + "x.w", (R, di), di ** -0.5)
        uni(p + "dt.w", (di, r), r ** -0.5)
        dt = torch.exp(math.log(1e-3) + math.log(100.0)
                       * torch.rand((di,), generator=g, device="cuda"))
        t[p + "dt.b"] = dt + torch.log(-torch.expm1(-dt))
        t[p + "alog"] = torch.log(torch.arange(1, ds + 1, device="cuda").float()).repeat(di, 1)
        full(p + "D", (di,), 1)
        uni(p + "out.w", (d, di), di ** -0.5)
        full(p + "out.b", (d,), 0)
        full(p + "ln2.w", (d,), 1)
        full(p + "ln2.b", (d,), 0)
        uni(p + "ff0.w", (4 * d, d), d ** -0.5)
        uni(p + "ff0.b", (4 * d,), d ** -0.5)
        uni(p + "ff2.w", (d, 4 * d), (4 * d) ** -0.5)
        uni(p + "ff2.b", (d,), (4 * d) ** -0.5)
    uni("h0.w", (d, d), d ** -0.5)
    uni("h0.b", (d,), d ** -0.5)
    uni("h2.w", (256, d), d ** -0.5)
    uni("h2.b", (256,), d ** -0.5)
    return t


def _n_bytes(case):
    return (case["chunks"] - 1) * case["chunk"] + case["last"]


def _data(case, seed):
    """Little-endian float32 records, rounded as an instrument writes them:
    half Gaussian, half exponential fields."""
    n = _n_bytes(case)
    g = torch.Generator("cuda").manual_seed(seed)
    k = (n + 7) // 8
    a = torch.randn((k,), generator=g, device="cuda")
    b = -10.0 * torch.log1p(-torch.rand((k,), generator=g, device="cuda"))
    v = torch.stack([torch.round(a * 1000) / 1000, b], 1).contiguous()
    return v.view(torch.uint8).reshape(-1)[:n].contiguous()


def _codec(case, seed):
    d, L, ds, prec, *_ = _dims(case)
    codec = boa.Codec(d, L, ds, max_lanes=case["lanes"], precision=prec)
    codec.set_stream(torch.cuda.current_stream().cuda_stream)
    flat = torch.cat([v.reshape(-1) for v in _weights(case, seed).values()]).cpu().numpy()
    blob = b"BOA\x00" + flat.tobytes()
    rc = boa.lib().boa_load_weights_mem(codec.h, blob, len(blob))
    if rc:
        raise RuntimeError("load_weights_mem: %d" % rc)
    return codec


def prepare(case, seed):
    path, n, chunk = case["path"], _n_bytes(case), case["chunk"]
    codec = _codec(case, seed)
    data = _data(case, seed)
    s = {"path": path, "codec": codec, "case": case}
    if path in ("forward", "step"):  # `chunks` lanes of `chunk` tokens
        lanes = case["chunks"]
        s["tokens"] = data.view(lanes, chunk)
        if path == "step":
            s["tokens"] = s["tokens"].t().contiguous()
        s["logits"] = torch.empty((lanes, chunk, 256) if path == "forward" else
                                  (chunk, lanes, 256), device="cuda")
        return s
    if path.startswith("file"):
        s["data"] = data.cpu().numpy().tobytes()
        if path == "file_decompress":
            s["blob"] = codec.compress(s.pop("data"), chunk_size=chunk)
        else:  # the caller's place for the container: streams hardly outgrow their data
            s["container"] = np.zeros(2 * n + 64 * case["chunks"] + 4096, np.uint8)
        return s
    s["cap"] = boa.payload_bound_words(n, chunk)
    payload = torch.zeros(s["cap"], dtype=torch.int32, device="cuda")
    if path == "compress":
        s["data"], s["payload"] = data, payload
        return s
    lens, first, words = codec.compress_device(data, n, chunk, payload, s["cap"])
    sizes = (lens // 4).astype(np.uint64)
    s["payload"] = payload[:words].clone()
    s["lens"], s["first"] = lens, first
    s["offsets"] = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.uint64)
    s["out"] = torch.empty(n, dtype=torch.uint8, device="cuda")
    return s


def run(state):
    path, codec, case = state["path"], state["codec"], state["case"]
    n, chunk = _n_bytes(case), case["chunk"]
    if path == "compress":
        lens, first, words = codec.compress_device(state["data"], n, chunk, state["payload"],
                                                   state["cap"])
        return {"payload": state["payload"], "lens": lens.astype(np.int64), "first": first,
                "words": words}
    if path == "decompress":
        codec.decompress_device(state["payload"], state["offsets"], state["lens"],
                                state["first"], chunk, case["last"], state["out"])
        return state["out"]
    if path == "file_compress":
        blob = codec.compress(state["data"], chunk_size=chunk)
        state["container"][:len(blob)] = np.frombuffer(blob, np.uint8)
        return {"container": state["container"], "length": len(blob)}
    if path == "file_decompress":
        return np.frombuffer(codec.decompress(state["blob"]), np.uint8)
    lanes = case["chunks"]
    codec.reset_state(lanes)  # every text and every stream starts from nothing
    if path == "forward":
        codec.forward_chunk(state["tokens"], lanes, chunk, state["logits"])
    else:
        for t in range(chunk):
            codec.step_batch(state["tokens"][t], lanes, state["logits"][t])
    return state["logits"]


# ----------------------------------------------------------- what it needs
def work(case):
    """Model operations of every token (multiply and add counted apart) and
    the bytes that have to move: weights once per model pass -- once per
    batch when the tokens are known, once per step when they are not --, the
    recurrent state once per step, input and output."""
    d, L, ds, prec, di, r, R = _dims(case)
    tokens, wb = _n_bytes(case), 2 if prec == "bf16" else 4
    per_layer = 2 * (2 * di * d + di * R + di * d + 8 * d * d)
    scan = di * (8 * ds + 2 * r + 30)
    flops = tokens * (L * (per_layer + scan) + 2 * (d * d + 256 * d))
    weights = wb * (L * (2 * di * d + di * R + di * d + 8 * d * d) + d * d + 256 * d)
    state = 2 * 4 * L * di * (ds + 4)
    passes = 1
    moved = 2 * tokens
    if case["path"] in ("forward", "step"):
        moved = tokens * (1 + 1024)
    if case["path"] == "step" or case["path"].endswith("decompress"):
        passes = case["chunk"]
        moved += tokens * state
    else:
        passes = -(-case["chunks"] // case["lanes"])
        moved += case["chunks"] * state
    return {"bytes": moved + passes * weights, "flops": flops}


def tolerance(case):
    if case["path"] not in ("forward", "step"):
        return "exact"  # containers, streams and decoded bytes
    if MODELS[case["model"]][3] == "bf16":
        return {"rel": 2e-2}
    return {"rel": 1e-5}


# -------------------------------------------------------------- in 64 bits
def exact(case, seed):
    """The data for a decode; logits of the model in float64 torch for
    scoring and streaming.  Coded streams have no such value."""
    path = case["path"]
    if path == "decompress":
        return _data(case, seed)
    if path == "file_decompress":
        return _data(case, seed).cpu().numpy()
    if path not in ("forward", "step") or case["chunks"] * case["chunk"] > 200000:
        return None
    d, L, ds, _, di, r, R = _dims(case)
    w = {k: v.double() for k, v in _weights(case, seed).items()}
    tok = _data(case, seed).view(case["chunks"], case["chunk"]).long()

    def ln(x, k):
        mu = x.mean(-1, keepdim=True)
        var = ((x - mu) ** 2).mean(-1, keepdim=True)
        return (x - mu) / torch.sqrt(var + 1e-5) * w[k + ".w"] + w[k + ".b"]

    def lin(x, k):
        y = x @ w[k + ".w"].t()
        return y + w[k + ".b"] if k + ".b" in w else y

    B, T = tok.shape
    x = w["emb"][tok]
    for i in range(L):
        p = "%d." % i
        xz = lin(ln(x, p + "ln1"), p + "in")
        xs, z = xz[..., :di], xz[..., di:]
        xp = torch.cat([xs.new_zeros(B, 3, di), xs], 1)
        conv = w[p + "conv.b"] + sum(w[p + "conv.w"][:, k] * xp[:, k:k + T] for k in range(4))
        u = conv * torch.sigmoid(conv)
        dbc = u @ w[p + "x.w"].t()
        dt = torch.nn.functional.softplus(lin(dbc[..., :r], p + "dt"), threshold=1e9)
        Bm, Cm = dbc[..., r:r + ds], dbc[..., r + ds:]
        A = -torch.exp(w[p + "alog"])
        h = x.new_zeros(B, di, ds)
        ys = []
        for t in range(T):
            h = torch.exp(dt[:, t, :, None] * A) * h \
                + (dt[:, t] * u[:, t])[:, :, None] * Bm[:, t, None, :]
            ys.append((h * Cm[:, t, None, :]).sum(-1))
        y = torch.stack(ys, 1) + w[p + "D"] * u
        out = lin(y * (z * torch.sigmoid(z)), p + "out")
        h1 = torch.nn.functional.gelu(lin(ln(out, p + "ln2"), p + "ff0"), approximate="tanh")
        x = x + lin(h1, p + "ff2")
    logits = lin(torch.relu(lin(x, "h0")), "h2")
    return logits if path == "forward" else logits.transpose(0, 1).contiguous()
