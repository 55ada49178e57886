"""The work that is timed on this backend, through its public entry points.

A node of the expert runtime holds some of the 20 ownership blocks of every
expert (32 neurons each) and answers one request per layer: y = sum over the
token's experts and the owned slices of gate * W_down (SiLU(W_gate x) * W_up x).
Four entry points carry that work:

  call    fr_hip_run: the backend table's run(), 1 to 8 tokens, x and y in host
          memory, once per layer;
  launch  fr_hip_launch_static: the same for one token whose plan is resident,
          y left in device memory, no host wait between layers;
  chunk   fr_hip_run_batch: a prefill chunk, x and y in host memory;
  resident  fr_hip_batch_launch and fr_hip_batch_output: a prefill chunk whose
          plan is resident, y fetched into pinned host memory.

The weights are the library's seeded synthetic units (fr_hip_synthetic), loaded
once for a configuration and kept, as a node keeps its units; routing, gates and
x are drawn from the seed. `exact` restates the published generator and the
block formats and computes the requests in 64 bits.
"""
import ctypes as C
import math

import numpy as np
import torch

import fronk_amd as fa

WEIGHT_SEED = 20261
FORMATS = {"native": fa.FMT_NATIVE, "q4kt": fa.FMT_Q4KT, "q8": fa.FMT_Q8, "mxfp4": fa.FMT_MXFP4}
MODES = {"f32": fa.MODE_F32, "q8": fa.MODE_Q8, "q8_256": fa.MODE_Q8_256}
ROUTED, TOPK, NEURONS, SHARED = 512, 10, 32, 512


def _case(name, entry, fmt, hidden, blocks, tokens, layers, routing="uniform", shared=False, mode="f32"):
    return {"name": name, "entry": entry, "fmt": fmt, "hidden": hidden, "blocks": blocks, "tokens": tokens,
            "layers": layers, "routing": routing, "shared": shared, "mode": mode}


def listed():
    return [
        # The smallest node: one owned block of the runtime's own units at its
        # own hidden size, one token with the shared expert, layer by layer.
        _case("call_1block", "call", "native", 2560, 1, 1, 4, shared=True),
        # The whole share of one token on the runtime's own units: what run()
        # does for every generated token.
        _case("call_native", "call", "native", 2560, 20, 1, 8, shared=True),
        # The same share resident at hidden 4096, in each weight format.
        _case("token_q4kt", "launch", "q4kt", 4096, 20, 1, 8),
        _case("token_q8", "launch", "q8", 4096, 20, 1, 8),
        _case("token_native", "launch", "native", 4096, 20, 1, 8, shared=True),
        # Bursts: speculative tokens of one stream or tokens of several, with
        # the skewed routing that experts see.
        _case("burst4_zipf", "call", "q4kt", 4096, 20, 4, 4, routing="zipf"),
        _case("burst8_native", "call", "native", 2560, 20, 8, 4, routing="zipf", shared=True),
        # The quantized arithmetic (ref-q8) that heterogeneous nodes agree on.
        _case("burst3_ref_q8", "call", "native", 2560, 20, 3, 4, routing="zipf", shared=True, mode="q8"),
        # A short prompt on a small node, sizes that fill no tile.
        _case("chunk_37", "chunk", "native", 2560, 7, 37, 1, routing="zipf", shared=True),
        # A prefill chunk of 512 tokens on the full share, plan resident, and
        # the runtime's own units from host memory.
        _case("prefill_512", "resident", "q4kt", 4096, 20, 512, 1),
        _case("chunk_512_native", "chunk", "native", 2560, 20, 512, 1, shared=True),
        # The largest chunk the entry point takes.
        _case("prefill_4096", "resident", "q4kt", 4096, 20, 4096, 1),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    entry = rng.choice(["call", "call", "launch", "chunk", "resident"])
    hidden = 256 * rng.choice([8, 9, 10, 10, 11, 12, 14, 15, 16, 16])
    blocks = _log_int(rng, 1, 20) if rng.random() < 0.5 else rng.randint(10, 20)
    routing = rng.choice(["uniform", "zipf"])
    shared = rng.random() < 0.5
    mode = "f32"
    if entry == "launch":
        fmt, tokens, layers = rng.choice(["native", "q4kt", "q8", "mxfp4"]), 1, rng.randint(5, 8)
    elif entry == "call":
        fmt, tokens, layers = rng.choice(["native", "native", "q4kt", "q8", "mxfp4"]), rng.randint(1, 8), rng.randint(2, 4)
        if fmt == "native":
            mode = rng.choice(["f32", "f32", "q8", "q8_256"])
    else:
        fmt, layers = rng.choice(["native", "q4kt"]), 1
        tokens = _log_int(rng, 9, 1024) if entry == "chunk" else _log_int(rng, 64, 3000)
    c = _case("", entry, fmt, hidden, blocks, tokens, layers, routing, shared, mode)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs

def _requests(case, seed):
    """One (layer, experts, gates, x) per layer: top-10 routing (uniform, or
    Zipf(1.1) over a permutation of the layer's experts), softmax gates, the
    shared expert's gate, and x of a normalised hidden state with a few outlier
    channels, scaled so that SiLU is met over its curved range."""
    rng = np.random.default_rng(seed)
    t, h = case["tokens"], case["hidden"]
    reqs = []
    for layer in range(case["layers"]):
        score = rng.gumbel(size=(t, ROUTED))
        if case["routing"] == "zipf":
            score = score - 1.1 * np.log(1.0 + rng.permutation(ROUTED))
        experts = np.argsort(-score, axis=1)[:, :TOPK].astype(np.uint16)
        logits = rng.standard_normal((t, TOPK))
        g = np.exp(logits - logits.max(axis=1, keepdims=True))
        gates = np.zeros((t, TOPK + 1), np.float32)
        gates[:, :TOPK] = g / g.sum(axis=1, keepdims=True)
        if case["shared"]:
            gates[:, TOPK] = 1.0 / (1.0 + np.exp(-rng.standard_normal(t)))
        x = 0.02 * rng.standard_normal((t, h), dtype=np.float32)
        x[:, rng.choice(h, 4, replace=False)] *= 8.0
        reqs.append((layer, experts, gates, np.ascontiguousarray(x, np.float32)))
    return reqs


_loaded = None


def _load(case):
    """The engine with this configuration's units in memory."""
    global _loaded
    key = (case["fmt"], case["hidden"], case["blocks"], case["layers"])
    eng = fa.Engine(0)
    if _loaded != key:
        torch.cuda.synchronize()
        for b in range(_loaded[2] if _loaded else 0):
            fa.check(eng.release(b), "fr_hip_release")
        _loaded = None
        for b in range(case["blocks"]):
            fa.check(eng.synthetic(b, case["hidden"], FORMATS[case["fmt"]], case["layers"], WEIGHT_SEED),
                     "fr_hip_synthetic")
        _loaded = key
    return eng


def prepare(case, seed):
    eng = _load(case)
    mode, t, h = MODES[case["mode"]], case["tokens"], case["hidden"]
    st = {"entry": case["entry"], "lib": fa.lib(), "keep": [], "steps": [], "out": []}
    for layer, experts, gates, x in _requests(case, seed):
        if case["entry"] in ("call", "chunk"):
            make = fa.make_request if case["entry"] == "call" else fa.make_batch
            req, keep = make(layer, experts, gates, x, mode)
            y = np.zeros((t, h), np.float32)
            st["keep"].append((req, keep))
            st["steps"].append((C.byref(req), fa.fptr(y)))
            st["out"].append(y)
            continue
        plan = eng.plan(layer, experts, gates, x, mode)[0] if case["entry"] == "launch" else \
            eng.batch_plan(layer, experts, gates, x, mode)
        dev = torch.from_numpy(plan).to("cuda")
        st["keep"].append((plan, dev))
        if case["entry"] == "launch":
            y = torch.zeros(h, dtype=torch.float32, device="cuda")
            status = torch.zeros(1, dtype=torch.int32, device="cuda")
            st["keep"].append(status)
            st["steps"].append((plan.ctypes.data, dev.data_ptr(), C.cast(y.data_ptr(), C.POINTER(C.c_float)),
                                status.data_ptr()))
            st["out"].append((y, status))
        else:
            y = torch.zeros((t, h), dtype=torch.float32, pin_memory=True)
            st["steps"].append((plan.ctypes.data, dev.data_ptr(), C.cast(y.data_ptr(), C.POINTER(C.c_float)), t * h))
            st["out"].append(y)
    torch.cuda.synchronize()
    return st


def run(state):
    lib, rc = state["lib"], 0
    if state["entry"] == "call":
        for req, y in state["steps"]:
            rc |= lib.fr_hip_run(req, y)
    elif state["entry"] == "launch":
        for plan, dev, y, status in state["steps"]:
            rc |= lib.fr_hip_launch_static(plan, dev, y, status, None)
    elif state["entry"] == "chunk":
        for req, y in state["steps"]:
            rc |= lib.fr_hip_run_batch(req, y)
    else:
        status = C.c_uint()
        for plan, dev, y, count in state["steps"]:
            rc |= lib.fr_hip_batch_launch(plan, dev, None)
            rc |= lib.fr_hip_batch_output(None, y, count, C.byref(status))
            rc |= status.value
    if rc:
        raise RuntimeError(f"{state['entry']} failed with {rc}")
    return state["out"]


# ------------------------------------------------------- work and tolerance

_ROW = {"q4k": (256, 144), "q8_0": (32, 34), "mx": (32, 17)}
_TYPES = {"native": ("q4k", "mx"), "q4kt": ("q4k", "q4k"), "q8": ("q8_0", "q8_0"), "mxfp4": ("mx", "mx")}


def _slice_parts(fmt, hidden, shared):
    """(gate/up type, down type, bytes of one projection, bytes of the down) of
    one slice; the all-Q4_K format stores its down transposed, [32][hidden]."""
    gu, dn = ("q8_0", "q8_0") if shared else _TYPES[fmt]
    (n, b), (m, d) = _ROW[gu], _ROW[dn]
    return gu, dn, NEURONS * hidden // n * b, NEURONS * hidden // m * d


def work(case):
    t, h, nb = case["tokens"], case["hidden"], case["blocks"]
    weights = 0
    for _, experts, gates, _ in _requests(dict(case, hidden=256), 0):
        for shared, n in ((False, len(np.unique(experts))), (True, 1 if case["shared"] else 0)):
            _, _, proj, down = _slice_parts(case["fmt"], h, shared)
            weights += n * nb * (2 * proj + down)
    pairs = t * (TOPK + (1 if case["shared"] else 0)) * case["layers"]
    return {"bytes": weights + 8 * t * h * case["layers"], "flops": 2 * 3 * NEURONS * h * nb * pairs}


def tolerance(case):
    """Four times the distance measured between the library and `exact` (3e-7
    with fp32 or split-f16 products, fp64 over experts and blocks). q8_256 forms
    SiLU in fp32, so an int8 code of h may land one step further: 1/127 of one
    neuron of the hundreds that an output sums."""
    if case["mode"] == "q8_256":
        return {"rel": 1e-3, "max": 4e-2}
    return {"rel": 1.5e-6, "max": 6e-5}


# ------------------------------------------------------- the result in 64 bits

_M64 = (1 << 64) - 1


def _i64(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _shr(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _mix(z):
    """The splitmix64 finaliser on int64 tensors (wrapping)."""
    z = z + _i64(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _i64(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _hash(keys, domain, words):
    return _mix(keys[:, None] ^ (domain << 60) ^ words[None, :])


def _bytes(keys, first, count):
    """Uniform bytes [first, first + count) of the generator, per key."""
    lo, hi = first // 8, (first + count + 7) // 8
    h = _hash(keys, 0, torch.arange(lo, hi, device=keys.device))
    return h.view(torch.uint8).reshape(len(keys), -1)[:, first - 8 * lo:first - 8 * lo + count]


def _half(h):
    """The fp16 scale of a hash, 1e-3 + 9e-3 * u rounded to nearest even."""
    v = 1e-3 + 9e-3 * (_shr(h, 40).double() * 2.0 ** -24)
    step = torch.exp2(torch.floor(torch.log2(v)) - 10)
    return torch.round(v / step) * step


def _rows(kind, keys, first, rows, cols):
    """Decoded weights [key][row][col] in 64 bits of the rows whose blocks start
    at slice byte `first`."""
    n, size = _ROW[kind]
    blocks = rows * cols // n
    at = first + size * torch.arange(blocks, device=keys.device)
    k = len(keys)
    if kind == "q8_0":
        pos = (at[:, None] + 2 + torch.arange(32, device=keys.device)).reshape(-1)
        q = (_shr(_hash(keys, 2, pos), 32) % 255 - 127).double().reshape(k, blocks, 32)
        w = q * _half(_hash(keys, 1, at))[:, :, None]
        return w.reshape(k, rows, cols)
    raw = _bytes(keys, first, size * blocks).reshape(k, blocks, size)
    if kind == "mx":
        e = 118 + _shr(_hash(keys, 1, at), 32) % 13
        nib = torch.cat([raw[:, :, 1:] & 15, raw[:, :, 1:] >> 4], dim=2).long()
        code = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64,
                            device=keys.device)
        return (code[nib] * torch.exp2((e - 127).double())[:, :, None]).reshape(k, rows, cols)
    d, dmin = _half(_hash(keys, 1, at)), _half(_hash(keys, 1, at + 2))
    s = raw[:, :, 4:16].int()
    sc = torch.cat([s[:, :, :4] & 63, (s[:, :, 8:12] & 15) | (s[:, :, :4] >> 6 << 4)], dim=2).double()
    mn = torch.cat([s[:, :, 4:8] & 63, (s[:, :, 8:12] >> 4) | (s[:, :, 4:8] >> 6 << 4)], dim=2).double()
    q = raw[:, :, 16:].reshape(k, blocks, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], dim=3).reshape(k, blocks, 8, 32).double()
    w = (d[:, :, None] * sc)[..., None] * q - (dmin[:, :, None] * mn)[..., None]
    return w.reshape(k, rows, cols)


def _quantize(v, group, narrow):
    """v as int8 codes times a scale per `group` values: with `narrow` the
    ref-q8 quantizer, which rounds code * scale to float; without it the exact
    product of code and scale."""
    g = v.float().reshape(-1, group)
    top = g.abs().amax(dim=1, keepdim=True)
    inv = torch.where(top > 0, 127.0 / top, torch.zeros_like(top))
    q = torch.round(g * inv).clamp(-127, 127).double() * (top / 127.0).double()
    q = q.float().double() if narrow else q
    return q.reshape(v.shape)


def exact(case, seed):
    h, nb, fmt, mode = case["hidden"], case["blocks"], case["fmt"], case["mode"]
    seed_mix = int(_mix(torch.tensor([WEIGHT_SEED], dtype=torch.int64))[0])
    out = []
    for layer, experts, gates, x in _requests(case, seed):
        x = torch.from_numpy(x).cuda()
        x = x.double() if mode == "f32" else _quantize(x, 64 if mode == "q8" else 256, mode == "q8")
        y = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
        ids = torch.from_numpy(experts.astype(np.int64)).cuda()
        g = torch.from_numpy(gates).cuda().double()
        for e in [int(v) for v in np.unique(experts)] + ([SHARED] if case["shared"] else []):
            gu, dn, proj, _ = _slice_parts(fmt, h, e == SHARED)
            if e == SHARED:
                tok = torch.nonzero(g[:, TOPK]).reshape(-1)
                weight = g[tok, TOPK]
            else:
                tok, col = torch.nonzero(ids == e, as_tuple=True)
                weight = g[tok, col]
            keys = torch.tensor([_i64(seed_mix ^ (b << 54) ^ (layer << 44) ^ (e << 32)) for b in range(nb)],
                                dtype=torch.int64, device="cuda")
            a = x[tok] @ _rows(gu, keys, 0, NEURONS, h).reshape(nb * NEURONS, h).T
            u = x[tok] @ _rows(gu, keys, proj, NEURONS, h).reshape(nb * NEURONS, h).T
            if mode != "f32":
                a, u = a.float().double(), u.float().double()
            v = a * torch.sigmoid(a) * u
            if mode != "f32":
                v = _quantize(v, NEURONS, mode == "q8")
            if fmt == "q4kt" and e != SHARED:
                down = _rows(dn, keys, 2 * proj, NEURONS, h).reshape(nb * NEURONS, h)
            else:
                down = _rows(dn, keys, 2 * proj, h, NEURONS).transpose(1, 2).reshape(nb * NEURONS, h)
            y[tok] += weight[:, None] * (v @ down)
        out.append(y)
    if case["entry"] == "launch":
        return [(y[0], torch.zeros(1, dtype=torch.int32)) for y in out]
    return [y.cpu().numpy() if case["entry"] in ("call", "chunk") else y for y in out]
