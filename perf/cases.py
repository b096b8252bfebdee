"""Performance cases: what a serving engine of the hybrid Gated DeltaNet + gated-attention family has this backend do.

Seven kinds of call, each through RocmBackend's public methods at the family's shapes (attention 8/2 heads x 256 or
16/4 x 128, KV blocks of 16, DeltaNet 16 heads x 128 x 128, conv 4, hidden 2048, MLP 6144):

  decode    paged_attention with the output gate: one attention layer of a decode step
  step      deltanet_decode_batch: one DeltaNet layer of a decode step
  delta     gated_delta_packed: the delta rule of a packed prefill, bf16 or fp32 inputs
  linattn   deltanet_prefill: a whole linear-attention layer of a packed prefill (conv, norms, delta rule, gated norm)
  prefill   paged_prefill_attention: a whole gated-attention layer of a packed prefill, with the KV write-back
  mlp       rms_norm -> swiglu -> linear with the residual: the MLP of a layer, for a decode batch or prefill tokens
  model     one decode step of the 24-layer 2B stack (INT4 layers, INT8 tied head) to logits

Each pass runs on what an engine keeps between calls: pools, tables, states and prepared weights. Lengths of packed or
batched sequences follow from the case alone ("sizes" seeds them); the values follow from prepare's seed.
"""
import math
import random
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path.cwd() / "metal-inference-engine_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
BLOCK, EPS = 16, 1e-6
H, DK, DV, CONV_K = 16, 128, 128, 4                     # DeltaNet heads, state and conv kernel
KEY, CHANNELS = H * DK, 2 * H * DK + H * DV
HIDDEN, INTER = 2048, 6144


def listed():
    return [
        # one user, a short context, the engine's fp32 pool: launches and latency count
        dict(name="decode_b1_f32", kind="decode", batch=1, lo=512, hi=512, sizes=1, dtype="f32", hq=8, hkv=2, d=256,
             window=0),
        # a full serving batch of mixed context lengths, bf16 pool
        dict(name="decode_b64_bf16", kind="decode", batch=64, lo=128, hi=8192, sizes=3, dtype="bf16", hq=8, hkv=2,
             d=256, window=0),
        # the sliding-window layers of the second model family at the same batch
        dict(name="decode_b64_window", kind="decode", batch=64, lo=128, hi=8192, sizes=3, dtype="bf16", hq=16, hkv=4,
             d=128, window=4096),
        # a small serving batch through one DeltaNet layer
        dict(name="step_b8", kind="step", batch=8, slots=64, layers=6),
        # long prompts through the delta rule, bf16 inputs
        dict(name="delta_bf16_4x4096", kind="delta", segs=4, lo=4096, hi=4096, sizes=4, dtype="bf16"),
        # a ragged pack of prompts through a whole linear-attention layer, fp32 activations as the linears return them
        dict(name="linattn_packed", kind="linattn", segs=8, lo=64, hi=2048, sizes=5, dtype="f32"),
        # a ragged pack of new tokens on cached prefixes through an attention layer, bf16 pool and activations
        dict(name="prefill_bf16", kind="prefill", segs=8, lo=64, hi=2048, past=16384, sizes=5, dtype="bf16", hq=8,
             hkv=2, d=256),
        # the same pack in the engine's default fp32 pool and activations
        dict(name="prefill_f32", kind="prefill", segs=8, lo=64, hi=2048, past=16384, sizes=5, dtype="f32", hq=8, hkv=2,
             d=256),
        # the MLP of one layer for a small decode batch, a full one, and a ragged pack of prompt tokens
        dict(name="mlp_int4_b8", kind="mlp", tokens=8, weights="int4"),
        dict(name="mlp_int4_b64", kind="mlp", tokens=64, weights="int4"),
        dict(name="mlp_bf16_t1777", kind="mlp", tokens=1777, weights="bf16"),
        # a whole decode step of the quantized model at a small batch
        dict(name="model_int4_b8", kind="model", batch=8, lo=256, hi=1024, sizes=9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "step", "delta", "linattn", "prefill", "prefill", "mlp", "mlp", "mlp"])
    sizes = rng.randrange(1, 1 << 20)
    heads = rng.choice([(8, 2, 256), (8, 2, 256), (16, 4, 128), (14, 2, 64)])
    if kind == "decode":
        hi = _log(rng, 64, 8192)
        return dict(kind=kind, batch=_log(rng, 1, 64), lo=max(1, hi // 64), hi=hi, sizes=sizes,
                    dtype=rng.choice(["f32", "bf16"]), hq=heads[0], hkv=heads[1], d=heads[2],
                    window=rng.choice([0, 0, 4096, 1000]))
    if kind == "step":
        return dict(kind=kind, batch=_log(rng, 1, 64), slots=64, layers=rng.choice([1, 3, 6]))
    if kind in ("delta", "linattn"):
        segs = rng.randrange(1, 9)
        hi = _log(rng, 16, 16384 // segs)
        return dict(kind=kind, segs=segs, lo=max(1, hi // rng.choice([1, 4, 32])), hi=hi, sizes=sizes,
                    dtype=rng.choice(["f32", "bf16"]))
    if kind == "prefill":
        segs = rng.randrange(1, 9)
        hi = _log(rng, 16, 2048)
        return dict(kind=kind, segs=segs, lo=max(1, hi // rng.choice([1, 4, 32])), hi=hi,
                    past=rng.choice([0, _log(rng, 16, 8192)]), sizes=sizes, dtype=rng.choice(["f32", "bf16"]),
                    hq=heads[0], hkv=heads[1], d=heads[2])
    return dict(kind=kind, tokens=_log(rng, 1, 4096), weights=rng.choice(["int4", "int8", "bf16"]))


# ---------------------------------------------------------------- sizes that follow from a case

def _between(case, n, lo, hi):
    rng = random.Random(case["sizes"] * 1000 + n + hi)
    return [rng.randint(lo, hi) for _ in range(n)]


def _lens(case):
    return _between(case, case["batch"], case["lo"], case["hi"])


def _segments(case):
    """(new tokens, cached prefix) of each packed segment."""
    new = _between(case, case["segs"], case["lo"], case["hi"])
    past = case.get("past", 0)
    return new, _between(case, case["segs"], 0, past) if past else [0] * case["segs"]


def _offsets(lengths):
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    return cu


# ---------------------------------------------------------------- inputs

def _tables(lens, gen):
    """Block tables whose blocks are a random, scattered choice of a pool a quarter larger than needed."""
    counts = [-(-n // BLOCK) for n in lens]
    blocks = math.ceil(1.25 * sum(counts))
    perm = torch.randperm(blocks, generator=gen, device=DEV).to(torch.int32)
    tables = torch.zeros(len(lens), max(counts), dtype=torch.int32, device=DEV)
    at = 0
    for i, c in enumerate(counts):
        tables[i, :c] = perm[at:at + c]
        at += c
    return tables, blocks


def _weight(rows, cols, scheme, gen):
    """A prepared [rows, cols] weight at a trained matrix's scale, in the resident format `scheme`."""
    if scheme == "bf16":
        return (torch.randn(rows, cols, generator=gen, device=DEV) / math.sqrt(cols)).to(torch.bfloat16)
    from quant import quantize
    return quantize(torch.randn(rows, cols, generator=gen, device=DEV) / math.sqrt(cols), scheme)


def prepare(case, seed):
    import workloads as wl
    from backend.rocm import RocmBackend
    gen = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *shape: torch.randn(*shape, generator=gen, device=DEV)
    kind = case["kind"]
    be = RocmBackend(DEV)
    st = {"kind": kind, "backend": be}
    dt = DTYPES.get(case.get("dtype"))
    if kind == "decode":
        lens = _lens(case)
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        tables, blocks = _tables(lens, gen)
        st.update(q=r(len(lens), hq, d), k=r(blocks, BLOCK, hkv, d).to(dt), v=r(blocks, BLOCK, hkv, d).to(dt),
                  gate=r(len(lens), hq * d), tables=tables, lens=torch.tensor(lens, dtype=torch.int32, device=DEV),
                  window=case["window"] or None)
    elif kind == "step":
        B = case["batch"]
        pool = wl.StateSlots(case["slots"], case["layers"], H, DK, DV, CHANNELS, CONV_K, DEV)
        pool.S.copy_(0.02 * r(*pool.S.shape))
        pool.conv.copy_(r(*pool.conv.shape))
        rows = torch.randperm(case["slots"], generator=gen, device=DEV)[:B].tolist()
        st.update(y=r(B, CHANNELS + H * DV + 2 * H), pool=pool, states=pool.views(rows), slot=case["layers"] // 2,
                  rows=rows, **_layer(r))
    elif kind == "delta":
        lengths, _ = _segments(case)
        N = sum(lengths)
        l2 = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        st.update(q=(l2(r(N, H, DK)) / math.sqrt(DK)).to(dt), k=l2(r(N, H, DK)).to(dt), v=r(N, H, DV).to(dt),
                  beta=torch.sigmoid(r(N, H)), g=-torch.nn.functional.softplus(r(N, H)),
                  S=0.05 * r(len(lengths), H, DK, DV), cu=_offsets(lengths))
    elif kind == "linattn":
        lengths, _ = _segments(case)
        pool = wl.StateSlots(len(lengths), 1, H, DK, DV, CHANNELS, CONV_K, DEV)
        pool.S.copy_(0.05 * r(*pool.S.shape))
        pool.conv.copy_(r(*pool.conv.shape))
        st.update(y=r(sum(lengths), CHANNELS + H * DV + 2 * H).to(dt), pool=pool,
                  states=pool.views(range(len(lengths))), cu=_offsets(lengths), **_layer(r))
    elif kind == "prefill":
        lengths, past = _segments(case)
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        N = sum(lengths)
        tables, blocks = _tables([n + p for n, p in zip(lengths, past)], gen)
        st.update(q=r(N, hq, d).to(dt), k_new=r(N, hkv, d).to(dt), v_new=r(N, hkv, d).to(dt),
                  gate=r(N, hq * d).to(dt), k=r(blocks, BLOCK, hkv, d).to(dt), v=r(blocks, BLOCK, hkv, d).to(dt),
                  tables=tables, cu=_offsets(lengths), starts=past)
    elif kind == "mlp":
        st.update(h=r(case["tokens"], HIDDEN), norm=1.0 + 0.1 * r(HIDDEN),
                  gate_up=_weight(2 * INTER, HIDDEN, case["weights"], gen),
                  down=_weight(HIDDEN, INTER, case["weights"], gen))
    else:
        cfg = wl.QWEN35_2B
        lens = _lens(case)
        seqs = wl.HybridDecodeState(cfg, lens, DEV, seed=seed)
        st.update(cfg=cfg, w=wl.random_device_weights(cfg, "int4", DEV, seed=seed), seqs=seqs,
                  tokens=torch.randint(0, cfg.vocab, (len(lens),), generator=gen, device=DEV), layout=seqs.layout())
    return st


def _layer(r):
    """The vectors of one linear-attention layer."""
    return dict(conv_w=0.5 * r(CHANNELS, CONV_K), A_log=0.5 * r(H), dt_bias=0.5 * r(H), norm=1.0 + 0.1 * r(DV))


def _columns(y):
    """qkv, z, b, a: the column slices of the fused in_proj output, as the model passes them."""
    z = CHANNELS + H * DV
    return y[:, :CHANNELS], y[:, CHANNELS:z], y[:, z:z + H], y[:, z + H:]


# ---------------------------------------------------------------- one pass

def run(st):
    be, kind = st["backend"], st["kind"]
    if kind == "decode":
        return be.paged_attention(st["q"], st["k"], st["v"], st["tables"], st["lens"], BLOCK, st["window"],
                                  gate=st["gate"])
    if kind == "step":
        o = be.deltanet_decode_batch(*_columns(st["y"]), st["states"], st["slot"], st["conv_w"], st["A_log"],
                                     st["dt_bias"], st["norm"], EPS, (H, DK, DV, KEY))
        return o, st["pool"].S, st["pool"].conv
    if kind == "delta":
        o = be.gated_delta_packed(st["q"], st["k"], st["v"], st["beta"], st["g"], st["cu"], st["S"])
        return o, st["S"]
    if kind == "linattn":
        o = be.deltanet_prefill(*_columns(st["y"]), st["states"], 0, st["cu"], st["conv_w"], st["A_log"],
                                st["dt_bias"], st["norm"], EPS, (H, DK, DV, KEY))
        return o, st["pool"].S, st["pool"].conv
    if kind == "prefill":
        o = be.paged_prefill_attention(st["q"], st["k_new"], st["v_new"], st["k"], st["v"], st["tables"], st["cu"],
                                       st["starts"], BLOCK, gate=st["gate"])
        return o, st["k"], st["v"]
    if kind == "mlp":
        act = be.swiglu(be.rms_norm(st["h"], st["norm"], EPS), st["gate_up"])
        return be.linear(act, st["down"], residual=st["h"])
    import workloads as wl
    logits = wl.hybrid_decode_step(be, st["w"], st["seqs"], st["tokens"], st["layout"])
    return logits, st["seqs"].pool.S, st["seqs"].pool.conv, st["seqs"].k, st["seqs"].v


# ---------------------------------------------------------------- what a pass cannot do without

WEIGHT_BYTES = {"int4": 20 / 32, "int8": 34 / 32, "bf16": 2.0}     # a weight's code with its share of scale and min


def work(case):
    kind = case["kind"]
    e = {"f32": 4, "bf16": 2}.get(case.get("dtype"))
    if kind == "decode":
        seen = [min(n, case["window"] or n) for n in _lens(case)]
        row = case["hq"] * case["d"]
        return {"bytes": 2 * sum(seen) * case["hkv"] * case["d"] * e + case["batch"] * (12 * row + 4)
                + 4 * sum(-(-n // BLOCK) for n in seen), "flops": 4 * row * sum(seen)}
    state = H * DK * DV * 4
    if kind == "step":
        row = 8 * (CONV_K - 1) * CHANNELS + 4 * CHANNELS + 8 * H * DV + 8 * H
        return {"bytes": case["batch"] * (2 * state + row) + 4 * CHANNELS * CONV_K + 4 * (2 * H + DV),
                "flops": case["batch"] * H * 7 * DK * DV}
    if kind in ("delta", "linattn"):
        lengths, _ = _segments(case)
        N = sum(lengths)
        chunks = sum(-(-n // 64) for n in lengths)
        flops = chunks * H * (5 * 2 * 64 * 64 * DK + 3 * 2 * 64 * DK * DV + 64 ** 3 // 3)
        if kind == "delta":
            return {"bytes": N * H * ((2 * DK + DV) * e + 8 + 4 * DV) + 2 * len(lengths) * state, "flops": flops}
        return {"bytes": N * ((CHANNELS + H * DV + 2 * H) * e + 4 * H * DV) + 4 * CHANNELS * CONV_K
                + len(lengths) * (2 * state + 8 * (CONV_K - 1) * CHANNELS), "flops": flops}
    if kind == "prefill":
        lengths, past = _segments(case)
        row = case["hq"] * case["d"]
        kv = 2 * case["hkv"] * case["d"] * e
        return {"bytes": sum((2 * n + p) * kv for n, p in zip(lengths, past)) + sum(lengths) * row * (2 * e + 4),
                "flops": sum(4 * row * (n * p + n * (n + 1) // 2) for n, p in zip(lengths, past))}
    if kind == "mlp":
        n = 3 * HIDDEN * INTER
        return {"bytes": n * WEIGHT_BYTES[case["weights"]] + 8 * case["tokens"] * HIDDEN,
                "flops": 2 * n * case["tokens"]}
    import workloads as wl
    cfg, lens = wl.QWEN35_2B, _lens(case)
    B, full = case["batch"], sum(wl.QWEN35_2B.is_full(i) for i in range(wl.QWEN35_2B.layers))
    mats = {n: s for n, s in wl.hybrid_weight_shapes(cfg).items() if len(s) == 2 and "conv1d" not in n}
    head = mats.pop("embed_tokens.weight")
    small = sum(a * b for a, b in mats.values())
    linear = cfg.layers - full
    nbytes = small * WEIGHT_BYTES["int4"] + head[0] * head[1] * WEIGHT_BYTES["int8"] + 4 * B * cfg.vocab \
        + full * 4 * sum(lens) * cfg.Hkv * cfg.d + linear * B * (2 * state + 8 * (CONV_K - 1) * CHANNELS)
    return {"bytes": nbytes, "flops": 2 * B * (small + head[0] * head[1]) + full * 4 * cfg.Hq * cfg.d * sum(lens)
            + linear * B * H * 7 * DK * DV}


# ---------------------------------------------------------------- tolerances

def tolerance(case):
    """Against 64 bits the fp32 paths are 2e-7 to 1.2e-6 off, bf16 attention (its probabilities rounded to bf16)
    1.6e-3, and a whole step, which carries every layer's rounding and rounds the new K / V rows to bf16, 2.6e-6;
    about four times that and more where few draws were seen."""
    kind = case["kind"]
    if kind == "prefill":
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1e-5}
    if kind == "model":
        return {"rel": 2e-5}
    return {"rel": 1e-5}


# ---------------------------------------------------------------- the same outputs in 64 bits

def _attend(q, K, V, start, window):
    """q [T, hq, d] at positions start .. start + T - 1 over K, V [S, hkv, d], causal, in 64 bits."""
    T, hq, d = q.shape
    S, hkv, _ = K.shape
    out = torch.empty(T, hq, d, dtype=torch.float64, device=DEV)
    pos = torch.arange(start, start + T, device=DEV)[:, None]
    key = torch.arange(S, device=DEV)[None, :]
    hidden = key > pos
    if window:
        hidden |= key <= pos - window
    for h in range(hq):
        kv = h // (hq // hkv)
        s = (q[:, h].double() @ K[:, kv].double().T.contiguous()) / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ V[:, kv].double().contiguous()
    return out


def _rows_of(pool, table, n):
    return pool[table[:-(-n // BLOCK)].long()].flatten(0, 1)[:n]


def _recurrence(q, k, v, beta, g, S, cu):
    """The gated delta rule token by token in 64 bits, all sequences side by side (shorter ones padded with rows that
    change nothing). q, k, v [N, H, *], beta, g [N, H], S [n, H, dk, dv] -> (o [N, H, dv], S)."""
    lens = [b - a for a, b in zip(cu, cu[1:])]
    n, T = len(lens), max(lens)

    def pad(x):
        out = torch.zeros(T, n, *x.shape[1:], dtype=torch.float64, device=DEV)
        for i, (a, b) in enumerate(zip(cu, cu[1:])):
            out[:b - a, i] = x[a:b].double()
        return out
    q, k, v, beta, decay = pad(q), pad(k), pad(v), pad(beta), pad(g).exp()
    S = S.double().clone()
    o = torch.empty(T, n, H, DV, dtype=torch.float64, device=DEV)
    for t in range(T):
        S *= decay[t][..., None, None]
        delta = (v[t] - (k[t][..., None, :] @ S)[..., 0, :]) * beta[t][..., None]
        S += k[t][..., :, None] * delta[..., None, :]
        o[t] = (q[t][..., None, :] @ S)[..., 0, :]
    return torch.cat([o[:m, i] for i, m in enumerate(lens)]), S


def _linear_attention(y, S, conv, cu, layer):
    """A linear-attention layer around the recurrence, in 64 bits -> (o [N, H * dv], S [n, ...], conv [n, K-1, C])."""
    qkv, z, b, a = (t.double() for t in _columns(y))
    us, tails = [], []
    w = layer["conv_w"].double()
    for i, (lo, hi) in enumerate(zip(cu, cu[1:])):
        hist = torch.cat([conv[i].double(), qkv[lo:hi]])
        u = sum(hist[j:j + hi - lo] * w[:, j] for j in range(CONV_K))
        us.append(u * torch.sigmoid(u))
        tails.append(hist[-(CONV_K - 1):])
    u = torch.cat(us)
    l2 = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    q = l2(u[:, :KEY].reshape(-1, H, DK)) / math.sqrt(DK)
    k = l2(u[:, KEY:2 * KEY].reshape(-1, H, DK))
    v = u[:, 2 * KEY:].reshape(-1, H, DV)
    g = -layer["A_log"].double().exp() * torch.nn.functional.softplus(a + layer["dt_bias"].double())
    o, S = _recurrence(q, k, v, torch.sigmoid(b), g, S, cu)
    z = z.reshape(-1, H, DV)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS) * layer["norm"].double() * z * torch.sigmoid(z)
    return o.reshape(-1, H * DV), S, torch.stack(tails)


def _dense(w, rows=slice(None)):
    """Rows of a weight in 64 bits."""
    if isinstance(w, torch.Tensor):
        return w[rows].double()
    N, K = w.shape
    data = w.data[rows]
    if w.scheme == "int8":
        codes = data.double()
    else:
        codes = torch.stack([data & 15, data >> 4], -1).reshape(data.shape[0], K).double()
    x = codes.view(codes.shape[0], K // 32, 32) * w.scales[rows].double()[..., None]
    if w.scheme == "int4":
        x = x + w.mins[rows].double()[..., None]
    return x.view(codes.shape[0], K)


def _product(x, w):
    """x @ w.T in 64 bits, a slab of rows at a time."""
    N = w.shape[0]
    return torch.cat([x @ _dense(w, slice(r, min(N, r + 32768))).T.contiguous() for r in range(0, N, 32768)], 1)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _mlp(h, norm, gate_up, down):
    y = _product(_rms(h, norm), gate_up)
    F = y.shape[1] // 2
    return h + _product(y[:, :F] * torch.sigmoid(y[:, :F]) * y[:, F:], down)


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "decode":
        out = torch.stack([_attend(st["q"][i:i + 1], _rows_of(st["k"], st["tables"][i], n),
                                   _rows_of(st["v"], st["tables"][i], n), n - 1, case["window"])[0]
                           for i, n in enumerate(_lens(case))])
        return out * torch.sigmoid(st["gate"].double()).view(out.shape)
    if kind == "step":
        pool, slot, rows = st["pool"], st["slot"], st["rows"]
        S, conv = pool.S.double(), pool.conv.double()
        o, S[rows, slot], conv[rows, slot] = _linear_attention(st["y"], pool.S[rows, slot], pool.conv[rows, slot],
                                                               list(range(len(rows) + 1)), st)
        return o, S, conv
    if kind == "delta":
        return _recurrence(st["q"], st["k"], st["v"], st["beta"], st["g"], st["S"], st["cu"])
    if kind == "linattn":
        o, S, conv = _linear_attention(st["y"], st["pool"].S[:, 0], st["pool"].conv[:, 0], st["cu"], st)
        return o, S[:, None], conv[:, None]
    if kind == "prefill":
        k, v, outs = st["k"].clone(), st["v"].clone(), []
        for i, (lo, hi, p) in enumerate(zip(st["cu"], st["cu"][1:], st["starts"])):
            pos = torch.arange(p, p + hi - lo, device=DEV)
            at = st["tables"][i, pos // BLOCK].long() * BLOCK + pos % BLOCK
            k.flatten(0, 1)[at] = st["k_new"][lo:hi]
            v.flatten(0, 1)[at] = st["v_new"][lo:hi]
            n = p + hi - lo
            outs.append(_attend(st["q"][lo:hi], _rows_of(k, st["tables"][i], n), _rows_of(v, st["tables"][i], n), p,
                                0))
        out = torch.cat(outs)
        return out * torch.sigmoid(st["gate"].double()).view(out.shape), k.double(), v.double()
    if kind == "mlp":
        return _mlp(st["h"].double(), st["norm"], st["gate_up"], st["down"])
    return _model(st)


def _model(st):
    cfg, w, seqs = st["cfg"], st["w"], st["seqs"]
    slots, tables, lens, positions = st["layout"]
    B = len(seqs.lens)
    S, conv, k, v = seqs.pool.S.double(), seqs.pool.conv.double(), seqs.k.double(), seqs.v.double()
    h = torch.cat([_dense(w["embed_tokens.weight"], slice(t, t + 1)) for t in st["tokens"].tolist()])
    inv = (1.0 / (cfg.theta ** (torch.arange(0, cfg.rot // 2, dtype=torch.float32) / (cfg.rot // 2)))).to(DEV)
    angle = positions.double()[:, None, None] * inv.double()
    cos, sin = torch.cos(angle), torch.sin(angle)

    def turn(x):
        a, b = x[..., :cfg.rot // 2], x[..., cfg.rot // 2:cfg.rot]
        return torch.cat([a * cos - b * sin, a * sin + b * cos, x[..., cfg.rot:]], -1)

    for i in range(cfg.layers):
        p, L = f"layers.{i}.", seqs.slot[i]
        x = _rms(h, w[p + "input_layernorm.weight"])
        if cfg.is_full(i):
            a = p + "self_attn."
            y = _product(x, w[a + "qkvg.weight"])
            nq, nk = cfg.Hq * cfg.d, cfg.Hkv * cfg.d
            q = turn(_rms(y[:, :nq].reshape(B, cfg.Hq, cfg.d), w[a + "q_norm.weight"]))
            kn = turn(_rms(y[:, nq:nq + nk].reshape(B, cfg.Hkv, cfg.d), w[a + "k_norm.weight"]))
            vn = y[:, nq + nk:nq + 2 * nk].reshape(B, cfg.Hkv, cfg.d)
            k[L].flatten(0, 1)[slots] = kn.to(seqs.k.dtype).double()
            v[L].flatten(0, 1)[slots] = vn.to(seqs.v.dtype).double()
            o = torch.cat([_attend(q[s:s + 1], _rows_of(k[L], tables[s], n + 1), _rows_of(v[L], tables[s], n + 1), n,
                                   0) for s, n in enumerate(seqs.lens)]).reshape(B, nq)
            h = h + _product(o * torch.sigmoid(y[:, nq + 2 * nk:]), w[a + "o_proj.weight"])
        else:
            a = p + "linear_attn."
            layer = dict(conv_w=w[a + "conv1d.weight"], A_log=w[a + "A_log"], dt_bias=w[a + "dt_bias"],
                         norm=w[a + "norm.weight"])
            o, S[:, L], conv[:, L] = _linear_attention(_product(x, w[a + "in_proj.weight"]), S[:, L], conv[:, L],
                                                       list(range(B + 1)), layer)
            h = h + _product(o, w[a + "out_proj.weight"])
        h = _mlp(h, w[p + "post_attention_layernorm.weight"], w[p + "mlp.gate_up.weight"],
                 w[p + "mlp.down_proj.weight"])
    return _product(_rms(h, w["norm.weight"]), w["embed_tokens.weight"]), S, conv, k, v
