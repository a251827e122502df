"""The work whose speed is measured: passes of the batched ragged decode pass
through `Context.step` and `Context.read_logits`, over the model shapes of
`chattorrent_amd.configs`.

A pass is what a peer's Runner does for the jobs that wait: decode rows,
verify rows of speculative decoding, prompt chunks, and mixes of them, on the
whole model or on the range of blocks (a stage) that the peer holds. A stage
takes the f16 rows [n, H] the previous peer hands it and returns its own.

`kind` says which:
  model   the whole model from token ids; the sampler has a temperature and
          no top-k, so the whole logits rows are read back;
  stage   `layers` blocks from f16 rows to f16 rows;
  head    the last position alone (final norm, LM head, the top candidates),
          as the peer that ends the line runs it.
`shape` names the model. A pass packs `chats` jobs of `rows` rows whose
contexts are log-uniform in [ctx_lo, ctx_hi], and `chunks` jobs of
`chunk_rows` rows of a prompt that already has `chunk_past` tokens in the
cache. `scales` is the weights' format: "f16" (one per 32 values) or "f32"
(one per 64, what the reference's converter writes).

Every pass of a state runs the same jobs again: the K/V rows it appends are
overwritten with themselves, and a hybrid stage's chats run a verify that
goes back to the state before it (a rejected verify), or a prompt's first
chunk, so the recurrent state it starts from is the same each time.
"""
import hashlib
import math
import random

import numpy as np
import torch

from chattorrent_amd import ccdecode as cc
from chattorrent_amd import configs

SHAPES = {"smollm2": configs.SMOLLM2, "27b": configs.M27B, "8b": configs.LLAMA8B, "qwen38": configs.QWEN38}
SEEDED_ROWS = 24   # rows of real history a hybrid chat's recurrent state holds


def case_of(name, **kw):
    c = dict(name=name, kind="stage", shape="27b", layers=4, scales="f16", chats=0, rows=1, ctx_lo=128, ctx_hi=16384,
             chunks=0, chunk_rows=0, chunk_past=0, topk=0, ctx_seed=1234)
    c.update(kw)
    return c


def listed():
    return [
        # one person chatting with the small model: a pass of one row, all latency
        case_of("small-model-one-chat", kind="model", shape="smollm2", layers=30, chats=1, ctx_lo=300, ctx_hi=300),
        # four people on it, at the contexts of the configuration that names it
        case_of("small-model-four-chats", kind="model", shape="smollm2", layers=30, chats=4, ctx_lo=17, ctx_hi=1024),
        # the 27B split over many peers, one block each, a dozen chats, a
        # checkpoint as the converter writes it
        case_of("27b-block-12-chats", layers=1, scales="f32", chats=12, ctx_lo=256, ctx_hi=16384),
        # a peer's stage for one long chat
        case_of("27b-stage-one-chat", chats=1, ctx_lo=9000, ctx_hi=9000),
        # the headline's batch: 32 ragged chats decoding
        case_of("27b-stage-32-chats", layers=8, chats=32),
        # 16 chats verifying 7 drafts each, long contexts
        case_of("27b-stage-verify", chats=16, rows=8, ctx_lo=4096, ctx_hi=32768),
        # a prompt chunk beside decode rows, in the converter's format
        case_of("8b-chunk-beside-decode", shape="8b", scales="f32", chats=24, ctx_lo=32, ctx_hi=4096, chunks=1,
                chunk_rows=512, chunk_past=512),
        # as full as a pass of the continuous batch gets: two chunks, 64 chats
        case_of("8b-two-chunks-64-chats", shape="8b", layers=8, chats=64, ctx_lo=32, ctx_hi=4096, chunks=2,
                chunk_rows=512, chunk_past=1024),
        # the last peer: 32 sampled rows with top-k 40
        case_of("27b-head-top-40", kind="head", chats=32, topk=40, layers=0),
        # the hybrid: 16 chats verifying, three recurrent blocks to a full one
        case_of("hybrid-stage-verify", shape="qwen38", chats=16, rows=8, ctx_lo=512, ctx_hi=8192),
        # the hybrid: a new prompt's first chunk, which the recurrence walks
        case_of("hybrid-stage-prompt", shape="qwen38", chunks=1, chunk_rows=512, chunk_past=0),
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    seed, scales = rng.randrange(1 << 20), rng.choice(["f16", "f32"])
    what = rng.choice(["model", "decode", "decode", "verify", "chunk", "chunk", "head", "hybrid-verify",
                       "hybrid-prompt"])
    if what == "model":
        lo = logu(16, 512)
        c = case_of("", kind="model", shape="smollm2", layers=30, chats=rng.randint(1, 8), ctx_lo=lo,
                    ctx_hi=logu(lo, 2000))
    elif what == "decode":
        shape, lo = rng.choice(["27b", "8b"]), logu(32, 4096)
        c = case_of("", shape=shape, layers=rng.randint(1, 4), scales=scales, chats=logu(1, 48), ctx_lo=lo,
                    ctx_hi=logu(lo, 16384))
    elif what == "verify":
        lo = logu(256, 8192)
        c = case_of("", layers=rng.randint(1, 3), scales=scales, chats=logu(1, 16), rows=rng.randint(2, 8), ctx_lo=lo,
                    ctx_hi=logu(lo, 32768))
    elif what == "chunk":
        c = case_of("", shape=rng.choice(["27b", "8b", "8b"]), layers=rng.randint(1, 3), scales=scales,
                    chats=rng.randint(0, 48), ctx_lo=32, ctx_hi=logu(32, 4096), chunks=rng.randint(1, 2),
                    chunk_rows=logu(17, 512), chunk_past=rng.choice([0, logu(1, 3000)]))
    elif what == "head":
        c = case_of("", kind="head", shape=rng.choice(["27b", "8b"]), chats=logu(1, 128), topk=logu(1, 256), layers=0)
    elif what == "hybrid-verify":
        lo = logu(64, 2048)
        c = case_of("", shape="qwen38", layers=rng.choice([1, 4]), chats=logu(1, 16), rows=rng.randint(1, 8),
                    ctx_lo=lo, ctx_hi=logu(lo, 8192))
    else:
        c = case_of("", shape="qwen38", layers=rng.choice([1, 4]), chunks=rng.randint(1, 2),
                    chunk_rows=logu(9, 400), chunk_past=0)
    del c["name"]
    c["ctx_seed"] = seed
    return c


# ------------------------------------------------------------ what a case is ---

def dims_of(case):
    d = dict(SHAPES[case["shape"]], n_layer=max(1, case["layers"]))
    if d.get("hybrid"):
        d["layer_types"] = d["layer_types"][:d["n_layer"]]
        d["mtp_vocab"] = 0
    return d


def is_linear(d, layer):
    return bool(d.get("layer_types")) and d["layer_types"][layer] == "linear_attention"


def jobs_of(case):
    """(past, rows) of each job, in slot order: the chats, then the chunks."""
    rng = random.Random(case["ctx_seed"])
    if case["kind"] == "head":
        return [(0, 1)] * case["chats"]
    out = []
    for _ in range(case["chats"]):
        t = math.exp(rng.uniform(math.log(case["ctx_lo"]), math.log(case["ctx_hi"])))
        out.append((max(int(round(t)), SEEDED_ROWS + 1), case["rows"]))
    return out + [(case["chunk_past"], case["chunk_rows"])] * case["chunks"]


def matrices(d, layer):
    """name -> (tensor id, generator stream, N, K) of one block's q8 tensors. The
    in-projection of a linear_attention block is one fused tensor: q, k, v, z,
    then b and a, each padded to whole 16-row tiles."""
    H, F, D = d["hidden"], d["ffn"], d["head_dim"]
    s, qd, kvd = (layer + 1) * 16, d["n_heads"] * D, d["n_kv_heads"] * D
    m = {"gate": (cc.T_GATE, s + 4, F, H), "up": (cc.T_UP, s + 5, F, H), "down": (cc.T_DOWN, s + 6, H, F)}
    if is_linear(d, layer):
        kd, vd, nvp = d["lin_nk"] * d["lin_dk"], d["lin_nv"] * d["lin_dv"], 16 * -(-d["lin_nv"] // 16)
        m.update(lin=(None, s + 7, 2 * kd + 2 * vd + 2 * nvp, H), out=(cc.T_OUT_PROJ, s + 8, H, vd))
    else:
        m.update(q=(cc.T_Q, s, qd, H), k=(cc.T_K, s + 1, kvd, H), v=(cc.T_V, s + 2, kvd, H), o=(cc.T_O, s + 3, H, qd))
        if d.get("hybrid"):
            m["attn_gate"] = (cc.T_ATTN_GATE, s + 12, qd, H)
    return m


def work(case):
    d = dims_of(case)
    H, D, jobs = d["hidden"], d["head_dim"], jobs_of(case)
    rows = sum(n for _, n in jobs)
    by = fl = 0.0
    if case["kind"] != "head":
        kv = 2 * d["n_kv_heads"] * (D + D // 8)
        for layer in range(case["layers"]):
            w = sum(N * K for _, _, N, K in matrices(d, layer).values())
            by += w * 1.0625
            fl += 2.0 * w * rows
            if is_linear(d, layer):
                S = d["lin_nv"] * d["lin_dk"] * d["lin_dv"]
                by += len(jobs) * 8 * S
                fl += 8.0 * S * rows
            else:
                by += sum((p + n) * kv for p, n in jobs)
                fl += sum(4.0 * n * d["n_heads"] * D * (p + (n + 1) / 2) for p, n in jobs)
    if case["kind"] != "stage":
        sampled = len(jobs)
        by += d["vocab"] * H * 1.0625 + sampled * (4 * d["vocab"] if case["kind"] == "model" else 8 * case["topk"])
        fl += 2.0 * d["vocab"] * H * sampled
    if case["kind"] != "model":
        by += (4 if case["kind"] == "stage" else 2) * rows * H
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times the relative 2-norm error measured against the same
    pass in 64 bits. A stage's rows are f16 after every block: a sum in another
    order moves a few of them (and K/V codes) by one step, and each block adds
    its own (4.6e-6 after one, 1.5e-4 to 2.5e-4 after four, 5e-4 after eight).
    The head's f32 logits carry the rounding of their sums alone (1e-7, and a
    few times that for sums in another order); a whole model's carry 30 blocks
    of such steps (1e-3)."""
    if case["kind"] == "model":
        return {"rel": 5e-3, "max": 0.05}
    if case["kind"] == "head":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.002}
    return {"rel": 2.5e-4 * case["layers"], "max": 0.02}


# ------------------------------------------------------------------- inputs ---

def generator(*key):
    h = hashlib.sha256(repr(key).encode()).digest()
    return torch.Generator(device="cuda").manual_seed(int.from_bytes(h[:6], "little"))


def uniform(shape, lo, hi, *key):
    return lo + (hi - lo) * torch.rand(shape, generator=generator(*key), device="cuda", dtype=torch.float32)


def rows_of(case, seed):
    """The f16 rows handed to a stage (or to the head), [rows, H]."""
    n = sum(n for _, n in jobs_of(case))
    return torch.randn((n, dims_of(case)["hidden"]), generator=generator("rows", seed), device="cuda").half()


def ids_of(case, seed):
    rng = np.random.default_rng(seed)
    return [rng.integers(0, dims_of(case)["vocab"], n).astype(np.int32) for _, n in jobs_of(case)]


def f32_weight(seed, layer, name, N, K):
    """Codes int8 [N, K] and f32 scales [N, K/64] as the converter writes them."""
    codes = torch.randint(-127, 128, (N, K), generator=generator("codes", seed, layer, name), device="cuda",
                          dtype=torch.int8)
    return codes, uniform((N, -(-K // 64)), 0.5e-4, 2e-4, "scales", seed, layer, name)


def norms_of(d, seed, layer):
    """Norm weights and a hybrid block's f32 parameters: name -> (tensor id, values)."""
    H, out = d["hidden"], {}
    for name, t in (("ln1", cc.T_LN1), ("ln2", cc.T_LN2)):
        out[name] = (t, uniform(H, 0.6, 1.4, name, seed, layer))
    if is_linear(d, layer):
        kd, vd, nv = d["lin_nk"] * d["lin_dk"], d["lin_nv"] * d["lin_dv"], d["lin_nv"]
        for name, t, n in (("conv_q", cc.T_CONV_Q, kd), ("conv_k", cc.T_CONV_K, kd), ("conv_v", cc.T_CONV_V, vd)):
            out[name] = (t, uniform((n, 4), -0.7, 0.9, name, seed, layer))
        out["gate_params"] = (cc.T_GATE_PARAMS, torch.cat([uniform(nv, -3.0, 0.5, "A_log", seed, layer),
                                                           uniform(nv, -1.5, 0.5, "dt", seed, layer)]))
        out["gated_norm"] = (cc.T_GATED_NORM, uniform(d["lin_dv"], 0.6, 1.4, "gnorm", seed, layer))
    elif d.get("hybrid"):
        for name, t in (("q_norm", cc.T_Q_NORM), ("k_norm", cc.T_K_NORM)):
            out[name] = (t, uniform(d["head_dim"], 0.6, 1.4, name, seed, layer))
    return out


def prepare(case, seed):
    d, jobs = dims_of(case), jobs_of(case)
    n_layer, hybrid = d["n_layer"], bool(d.get("hybrid"))
    rows = sum(n for _, n in jobs)
    seeding = hybrid and any(p > 0 for p, _ in jobs)
    lo, hi = {"model": (0, n_layer + 2), "stage": (1, n_layer + 1), "head": (n_layer + 1, n_layer + 2)}[case["kind"]]
    pages = [-(-(p + n) // 64) for p, n in jobs]
    n_max = 64 * max(pages)
    ctx = cc.Context(d, n_max=n_max, t_max=max(rows, SEEDED_ROWS * len(jobs) if seeding else 0),
                     slots=-(-sum(pages) // max(pages)), sessions=len(jobs), lo=lo, hi=hi)
    if case["scales"] == "f16":
        ctx.fill_random(seed)
    held = range(case["layers"]) if case["kind"] != "head" else ()
    for layer in held:
        if case["scales"] == "f32":
            for name, (t, _, N, K) in matrices(d, layer).items():
                codes, sc = f32_weight(seed, layer, name, N, K)
                ctx.upload_q8(layer, t, codes.cpu().numpy(), sc.cpu().numpy(), group=64)
        for t, v in norms_of(d, seed, layer).values():
            ctx.upload_norm(layer, t, v.cpu().numpy())
    if case["kind"] != "stage":
        if case["scales"] == "f32":
            codes, sc = f32_weight(seed, -1, "head", d["vocab"], d["hidden"])
            ctx.upload_q8(-1, cc.T_WTE if d.get("tied", True) else cc.T_LM_HEAD, codes.cpu().numpy(), sc.cpu().numpy(),
                          group=64)
        ctx.upload_norm(-1, cc.T_NORM, uniform(d["hidden"], 0.6, 1.4, "norm", seed).cpu().numpy())
    for slot, (past, n) in enumerate(jobs):
        if case["kind"] != "head" and past > 0:
            ctx.fill_random_kv(slot, past - SEEDED_ROWS if hybrid else past, seed, slot + 1)
    if seeding:   # the chats' last rows, through the recurrent blocks
        hist = history(case, seed).cpu().numpy().view(np.uint16)
        ctx.step([dict(slot=s, past=p - SEEDED_ROWS, n=SEEDED_ROWS, hidden=hist[s]) for s, (p, _) in enumerate(jobs)],
                 at=lo, to=hi)
    out, at = [], 0
    given = ids_of(case, seed) if case["kind"] == "model" else rows_of(case, seed).cpu().numpy().view(np.uint16)
    for slot, (past, n) in enumerate(jobs):
        j = dict(slot=slot, past=past, n=n)
        if case["kind"] == "model":
            j["ids"] = given[slot]
        else:
            j["hidden"] = given[at:at + n]
        if case["kind"] != "stage":
            j["sampled"] = 1
        if hybrid and past > 0:
            j["snap"] = True
        out.append(j)
        at += n
    state = dict(ctx=ctx, jobs=out, at=lo, to=hi, kind=case["kind"], topk=max(1, case["topk"]))
    if seeding:   # the verify that run() goes back from
        ctx.step(out, at=lo, to=hi)
        for j in out:
            j["keep"] = 0
    return state


def history(case, seed):
    """The f16 rows a hybrid stage's chats have just been through, [chats, SEEDED_ROWS, H]."""
    d = dims_of(case)
    return torch.randn((len(jobs_of(case)), SEEDED_ROWS, d["hidden"]), generator=generator("history", seed),
                       device="cuda").half()


def run(state):
    ctx, jobs = state["ctx"], state["jobs"]
    if state["kind"] == "stage":
        return {"rows": ctx.step(jobs, at=state["at"], to=state["to"]).view(np.float16)}
    vals, ids = ctx.step(jobs, at=state["at"], to=state["to"], topk=state["topk"])
    if state["kind"] == "model":
        return {"logits": ctx.read_logits(len(jobs))}
    return {"logits": vals, "ids": ids.view(np.int32)}


# ------------------------------------------------- the same pass in 64 bits ---
# The synthetic weights and caches come from a counter-based generator:
# splitmix64 keyed by (seed, stream), at an index. int64 arithmetic wraps.

def _i64(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _shr(z, n):
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    z = z + _i64(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _i64(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def draws(seed, stream, index):
    key = torch.tensor(_i64(seed ^ ((stream * 0xD1B54A32D192ED03) & ((1 << 64) - 1))), device="cuda")
    return _mix(_mix(key) + index)


def f16_scales(seed, stream, index, lo, hi):
    u = _shr(draws(seed, stream ^ 0x5CA1E, index), 40).double()
    return (lo + (hi - lo) * (u / 16777216.0)).float().half().double()


def weight(case, seed, layer, name, stream, N, K):
    """The dequantised matrix [N, K] in 64 bits."""
    if case["scales"] == "f32":
        codes, sc = f32_weight(seed, layer, name, N, K)
        return codes.double() * sc.double().repeat_interleave(64, 1)[:, :K]
    W = torch.empty((N, K), dtype=torch.float64, device="cuda")
    ng = -(-K // 32)
    for a in range(0, N, 4096):   # rows at a time: the generator's 64-bit values take room
        b = min(N, a + 4096)
        r = draws(seed, stream, torch.arange(a * K, b * K, device="cuda"))
        s = (r & 0xFFFF) + (_shr(r, 16) & 0xFFFF) + (_shr(r, 32) & 0xFFFF) + _shr(r, 48) - 131070
        codes = ((s * 277 + 131072) >> 18).clamp(-127, 127).double().view(b - a, K)
        sc = f16_scales(seed, stream, torch.arange(a * ng, b * ng, device="cuda"), 1e-4, 4e-4).view(b - a, ng)
        W[a:b] = codes * sc.repeat_interleave(32, 1)[:, :K]
    return W


def cached(d, seed, key, layer, which, tokens):
    """A chat's K (which 0) or V rows before the pass, [nKV, tokens, D]."""
    nkv, D, stream = d["n_kv_heads"], d["head_dim"], 0x4B560000 + layer * 2 + which
    base = ((key << 24) + torch.arange(tokens, device="cuda"))[:, None] * nkv + torch.arange(nkv, device="cuda")
    r = draws(seed, stream, base[..., None] * D + torch.arange(D, device="cuda"))
    codes = (_shr(r, 8) % 255 - 127).double()
    return (codes * f16_scales(seed, stream, base, 0.005, 0.02)[..., None]).permute(1, 0, 2)


def quantised(v):
    """store_kv: int8 codes by 32 values, scale = largest / 127."""
    g = v.reshape(*v.shape[:-1], -1, 32)
    sc = g.abs().amax(-1, keepdim=True) / 127.0
    q = torch.where(sc > 0, g / sc.clamp_min(1e-300), torch.zeros_like(g)).round().clamp(-127, 127)
    return (q * sc).reshape(v.shape)


def rmsnorm(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def rope(x, pos, d):
    """Split-half RoPE over the first rot_dim channels of x [..., rows, D]."""
    rot = d.get("rot_dim") or d["head_dim"]
    inv = torch.pow(torch.tensor(float(d["rope_theta"]), dtype=torch.float64),
                    -2.0 * torch.arange(rot // 2, dtype=torch.float64) / rot)
    sc = d.get("rope_scaling")
    if sc:   # the llama3 rule
        old, lof, hif = sc["original_max_position_embeddings"], sc["low_freq_factor"], sc["high_freq_factor"]
        wl = 2 * math.pi / inv
        sm = (old / wl - lof) / (hif - lof)
        mid = sm * inv + (1 - sm) * inv / sc["factor"]
        inv = torch.where(wl < old / hif, inv, torch.where(wl > old / lof, inv / sc["factor"], mid))
    ang = pos.double()[:, None] * inv.cuda()
    a, b, rest = x[..., :rot // 2], x[..., rot // 2:rot], x[..., rot:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), rest], -1)


def attention(case, d, seed, layer, h, jobs, W, p, kv):
    """The attention half on the normed rows h [rows, H]; kv[slot] holds the K/V rows of earlier passes."""
    D, nh, nkv, eps = d["head_dim"], d["n_heads"], d["n_kv_heads"], d["rms_eps"]
    q, k, v = ((h @ W[n].T).view(len(h), -1, D) for n in ("q", "k", "v"))
    if d.get("hybrid"):
        q, k = rmsnorm(q, p["q_norm"], eps), rmsnorm(k, p["k_norm"], eps)
    out, at = torch.empty((len(h), nh, D), dtype=torch.float64, device="cuda"), 0
    for slot, (past, n) in enumerate(jobs):
        if n == 0:
            continue
        pos = torch.arange(past, past + n, device="cuda")
        qs = rope(q[at:at + n].transpose(0, 1), pos, d)
        ks = quantised(rope(k[at:at + n].transpose(0, 1), pos, d))
        vs = quantised(v[at:at + n].transpose(0, 1))
        if (layer, slot) not in kv:
            kv[layer, slot] = [cached(d, seed, slot + 1, layer, w, past) for w in (0, 1)]
        K, V = (torch.cat([o[:, :past], x], 1) for o, x in zip(kv[layer, slot], (ks, vs)))
        kv[layer, slot] = [K, V]
        s = qs.reshape(nkv, nh // nkv * n, D) @ K.transpose(1, 2) / math.sqrt(D)
        s = s.view(nh, n, -1).masked_fill(torch.arange(past + n, device="cuda") > pos[:, None], -math.inf)
        o = torch.softmax(s, -1).view(nkv, nh // nkv * n, -1) @ V
        out[at:at + n] = o.view(nh, n, D).transpose(0, 1)
        at += n
    out = out.reshape(len(h), nh * D)
    return (out * torch.sigmoid(h @ W["attn_gate"].T) if d.get("hybrid") else out) @ W["o"].T


def gated_delta(d, layer, h, jobs, W, p, rec):
    """The linear_attention half on the normed rows h; rec[slot] holds (state, the last raw conv rows)."""
    nk, nv, dk, dv = (d[n] for n in ("lin_nk", "lin_nv", "lin_dk", "lin_dv"))
    kd, vd, nvp = nk * dk, nv * dv, 16 * -(-nv // 16)
    cd, eps = 2 * kd + vd, d["rms_eps"]
    y = h @ W["lin"].T
    z, b, a = y[:, cd:cd + vd], y[:, cd + vd:][:, :nv], y[:, cd + vd + nvp:][:, :nv]
    conv = torch.cat([p["conv_q"], p["conv_k"], p["conv_v"]]).double()
    core, at = torch.empty((len(h), nv, dv), dtype=torch.float64, device="cuda"), 0
    alog, dt = p["gate_params"].double().split(nv)
    for slot, (past, n) in enumerate(jobs):
        zeros = (torch.zeros((nv, dk, dv), dtype=torch.float64, device="cuda"),
                 torch.zeros((3, cd), dtype=torch.float64, device="cuda"))
        S, ring = rec.get((layer, slot), zeros)
        x = torch.cat([ring, y[at:at + n, :cd]])
        c = sum(x[i:i + n] * conv[:, i] for i in range(4))
        c = c * torch.sigmoid(c)

        def heads(t):
            t = t.view(n, nk, dk)
            t = t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-6)
            return t.repeat_interleave(nv // nk, 1)
        q, k, v = heads(c[:, :kd]) / math.sqrt(dk), heads(c[:, kd:2 * kd]), c[:, 2 * kd:].view(n, nv, dv)
        g = torch.exp(-alog.exp() * torch.nn.functional.softplus(a[at:at + n] + dt))
        beta = torch.sigmoid(b[at:at + n])
        for i in range(n):
            S = S * g[i][:, None, None]
            delta = (v[i] - (S * k[i][..., None]).sum(1)) * beta[i][:, None]
            S = S + k[i][..., None] * delta[:, None]
            core[at + i] = (S * q[i][..., None]).sum(1)
        rec[layer, slot] = (S, x[n:])
        at += n
    o = rmsnorm(core, p["gated_norm"], eps).reshape(len(h), vd)
    return (z * torch.sigmoid(z) * o) @ W["out"].T


def exact(case, seed):
    d, jobs = dims_of(case), jobs_of(case)
    eps, H = d["rms_eps"], d["hidden"]
    x = ids = None
    if case["kind"] == "model":
        ids = torch.from_numpy(np.concatenate(ids_of(case, seed)).astype(np.int64)).cuda()
        head = weight(case, seed, -1, "head", 1, d["vocab"], H)
        passes = [(head[ids].half().double(), jobs)]
    else:
        passes = [(rows_of(case, seed).double(), jobs)]
    if case["kind"] == "head":
        head = weight(case, seed, -1, "head", 1 if d.get("tied", True) else 2, d["vocab"], H)
    elif d.get("hybrid") and case["chunks"] == 0:
        passes.insert(0, (history(case, seed).double().view(-1, H), [(p - SEEDED_ROWS, SEEDED_ROWS) for p, _ in jobs]))
    kv, rec = {}, {}
    for layer in range(case["layers"] if case["kind"] != "head" else 0):
        W = {n: weight(case, seed, layer, n, s, N, K) for n, (_, s, N, K) in matrices(d, layer).items()}
        p = {n: v for n, (_, v) in norms_of(d, seed, layer).items()}
        for i, (x, js) in enumerate(passes):
            h = rmsnorm(x, p["ln1"], eps)
            x = x + (gated_delta(d, layer, h, js, W, p, rec) if is_linear(d, layer) else
                     attention(case, d, seed, layer, h, js, W, p, kv))
            h = rmsnorm(x, p["ln2"], eps)
            gate = h @ W["gate"].T
            x = x + (gate * torch.sigmoid(gate) * (h @ W["up"].T)) @ W["down"].T
            passes[i] = (x.half().double(), js)
        kv.clear()
        rec.clear()
    x = passes[-1][0]
    if case["kind"] == "stage":
        return {"rows": x}
    last = torch.tensor(np.cumsum([n for _, n in jobs]) - 1, device="cuda")
    logits = rmsnorm(x[last], uniform(H, 0.6, 1.4, "norm", seed), eps) @ head.T
    if case["kind"] == "model":
        return {"logits": logits}
    return {"logits": logits.topk(case["topk"], -1).values, "ids": None}
