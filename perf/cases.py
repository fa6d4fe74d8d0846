"""What the performance of this framework is measured on.

The framework serves the paged KV-cache attention path of an LLM engine, so the
cases are the work such an engine gives it, one layer (or one layer's share) at
a time, through the public Python entry points:

  session  one sequence through one layer of a PagedAttentionManager, as the
           engine runs it: the cache is reset for the new sequence, an earlier
           part of the conversation may be written back (its K/V rows exist
           already), the new prompt goes through the op chunk by chunk, then
           tokens are decoded one op call (append + attend) each
  decode   the stateless decode attention of one token (or a few) over paged
           K/V, layer after layer, launched eagerly or as a captured graph
  prefill  the stateless causal attention of a prompt over paged K/V
  flash    the non-paged attention op (kv_cache_per_layer = 0) over a batch
  append   the fused q/k norm -> RoPE -> page scatter of a prompt chunk
  front    the ops in front of the attention, node by node as the reference's
           graph has them: hidden norm, Q/K/V projections, head norms, RoPE

Shapes are the repository's own: 16 q / 8 kv heads of 128 (Qwen3-0.6B and 1.7B),
32 / 8 of 128 (Qwen3-4B), 8 / 2 of 256 with 64 rotated dims (Qwen3.5), and
generic head counts of the tests in the drawn cases.  Activations and K/V are
N(0, 1), gammas U(0.5, 1.5), pages come from a shuffled pool where the entry
point takes a page table.
"""
import math

import torch

from genllm_amd import paged

PAGE = 16
EPS = 1e-6
THETA = 1e6
POS_ROWS = 16384  # rows of the RoPE tables


def _session(name, hq, hkv, d, prefix, prompt, chunk, steps, dtype="bf16"):
    return {"name": name, "kind": "session", "hq": hq, "hkv": hkv, "d": d, "prefix": prefix, "prompt": prompt,
            "chunk": chunk, "steps": steps, "dtype": dtype}


def _decode(name, hq, hkv, d, layers, n, s, graph):
    return {"name": name, "kind": "decode", "hq": hq, "hkv": hkv, "d": d, "layers": layers, "n": n, "s": s,
            "graph": graph}


def listed():
    return [
        # a short question to a small model on fp16 layers: tiny calls, where latency and launches count
        _session("session_short_f16", 16, 8, 128, 0, 40, 40, 16, "f16"),
        # a long prompt, prefilled in chunks so that other work can run between them (Qwen3-4B)
        _session("session_prompt_4k", 32, 8, 128, 0, 4096, 512, 0),
        # the next turn of a conversation: 8K tokens written back, 64 new ones, then the answer (Qwen3-4B)
        _session("session_turn_8k", 32, 8, 128, 8192, 64, 64, 8),
        # a resumed conversation with a ragged prompt at head_dim 256 (Qwen3.5)
        _session("session_turn_d256", 8, 2, 256, 1000, 700, 128, 8),
        # one decode call over a short context (Qwen3-0.6B, 1K tokens in 64 pages): the smallest call
        _decode("decode_1k", 16, 8, 128, 1, 1024, 1, False),
        # a decode step's attention over 8 layers at 8K context, captured once and replayed (Qwen3-4B)
        _decode("decode_layers_8k", 32, 8, 128, 8, 8193, 1, True),
        # one layer of a long-context decode step, the last page partly filled (Qwen3-4B)
        _decode("decode_32k", 32, 8, 128, 1, 32761, 1, False),
        # a whole 2K prompt in one call (Qwen3-1.7B)
        {"name": "prefill_2k", "kind": "prefill", "hq": 16, "hkv": 8, "d": 128, "n": 2048, "s": 2048, "causal": True},
        # two prompts of a ragged 1000 tokens without a cache (Qwen3-1.7B)
        {"name": "flash_batch", "kind": "flash", "b": 2, "hq": 16, "hkv": 8, "d": 128, "s": 1000, "causal": True},
        # one 4096-token chunk's norm, RoPE and scatter, q with it (Qwen3-4B)
        {"name": "append_4k", "kind": "append", "hq": 32, "hkv": 8, "d": 128, "rope": 128, "s": 4096},
        # the front of a decode step, one token, as a captured graph (Qwen3-4B)
        {"name": "front_decode", "kind": "front", "hidden": 2560, "hq": 32, "hkv": 8, "d": 128, "rope": 128, "rows": 1,
         "bias": False, "graph": True},
        # the front of a prompt chunk, projections with biases (Qwen3-4B)
        {"name": "front_chunk", "kind": "front", "hidden": 2560, "hq": 32, "hkv": 8, "d": 128, "rope": 128,
         "rows": 1500, "bias": True, "graph": False},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["session", "session", "session", "decode", "decode", "prefill", "flash", "append", "front"])
    hq, hkv, d = rng.choice([(16, 8, 128), (32, 8, 128), (32, 8, 128), (8, 2, 256), (8, 8, 128), (16, 1, 128),
                             (12, 4, 128), (16, 4, 256)])
    if kind == "session":
        dtype = rng.choice(["bf16", "bf16", "f16"])
        prompt = _log(rng, 5, 4096 if d == 128 else 2048)
        prefix = 0 if dtype == "f16" else rng.choice([0, _log(rng, 100, 8192 - prompt)])
        chunk = min(prompt, max(_log(rng, 5, 1024), -(-prompt // 12)))
        return _session("", hq, hkv, d, prefix, prompt, chunk, rng.choice([0, 1, _log(rng, 2, 24)]), dtype)
    if kind == "decode":
        s = rng.choice([1, 1, 1, 2, 3]) if hq // hkv <= 4 else 1
        n = _log(rng, 17, 32768)
        layers = max(1, min(8, 32768 // n)) if rng.random() < 0.5 else 1
        return _decode("", hq, hkv, d, layers, n, s, layers > 1)
    if kind == "prefill":
        s = _log(rng, 17, 2048)
        return {"kind": kind, "hq": hq, "hkv": hkv, "d": d, "n": s + rng.choice([0, _log(rng, 16, 2048)]), "s": s,
                "causal": rng.random() < 0.9}
    if kind == "flash":
        return {"kind": kind, "b": rng.choice([1, 2, 3, 4]), "hq": hq, "hkv": hkv, "d": d, "s": _log(rng, 5, 1024),
                "causal": rng.random() < 0.8}
    if kind == "append":
        return {"kind": kind, "hq": hq, "hkv": hkv, "d": d, "rope": d if d == 128 else 64, "s": _log(rng, 1, 4096)}
    hidden, hq, hkv = rng.choice([(1024, 16, 8), (2048, 16, 8), (2560, 32, 8)])
    rows = rng.choice([1, 2, _log(rng, 5, 1500)])
    return {"kind": kind, "hidden": hidden, "hq": hq, "hkv": hkv, "d": 128, "rope": 128, "rows": rows,
            "bias": rng.random() < 0.5, "graph": rows <= 4}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype=torch.bfloat16, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _gamma(g, n):
    return torch.rand(n, generator=g, device="cuda") + 0.5


def _perm(g, n):
    return torch.randperm(n, generator=g, device="cuda").to(torch.int32)


def _tables(rope_dim, rows):
    cos, sin = paged.rope_cache(THETA, rope_dim, rows)
    return torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()


class _Pool:
    """A layer's K or V pool as a tensor that keeps its manager alive."""

    def __init__(self, mgr, ptr, shape):
        self.mgr = mgr
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i2", "data": (ptr, False), "version": 3,
                                         "strides": None}


def _manager(c, pages, dtype):
    hkv, d = c["hkv"], c["d"]
    mgr = paged.PagedAttentionManager(2 * pages * PAGE * hkv * d * 2 + 4096)
    mgr.init_layer(0, hkv, d, paged.DTYPE_F16 if dtype == torch.float16 else paged.DTYPE_BF16)
    mgr.reserve_layer(0, pages)
    info = mgr.get_layer(0)
    shape = (pages, PAGE, hkv, d)
    return mgr, [torch.as_tensor(_Pool(mgr, p, shape), device="cuda").view(dtype) for p in (info.k_pool, info.v_pool)]


def _fill_blocks(mgr, pages):
    """Hands every block out once, so that each reset returns all of them to
    the free lists in one order (a pool that has been in use)."""
    mgr.append_kv_pages(0, pages * PAGE)
    mgr.reset()


def _cuts(total, piece):
    return [(a, min(a + piece, total)) for a in range(0, total, piece)]


def _inputs(c, seed):
    """The named input tensors of a case: made from the seed alone."""
    g = _gen(seed)
    k = c["kind"]
    if k == "session":
        dt = torch.float16 if c["dtype"] == "f16" else torch.bfloat16
        n, t = c["prompt"], c["steps"]
        return {
            "prefix": [_normal(g, (c["prefix"], c["hkv"], c["d"]), dt) for _ in range(2)],
            "chunks": [[_normal(g, (1, h, b - a, c["d"]), dt) for h in (c["hq"], c["hkv"], c["hkv"])]
                       for a, b in _cuts(n, c["chunk"])],
            "steps": [[_normal(g, (1, h, 1, c["d"]), dt) for h in (c["hq"], c["hkv"], c["hkv"])] for _ in range(t)],
        }
    if k == "decode":
        pages = -(-c["n"] // PAGE)
        pool = pages + pages // 4 + 1  # a pool that other sequences use as well
        lay = []
        for _ in range(c["layers"]):
            lay.append([_normal(g, (pool, PAGE, c["hkv"], c["d"])) for _ in range(2)] +
                       [_perm(g, pool)[:pages].contiguous() for _ in range(2)] +
                       [_normal(g, (c["hq"], c["s"], c["d"]))])
        return {"layers": lay}
    if k == "prefill":
        pages = -(-c["n"] // PAGE)
        return {"kv": [_normal(g, (pages + 3, PAGE, c["hkv"], c["d"])) for _ in range(2)],
                "ids": [_perm(g, pages + 3)[:pages].contiguous() for _ in range(2)],
                "q": _normal(g, (c["s"], c["hq"], c["d"]))}  # token-major, as the projection writes it
    if k == "flash":
        return {"q": _normal(g, (c["b"], c["hq"], c["s"], c["d"])),
                "kv": [_normal(g, (c["b"], c["hkv"], c["s"], c["d"])) for _ in range(2)]}
    if k == "append":
        return {"q": _normal(g, (c["s"], c["hq"], c["d"])),
                "kv": [_normal(g, (c["s"], c["hkv"], c["d"])) for _ in range(2)],
                "gamma": [_gamma(g, c["d"]) for _ in range(2)]}
    heads = (c["hq"], c["hkv"], c["hkv"])
    return {"x": _normal(g, (c["rows"], c["hidden"])), "gamma": [_gamma(g, c["hidden"])] + [_gamma(g, c["d"]) for _ in range(2)],
            "w": [_normal(g, (h * c["d"], c["hidden"]), std=0.05) for h in heads],
            "b": [_normal(g, (h * c["d"],)) if c["bias"] else None for h in heads],
            "pos": int(torch.randint(0, POS_ROWS - c["rows"], (1,), generator=g, device="cuda"))}


def prepare(case, seed):
    c = case
    s = {"c": c, "in": _inputs(c, seed)}
    i, k = s["in"], c["kind"]
    s["scale"] = 1.0 / math.sqrt(c["d"])
    if k == "session":
        dt = torch.float16 if c["dtype"] == "f16" else torch.bfloat16
        pages = -(-(c["prefix"] + c["prompt"] + c["steps"]) // PAGE)
        s["mgr"], s["pools"] = _manager(c, pages, dt)
        _fill_blocks(s["mgr"], pages)
        s["prefix"] = [(i["prefix"][0][a:b], i["prefix"][1][a:b]) for a, b in _cuts(c["prefix"], 4096)]
        s["calls"] = [(q, kk, v, torch.empty_like(q)) for q, kk, v in i["chunks"] + i["steps"]]
    elif k == "decode":
        s["ws"] = torch.zeros(paged.decode_workspace_bytes(c["hq"], c["hkv"], c["s"], c["d"], -(-c["n"] // PAGE)),
                              dtype=torch.uint8, device="cuda")
        s["out"] = [torch.empty_like(lay[4]) for lay in i["layers"]]
    elif k == "prefill":
        s["out"] = torch.empty_like(i["q"])
    elif k == "flash":
        s["out"] = torch.empty_like(i["q"])
    elif k == "append":
        pages = -(-c["s"] // PAGE)
        s["mgr"], s["pools"] = _manager(c, pages, torch.bfloat16)
        _fill_blocks(s["mgr"], pages)
        s["tab"] = _tables(c["rope"], c["s"])
        s["q_out"] = torch.empty((c["hq"], c["s"], c["d"]), dtype=torch.bfloat16, device="cuda")
    else:
        r = c["rows"]
        s["tab"] = _tables(c["rope"], POS_ROWS)
        s["h"] = torch.empty_like(i["x"])
        s["qkv"] = [torch.empty((r, w.shape[0]), dtype=torch.bfloat16, device="cuda") for w in i["w"]]
        s["normed"] = [torch.empty((r, n, c["d"]), dtype=torch.bfloat16, device="cuda") for n in (c["hq"], c["hkv"])]
        s["roped"] = [torch.empty((n, r, c["d"]), dtype=torch.bfloat16, device="cuda") for n in (c["hq"], c["hkv"])]
        need = max(paged.linear_workspace_bytes(r, c["hidden"], w.shape[0]) for w in i["w"])
        s["ws"] = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    if c.get("graph"):
        _RUN[k](s)  # first call outside the capture
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["outs"] = _RUN[k](s)
    return s


# --------------------------------------------------------------------- run
def _run_session(s):
    c, mgr = s["c"], s["mgr"]
    groups, scale = c["hq"] // c["hkv"], s["scale"]
    mgr.reset()
    for k, v in s["prefix"]:  # rows as an earlier pass left them: no norm, no RoPE
        paged.qk_norm_rope_append(mgr, 0, k, v, None, EPS, None, None, 0)
    for q, k, v, out in s["calls"]:
        paged.paged_attention(mgr, 0, q, k, v, out, groups, scale)
    return {"out": [x[3] for x in s["calls"]], "pools": s["pools"]}


def _run_decode(s):
    c, pages = s["c"], -(-s["c"]["n"] // PAGE)
    for (k, v, kid, vid, q), out in zip(s["in"]["layers"], s["out"]):
        paged.paged_decode(q, out, k, v, kid, vid, pages, c["n"], c["hkv"], s["scale"], s["ws"])
    return s["out"]


def _run_prefill(s):
    c, i = s["c"], s["in"]
    paged.paged_prefill(i["q"], s["out"], i["kv"][0], i["kv"][1], i["ids"][0], i["ids"][1], -(-c["n"] // PAGE), c["n"],
                        c["hkv"], s["scale"], c["causal"], "token")
    return s["out"]


def _run_flash(s):
    c, i = s["c"], s["in"]
    paged.flash_attention(i["q"], i["kv"][0], i["kv"][1], s["out"], c["hq"] // c["hkv"], s["scale"], c["causal"])
    return s["out"]


def _run_append(s):
    i, mgr = s["in"], s["mgr"]
    mgr.reset()
    paged.qk_norm_rope_append(mgr, 0, i["kv"][0], i["kv"][1], i["gamma"][1], EPS, s["tab"][0], s["tab"][1], 0, i["q"],
                              i["gamma"][0], s["q_out"])
    return {"q": s["q_out"], "pools": s["pools"]}


def _run_front(s):
    c, i = s["c"], s["in"]
    paged.rms_norm(s["h"], i["x"], i["gamma"][0], EPS)
    for w, b, out in zip(i["w"], i["b"], s["qkv"]):
        paged.linear(s["h"], w, out, b, s["ws"])
    for n in range(2):
        x, d = s["normed"][n], c["d"]
        paged.rms_norm(x, s["qkv"][n], i["gamma"][1 + n], EPS)
        x = x.view(x.shape[1], 1, d) if c["rows"] == 1 else x.transpose(0, 1).contiguous()
        paged.apply_rope(s["roped"][n], x, s["tab"][0], s["tab"][1], i["pos"])
    return {"q": s["roped"][0], "k": s["roped"][1], "v": s["qkv"][2]}


_RUN = {"session": _run_session, "decode": _run_decode, "prefill": _run_prefill, "flash": _run_flash,
        "append": _run_append, "front": _run_front}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    return _RUN[state["c"]["kind"]](state)


# -------------------------------------------------------------------- work
def _pairs(n, s, causal=True):
    """(query, key) pairs of s queries at the end of n keys."""
    return s * (n - s) + s * (s + 1) // 2 if causal else s * n


def work(case):
    c = case
    k, hq, hkv, d = c["kind"], c["hq"], c["hkv"], c["d"]
    row = hkv * d * 4  # K and V bytes of one token
    if k == "session":
        n, moved, pairs = c["prefix"], 2 * c["prefix"] * row, 0
        for a, b in _cuts(c["prompt"], c["chunk"]) + [(0, 1)] * c["steps"]:
            s = b - a
            moved += 2 * s * row + n * row + 4 * s * hq * d  # append, the earlier keys, q and out
            n += s
            pairs += _pairs(n, s)
        return {"bytes": moved, "flops": 4 * d * hq * pairs}
    if k == "decode":
        return {"bytes": c["layers"] * (c["n"] * row + 8 * -(-c["n"] // PAGE) + 4 * c["s"] * hq * d),
                "flops": c["layers"] * 4 * d * hq * _pairs(c["n"], c["s"])}
    if k == "prefill":
        return {"bytes": c["n"] * row + 4 * c["s"] * hq * d, "flops": 4 * d * hq * _pairs(c["n"], c["s"], c["causal"])}
    if k == "flash":
        return {"bytes": c["b"] * c["s"] * (row + 4 * hq * d),
                "flops": 4 * d * hq * c["b"] * _pairs(c["s"], c["s"], c["causal"])}
    if k == "append":
        return {"bytes": c["s"] * (2 * row + 4 * hq * d + 4 * c["rope"]), "flops": c["s"] * (hq + hkv) * d * 8}
    cols, r = (hq + 2 * hkv) * d, c["rows"]
    return {"bytes": 2 * cols * c["hidden"] + r * (2 * c["hidden"] + 2 * cols + 4 * c["rope"]),
            "flops": 2 * r * cols * c["hidden"]}


def tolerance(case):
    """About four times the error against 64 bits that each path shows: 2.4e-3
    for attention in bf16 and 2.6e-4 in fp16 (results and probabilities in 16
    bits), 3.7e-3 for norm and RoPE (the norm's truncating store), 4.5e-3 for
    the front."""
    rel = {"append": 1.5e-2, "front": 1.8e-2}.get(case["kind"], 1e-2)
    if case.get("dtype") == "f16":
        return {"rel": 1.1e-3, "max": 0.01}
    return {"rel": rel, "max": 0.05}


# ------------------------------------------------------------------- exact
def _attend(q, k, v, groups, scale, causal):
    """q [Hq][S][D] at the end of k, v [Hkv][N][D], in 64 bits."""
    hq, s, d = q.shape
    n = k.shape[1]
    out = torch.empty((hq, s, d), dtype=torch.float64, device="cuda")
    keys = torch.arange(n, device="cuda")
    for h in range(hq):
        kd, vd = k[h // groups].double(), v[h // groups].double()
        for a, b in _cuts(s, 1024):
            x = q[h, a:b].double() @ kd.t() * scale
            if causal:
                x = x.masked_fill(keys[None, :] > (n - s + torch.arange(a, b, device="cuda"))[:, None], -math.inf)
            out[h, a:b] = torch.softmax(x, 1) @ vd
    return out


def _norm(x, gamma):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _rope(x, pos0, rope_dim):
    """x [S][H][D] at positions pos0 + s: dims (i, i + rope_dim / 2) rotate."""
    half = rope_dim // 2
    inv = THETA ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / rope_dim)
    a = (pos0 + torch.arange(x.shape[0], device="cuda", dtype=torch.float64))[:, None, None] * inv
    x0, x1 = x[..., :half], x[..., half:rope_dim]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos(), x[..., rope_dim:]], -1)


def _paged_rows(rows, pages):
    """Token rows [N][Hkv][D] in a pool whose blocks are handed out from the last down."""
    full = torch.zeros((pages * PAGE,) + tuple(rows.shape[1:]), dtype=torch.float64, device="cuda")
    full[: rows.shape[0]] = rows.double()
    return full.view(pages, PAGE, *rows.shape[1:]).flip(0)


def exact(case, seed):
    c, i = case, _inputs(case, seed)
    k, scale = c["kind"], 1.0 / math.sqrt(c["d"])
    groups = c["hq"] // c["hkv"]
    if k == "session":
        kv = [x.transpose(0, 1) for x in i["prefix"]]  # [Hkv][N][D]
        outs = []
        for q, kk, v in i["chunks"] + i["steps"]:
            kv = [torch.cat([kv[0], kk[0]], 1), torch.cat([kv[1], v[0]], 1)]
            outs.append(_attend(q[0], kv[0], kv[1], groups, scale, True)[None])
        pages = -(-kv[0].shape[1] // PAGE)
        return {"out": outs, "pools": [_paged_rows(x.transpose(0, 1), pages) for x in kv]}
    if k == "decode":
        got = []
        for kp, vp, kid, vid, q in i["layers"]:
            rows = [p[ids.long()].reshape(-1, c["hkv"], c["d"])[: c["n"]].transpose(0, 1) for p, ids in ((kp, kid), (vp, vid))]
            got.append(_attend(q, rows[0], rows[1], groups, scale, True))
        return got
    if k == "prefill":
        rows = [p[ids.long()].reshape(-1, c["hkv"], c["d"])[: c["n"]].transpose(0, 1) for p, ids in zip(i["kv"], i["ids"])]
        return _attend(i["q"].transpose(0, 1), rows[0], rows[1], groups, scale, c["causal"]).transpose(0, 1).contiguous()
    if k == "flash":
        return torch.stack([_attend(i["q"][b], i["kv"][0][b], i["kv"][1][b], groups, scale, c["causal"])
                            for b in range(c["b"])])
    if k == "append":
        pages = -(-c["s"] // PAGE)
        kr = _rope(_norm(i["kv"][0], i["gamma"][1]), 0, c["rope"])
        qr = _rope(_norm(i["q"], i["gamma"][0]), 0, c["rope"])
        return {"q": qr.transpose(0, 1).contiguous(), "pools": [_paged_rows(kr, pages), _paged_rows(i["kv"][1], pages)]}
    h = _norm(i["x"], i["gamma"][0])
    qkv = [h @ w.double().t() + (b.double() if b is not None else 0.0) for w, b in zip(i["w"], i["b"])]
    roped = [_rope(_norm(x.view(c["rows"], -1, c["d"]), i["gamma"][1 + n]), i["pos"], c["rope"]).transpose(0, 1).contiguous()
             for n, x in enumerate(qkv[:2])]
    return {"q": roped[0], "k": roped[1], "v": qkv[2]}
