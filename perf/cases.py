"""The framework's work as its users have it done, case by case, for timing.

Each case is one call sequence of a serving program through the package's public entry points:
decode, verify and prefill attention steps over paged KV pools, the engine's own step, the
query/key rotation with its append, FP8 page quantisation, sampling, and page transfers.

    listed()            the cases, by name
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the program holds before the call: pools, tables, plans, handles
    run(state)          one pass; its outputs whole
    work(case)          the bytes and operations a pass cannot do without
    exact(case, seed)   the pass in 64 bits, in plain torch
    tolerance(case)     how far two correct implementations may be apart

A ragged batch is given by two texts: `new`, the step's rows of each sequence, and `cached`, the
keys each sequence already has.  Pool pages are scattered by a seeded permutation.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

F32, F16, BF16, FP8 = 0, 1, 2, 3
CODE = {"f32": F32, "f16": F16, "bf16": BF16, "fp8": FP8}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


def package():
    """The package of the working folder's tree (its folder name is no Python identifier)."""
    if "lia_rs_amd" not in sys.modules:
        folder = os.path.join(os.getcwd(), "lia.rs_amd")
        spec = importlib.util.spec_from_file_location(
            "lia_rs_amd", os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
        sys.modules["lia_rs_amd"] = module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
    return sys.modules["lia_rs_amd"]


# ------------------------------------------------------------------ the cases

def _text(values):
    return ",".join(str(int(v)) for v in values)


def _ints(text):
    return np.array([int(v) for v in text.split(",")], dtype=np.int64)


def _step(name, new, cached, hq=16, hkv=2, d=128, page=16, kv="bf16", q="bf16", out="bf16", layers=1):
    case = dict(kind="step", new=_text(new), cached=_text(cached), hq=hq, hkv=hkv, d=d, page=page,
                kv=kv, q=q, out=out, layers=layers)
    return dict(name=name, **case) if name else case


def listed():
    r = np.random.default_rng(0)
    ctx8 = r.integers(1024, 32768, size=8, endpoint=True)
    r = np.random.default_rng(0)
    dec5 = r.integers(2048, 16384, size=5, endpoint=True)
    r = np.random.default_rng(0)
    new32 = 1 + r.integers(1, 3, size=32, endpoint=True)
    ctx32 = r.integers(512, 16384, size=32, endpoint=True)
    r = np.random.default_rng(0)
    ctx64 = np.exp(r.uniform(np.log(1024), np.log(131072), size=64)).astype(np.int64)
    ones = lambda n: np.ones(n, np.int64)  # noqa: E731
    return [
        # the smallest step of a server that has just started: four short chats, two layers
        _step("decode_short", ones(4), np.array([17, 64, 200, 511]) - 1, hq=8, d=64, layers=2),
        # one user's chat through the engine object with its default types, four layers
        dict(name="engine_chat", kind="engine", new="1", cached="6001", hq=16, hkv=2, d=128, page=32,
             kv="f16", layers=4),
        # the ordinary decode step: eight ragged contexts, four layers on one plan
        _step("decode_b8", ones(8), ctx8 - 1, layers=4),
        # speculative decoding: 32 sequences verify two or three rows each, two layers
        _step("verify_b32", new32, ctx32 - new32, layers=2),
        # the fullest decode step: 64 sequences of up to 128k keys on an FP8 pool
        _step("decode_fp8_b64", ones(64), ctx64 - 1, kv="fp8"),
        # continuous batching: three prompt chunks (two over cached prefixes) beside five decodes
        _step("prefill_mixed", [512, 1024, 2048, 1, 1, 1, 1, 1], [0, 4096, 8192, *(dec5 - 1)]),
        # four odd prompt chunks on an FP8 pool with more heads
        _step("prefill_fp8", [777, 1500, 33, 2048], [0, 3001, 12000, 513], hq=32, hkv=8, kv="fp8"),
        # a prompt chunk of 512 rows as the model's attention block does it on the engine's default
        # types: coefficients, rotation with the append, attention, the gather of the output rows
        dict(name="block_chunk", kind="block", new="300,212", cached="1700,0", hq=16, hkv=2, d=128,
             page=32, kv="f16", q="f32"),
        # the rotation and append of a large packed batch on bf16
        dict(name="rope_append", kind="rope", rows=4096, first=3000, hq=16, hkv=2, d=128, page=16,
             kv="bf16", q="bf16"),
        # finished pages of a long prompt quantised to FP8
        dict(name="quantize_pages", kind="quantize", pages=2048, hkv=2, d=128, page=16, src="bf16"),
        # the sampling of a full batch of output rows, greedy, top-k and nucleus requests mixed
        dict(name="sample_b64", kind="sample", rows=64, vocab=130560),
        # the page cache's window: 16 pages of 42 layers restored and 16 saved
        dict(name="page_swap", kind="swap", pages=16, hkv=2, d=128, page=32, kv="f16", layers=42),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "prefill", "prefill", "engine", "block", "rope",
                       "quantize", "sample", "swap"])
    heads = dict(zip(("hq", "hkv", "d"), rng.choice([(16, 2, 128), (16, 2, 128), (32, 8, 128), (8, 2, 64)])))
    page = rng.choice([16, 16, 32, 64])
    kv = rng.choice(["bf16", "f16", "fp8"])
    if kind in ("decode", "verify"):
        n = _log(rng, 1, 64)
        new = [1 if kind == "decode" else rng.randint(2, 4) for _ in range(n)]
        top = _log(rng, 64, 65536)
        cached = [_log(rng, 1, top) for _ in range(n)]
        q = rng.choice(["bf16", "bf16", "f32"])
        case = _step(None, new, cached, page=page, kv=kv, q=q, out=q, layers=rng.randint(1, 4), **heads)
        while work(case)["bytes"] > 8e8:
            cached = [max(1, c // 2) for c in cached]
            case["cached"] = _text(cached)
        return case
    if kind == "prefill":
        n = rng.randint(1, 6)
        new = [_log(rng, 17, 2048) for _ in range(n)]
        cached = [rng.choice([0, _log(rng, 1, 12000)]) for _ in range(n)]
        more = rng.randint(0, min(6, sum(new) // 16 - n)) if sum(new) // 16 > n else 0  # decodes beside them
        new += [1] * more
        cached += [_log(rng, 100, 16000) for _ in range(more)]
        case = _step(None, new, cached, page=page, kv=kv, **heads)
        while work(case)["flops"] > 1.9e11:
            cached = [c // 2 for c in cached]
            new = [max(1, c * 3 // 4) for c in new]
            case.update(new=_text(new), cached=_text(cached))
        return case
    if kind == "engine":
        n = _log(rng, 1, 16)
        return dict(kind="engine", new=_text([1] * n), cached=_text([_log(rng, 16, 12000) for _ in range(n)]),
                    page=rng.choice([16, 32]), kv=rng.choice(["f16", "bf16"]), layers=rng.randint(1, 4), **heads)
    if kind == "block":
        n = rng.randint(1, 4)
        return dict(kind="block", new=_text([_log(rng, 9, 512 // n) for _ in range(n)]),
                    cached=_text([rng.choice([0, _log(rng, 1, 6000)]) for _ in range(n)]), page=page,
                    kv=rng.choice(["f16", "bf16"]), q=rng.choice(["f32", "bf16"]), **heads)
    if kind == "rope":
        return dict(kind="rope", rows=_log(rng, 1, 8192), first=_log(rng, 1, 60000), page=page, kv=kv,
                    q=rng.choice(["f32", "bf16"]), **heads)
    if kind == "quantize":
        return dict(kind="quantize", pages=_log(rng, 1, 2048), hkv=heads["hkv"], d=heads["d"], page=page,
                    src=rng.choice(["bf16", "f32", "f16"]))
    if kind == "sample":
        return dict(kind="sample", rows=_log(rng, 1, 64), vocab=rng.choice([1000, 32000, 73448, 130560]))
    return dict(kind="swap", pages=rng.randint(1, 16), hkv=2, d=heads["d"], page=rng.choice([16, 32]),
                kv=kv, layers=_log(rng, 1, 42))


# ------------------------------------------------------------------ inputs (plain torch)

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _i32(values):
    return torch.from_numpy(np.asarray(values, np.uint32).view(np.int32).copy()).to(DEV)


class _Batch:
    """The ragged batch of a case: per-sequence counts and a block table of scattered pages."""

    def __init__(self, case, seed, slack=5):
        self.new, self.cached, P = _ints(case["new"]), _ints(case["cached"]), case["page"]
        self.ctx = self.new + self.cached
        self.n, self.rows, self.page = len(self.new), int(self.new.sum()), P
        need = -(-self.ctx // P)
        self.pool_pages = int(need.sum()) + slack
        perm = np.random.default_rng(seed).permutation(self.pool_pages).astype(np.uint32)
        at = np.concatenate([[0], np.cumsum(need)])
        self.tables = [perm[at[i]:at[i + 1]] for i in range(self.n)]
        self.stride = int(need.max()) + 1
        flat = np.full((self.n, self.stride), 0xFFFFFFFF, np.uint32)
        for i, t in enumerate(self.tables):
            flat[i, :len(t)] = t
        self.flat = flat.reshape(-1)
        self.positions = np.concatenate([np.arange(c, c + m) for c, m in zip(self.cached, self.new)])
        self.sequences = np.repeat(np.arange(self.n), self.new)
        self.cu = np.concatenate([[0], np.cumsum(self.new)])
        page = flat[self.sequences, self.positions // P]
        self.slots = page.astype(np.int64) * P + self.positions % P


def _plane(g, tokens, hkv, d, kv):
    """One pool plane [tokens][hkv][d] of N(0, 1) keys or values, and its FP8 page scales' values."""
    if kv == "fp8":  # codes of a page whose largest value is about 3.6 standard deviations
        return (_randn(g, tokens, hkv, d) * 125.0).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    return _randn(g, tokens, hkv, d).to(TORCH[kv])


def _scales(g, pages, hkv):
    return (1.0 + 0.25 * torch.rand(pages * hkv, generator=g, device=DEV)) / 125.0


def _layers(case, batch, seed):
    """Each layer's pool planes, scales and the step's rows."""
    g, hkv, d, kv = _gen(seed), case["hkv"], case["d"], case["kv"]
    tokens = batch.pool_pages * case["page"]
    got = []
    for _ in range(case.get("layers", 1)):
        t = dict(k=_plane(g, tokens, hkv, d, kv), v=_plane(g, tokens, hkv, d, kv))
        if kv == "fp8":
            t["ks"], t["vs"] = _scales(g, batch.pool_pages, hkv), _scales(g, batch.pool_pages, hkv)
        row_type = torch.bfloat16 if kv == "fp8" else TORCH[kv]
        t["q"] = _randn(g, batch.rows, case["hq"], d).to(TORCH[case.get("q", "f32")])
        t["new_k"] = _randn(g, batch.rows, hkv * d).to(row_type)
        t["new_v"] = _randn(g, batch.rows, hkv * d).to(row_type)
        got.append(t)
    return got


def _logits(case, seed):
    """Peaked rows, as a language model's: a broad body and a few dozen likely tokens."""
    g = _gen(seed)
    x = 1.5 * _randn(g, case["rows"], case["vocab"])
    likely = torch.randint(0, case["vocab"], (case["rows"], 40), generator=g, device=DEV)
    return x.scatter_add_(1, likely, 6.0 + 8.0 * torch.rand(likely.shape, generator=g, device=DEV))


def _bits(t):
    """A tensor's storage as whole numbers, for outputs that are bytes and not computed values."""
    return t if t.dtype == torch.uint8 else t.view(torch.int16)


# ------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _config(lia, case, b, q, out):
    return lia.AttentionConfig(case["hq"], case["hkv"], case["d"], case["page"], b.pool_pages, b.stride,
                               CODE[q], CODE[case["kv"]], CODE[out], 1.0 / math.sqrt(case["d"]), b.n,
                               b.rows, int(b.ctx.max()))


def _prepare_step(case, seed):
    lia, b = package(), _Batch(case, seed)
    layers = _layers(case, b, seed)
    cfg = _config(lia, case, b, case["q"], case["out"])
    for t in layers:
        t["o"] = torch.empty((b.rows, case["hq"], case["d"]), dtype=TORCH[case["out"]], device=DEV)
    z = lambda n: torch.zeros(n, dtype=torch.int32, device=DEV)  # noqa: E731
    return dict(run=_run_step, lia=lia, b=b, cfg=cfg, layers=layers, fp8=case["kv"] == "fp8",
                slots_of=_i32(np.arange(b.n)), q_lens=_i32(b.new), cached=_i32(b.cached), flat=_i32(b.flat),
                cu=z(b.n + 1), positions=z(b.rows), sequences=z(b.rows), slots=z(b.rows), status=z(1),
                ws=torch.zeros(lia.workspace_bytes(cfg), dtype=torch.uint8, device=DEV))


def _run_step(s):
    """Packing and plan once, then each layer's attention with its append fused in, and the combine."""
    lia, b, cfg, ws, flat = s["lia"], s["b"], s["cfg"], s["ws"], s["flat"]
    lia.pack_plan_device(cfg, s["slots_of"], s["q_lens"], s["cached"], flat, b.rows, b.stride * b.page,
                         s["cu"], s["positions"], s["sequences"], s["slots"], s["status"], ws)
    for t in s["layers"]:
        if s["fp8"]:
            lia.attention_partial_append_fp8(cfg, b.n, flat, s["slots"], t["q"], t["new_k"], t["new_v"],
                                             t["k"], t["v"], t["ks"], t["vs"], t["o"], ws)
        else:
            lia.attention_partial_append(cfg, b.n, flat, s["slots"], t["q"], t["new_k"], t["new_v"],
                                         t["k"], t["v"], t["o"], ws)
        lia.attention_merge(cfg, b.n, b.rows, t["o"], ws)
    return dict(status=s["status"], slots=s["slots"],
                layers=[dict(o=t["o"], k=_bits(t["k"]), v=_bits(t["v"])) for t in s["layers"]])


def _prepare_engine(case, seed):
    lia, b = package(), _Batch(case, seed)
    layers = _layers(case, b, seed)
    e = lia.Engine(case["hq"], case["hkv"], case["d"], pool_tokens=b.pool_pages * case["page"],
                   layers=case["layers"], page_size=case["page"], kv_dtype=CODE[case["kv"]])
    e.configure_paging(max(8, b.n), 16384)
    for i, t in enumerate(layers):
        e.k[i].view(torch.int16).copy_(t.pop("k").view(torch.int16))
        e.v[i].view(torch.int16).copy_(t.pop("v").view(torch.int16))
    rows = [(1, int(p), int(q)) for p, q in zip(b.positions, b.sequences)]
    return dict(run=_run_engine, e=e, layers=layers, rows=rows, tables=[t.tolist() for t in b.tables],
                outputs=list(range(b.rows)))


def _run_engine(s):
    e = s["e"]
    e.stage(s["rows"], s["tables"], s["outputs"])
    outs = [e.attention(i, t["q"], t["new_k"], t["new_v"]) for i, t in enumerate(s["layers"])]
    return dict(layers=[dict(o=o, k=_bits(e.k[i]), v=_bits(e.v[i])) for i, o in enumerate(outs)])


def _combined(case, rows, seed):
    """Packed projection rows: q heads | k heads | v heads, f32."""
    return _randn(_gen(seed + 7919), rows, (case["hq"] + 2 * case["hkv"]) * case["d"])


def _prepare_block(case, seed):
    lia, b = package(), _Batch(case, seed)
    g = _gen(seed)
    tokens, d, hq = b.pool_pages * case["page"], case["d"], case["hq"]
    cfg = _config(lia, case, b, case["q"], case["q"])
    o = torch.empty((b.rows, hq, d), dtype=TORCH[case["q"]], device=DEV)
    return dict(run=_run_block, lia=lia, b=b, cfg=cfg, hq=hq, d=d, combined=_combined(case, b.rows, seed),
                layout=lia.KVLayout(case["hkv"], d, case["page"], b.pool_pages, CODE[case["kv"]]),
                k=_plane(g, tokens, case["hkv"], d, case["kv"]), v=_plane(g, tokens, case["hkv"], d, case["kv"]),
                positions=_i32(b.positions), sequences=_i32(b.sequences), cu=_i32(b.cu), flat=_i32(b.flat),
                slots=_i32(b.slots), last=_i32(b.cu[1:] - 1), query=torch.empty_like(o), o=o,
                coefficients=torch.empty((b.rows, d // 2, 2), device=DEV),
                picked=torch.empty((b.n, hq, d), dtype=o.dtype, device=DEV),
                ws=torch.zeros(lia.workspace_bytes(cfg), dtype=torch.uint8, device=DEV))


def _run_block(s):
    lia, b = s["lia"], s["b"]
    lia.rope_coefficients(s["positions"], s["d"], s["coefficients"])
    lia.rope_kv_append(s["layout"], s["hq"], s["coefficients"], s["combined"], s["query"], s["k"], s["v"],
                       slot_mapping=s["slots"])
    lia.paged_attention(s["cfg"], b.n, s["cu"], s["positions"], s["sequences"], s["flat"], s["query"], s["k"],
                        s["v"], s["o"], s["ws"])
    lia.gather_rows(s["last"], s["o"], s["picked"])
    return dict(coefficients=s["coefficients"], query=s["query"], o=s["o"], picked=s["picked"],
                k=_bits(s["k"]), v=_bits(s["v"]))


def _prepare_rope(case, seed):
    lia, g = package(), _gen(seed)
    rows, P, hkv, d = case["rows"], case["page"], case["hkv"], case["d"]
    pages = -(-rows // P) + 5
    slots = np.random.default_rng(seed).permutation(pages)[np.arange(rows) // P] * P + np.arange(rows) % P
    s = dict(run=_run_rope, lia=lia, hq=case["hq"], d=d, combined=_combined(case, rows, seed),
             layout=lia.KVLayout(hkv, d, P, pages, CODE[case["kv"]]),
             positions=_i32(case["first"] + np.arange(rows)), slots=_i32(slots),
             k=_plane(g, pages * P, hkv, d, case["kv"]), v=_plane(g, pages * P, hkv, d, case["kv"]),
             ks=None, vs=None, coefficients=torch.empty((rows, d // 2, 2), device=DEV),
             query=torch.empty((rows, case["hq"], d), dtype=TORCH[case["q"]], device=DEV))
    if case["kv"] == "fp8":
        s["ks"], s["vs"] = _scales(g, pages, hkv), _scales(g, pages, hkv)
    return s


def _run_rope(s):
    s["lia"].rope_coefficients(s["positions"], s["d"], s["coefficients"])
    s["lia"].rope_kv_append(s["layout"], s["hq"], s["coefficients"], s["combined"], s["query"], s["k"], s["v"],
                            slot_mapping=s["slots"], k_scales=s["ks"], v_scales=s["vs"])
    return dict(coefficients=s["coefficients"], query=s["query"], k=_bits(s["k"]), v=_bits(s["v"]))


def _prepare_quantize(case, seed):
    lia, g = package(), _gen(seed)
    n, P, hkv, d = case["pages"], case["page"], case["hkv"], case["d"]
    pool = n + 5
    ids = np.random.default_rng(seed).permutation(pool)[:n]
    z = lambda: torch.zeros((pool * P, hkv, d), dtype=torch.uint8, device=DEV)  # noqa: E731
    ones = lambda: torch.ones(pool * hkv, device=DEV)  # noqa: E731
    return dict(run=_run_quantize, lia=lia, ids=_i32(ids), kc=z(), vc=z(), ks=ones(), vs=ones(),
                layout=lia.KVLayout(hkv, d, P, pool, FP8),
                k=_randn(g, n * P, hkv, d).to(TORCH[case["src"]]), v=_randn(g, n * P, hkv, d).to(TORCH[case["src"]]))


def _run_quantize(s):
    s["lia"].kv_quantize_pages(s["layout"], s["ids"], s["k"], s["v"], s["kc"], s["vc"], s["ks"], s["vs"])
    return dict(k=s["kc"], v=s["vc"], ks=s["ks"], vs=s["vs"])


def _prepare_sample(case, seed):
    lia = package()
    # position-keyed draws, so that a pass can be repeated: half nucleus, a quarter each top-k and greedy
    samplers = [None if i % 4 == 3 else lia.Sampler(0.8, 20 if i % 4 == 1 else 0, 0.9, seed + i, position_keyed=True)
                for i in range(case["rows"])]
    return dict(run=_run_sample, sampler=lia.PagedSampler(case["vocab"], case["rows"]), samplers=samplers,
                logits=_logits(case, seed), positions=[100 + 37 * i for i in range(case["rows"])])


def _run_sample(s):
    return s["sampler"].sample(s["logits"], s["samplers"], s["positions"])


def _prepare_swap(case, seed):
    lia, g = package(), _gen(seed)
    P, hkv, d, n = case["page"], case["hkv"], case["d"], case["pages"]
    pool = 3 * 16
    k, v = ([_plane(g, pool * P, hkv, d, case["kv"]) for _ in range(case["layers"])] for _ in "kv")
    ks = vs = None
    if case["kv"] == "fp8":
        ks, vs = ([_scales(g, pool, hkv) for _ in k] for _ in "kv")
    t = lia.KVTransfer(lia.KVLayout(hkv, d, P, pool, CODE[case["kv"]]), k, v, ks, vs)
    r = np.random.default_rng(seed)
    ids = [int(x) for x in r.permutation(pool)]
    payloads = []
    for _ in range(n):  # saved pages: 16-bit values or codes, and scales of an FP8 pool behind them
        words = torch.randint(0, 0x3C00, (t.page_bytes // 2,), generator=g, device=DEV, dtype=torch.int16)
        payloads.append(words.cpu().numpy().tobytes())
    # half of the pages read back are among those just written
    return dict(run=_run_swap, t=t, write=list(zip(ids[:n], payloads)), read=ids[n // 2:n // 2 + n])


def _run_swap(s):
    s["t"].write_kv_pages(s["write"])
    return [np.frombuffer(p, np.uint8) for p in s["t"].read_kv_pages(s["read"])]


# ------------------------------------------------------------------ work, exact, tolerance

_SIZE = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}


def work(case):
    kind = case["kind"]
    if kind in ("step", "engine", "block"):
        new, cached = _ints(case["new"]), _ints(case["cached"])
        rows, ctx = int(new.sum()), new + cached
        hq, hkv, d, eb = case["hq"], case["hkv"], case["d"], _SIZE[case["kv"]]
        pages = int((-(-ctx // case["page"])).sum())
        qb = _SIZE[case.get("q", "f32")]
        ob = _SIZE[case.get("out", case.get("q", "f32"))]
        # cached keys and values, queries, outputs, block table (and scales), the step's rows read
        # and appended
        rb = 4 if kind == "block" else 2
        byte = (int(cached.sum()) * hkv * d * 2 * eb + rows * hq * d * (qb + ob) + pages * 4
                + rows * hkv * d * 2 * (rb + eb))
        if case["kv"] == "fp8":
            byte += pages * hkv * 8
        if kind == "block":  # the projection rows and the written query, the coefficients, the gathered rows
            byte += rows * hq * d * (4 + qb) + rows * d * 4 * 2 + len(new) * hq * d * 2 * qb
        keys = int((new * cached + new * (new + 1) // 2).sum())
        layers = case.get("layers", 1)
        return dict(bytes=byte * layers, flops=4 * hq * d * keys * layers)
    if kind == "rope":
        rows, hq, hkv, d = (case[k] for k in ("rows", "hq", "hkv", "d"))
        return dict(bytes=rows * ((hq + 2 * hkv) * d * 4 + hq * d * _SIZE[case["q"]] + 2 * hkv * d * _SIZE[case["kv"]]
                                  + d * 4), flops=rows * (hq + hkv) * d * 3)
    if kind == "quantize":
        values = 2 * case["pages"] * case["page"] * case["hkv"] * case["d"]
        return dict(bytes=values * (_SIZE[case["src"]] + 1) + 2 * case["pages"] * case["hkv"] * 4, flops=2 * values)
    if kind == "sample":
        return dict(bytes=case["rows"] * case["vocab"] * 4, flops=2 * case["rows"] * case["vocab"])
    page = 2 * case["layers"] * case["page"] * case["hkv"] * case["d"] * _SIZE[case["kv"]]
    return dict(bytes=4 * case["pages"] * page, flops=0)


def _attend(b, q, k, v, hq, hkv, d):
    """softmax(q k / sqrt(d)) v in 64 bits; k and v: [tokens][hkv][d] by pool slot."""
    out = torch.empty((b.rows, hq, d), dtype=torch.float64, device=DEV)
    group = hq // hkv
    for i in range(b.n):
        n, r0, r1 = int(b.ctx[i]), int(b.cu[i]), int(b.cu[i + 1])
        pos = np.arange(n)
        at = torch.from_numpy(b.tables[i].astype(np.int64)[pos // b.page] * b.page + pos % b.page).to(DEV)
        late = torch.arange(n, device=DEV)[None, :] > torch.arange(n - (r1 - r0), n, device=DEV)[:, None]
        for h in range(hkv):
            kh, vh = k[at, h], v[at, h]
            kt = kh.t().contiguous()
            for j in range(h * group, (h + 1) * group):
                s = q[r0:r1, j].double() @ kt / math.sqrt(d)
                out[r0:r1, j] = torch.softmax(s.masked_fill_(late, -math.inf), 1) @ vh
    return out


def _appended(plane, rows, slots, kv, scale, page, hkv, d):
    """A pool plane with the step's rows in place: its stored values in 64 bits."""
    rows = rows.reshape(-1, hkv, d)
    at = torch.from_numpy(slots).to(DEV)
    if kv != "fp8":
        plane = plane.clone()
        plane[at] = rows.to(plane.dtype)
        return plane.double()
    s = scale.reshape(-1, hkv)
    codes = (rows.float() / s[at // page][:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    x = plane.view(torch.float8_e4m3fn).to(torch.float32)
    x[at] = codes.to(torch.float32)
    return x.double() * s.repeat_interleave(page, 0)[:, :, None].double()


def _rotation(positions, d):
    """cos and sin of f32(position) * f32(1 / f32(base^(2i/d))), the table's defined angles."""
    i = torch.arange(d // 2, device=DEV, dtype=torch.float32)
    p = torch.pow(torch.tensor(5e6, dtype=torch.float64, device=DEV), (2.0 * i / d).double()).float()
    angle = (torch.from_numpy(np.asarray(positions)).to(DEV).float()[:, None] * (1.0 / p)[None, :]).double()
    return torch.stack([angle.cos(), angle.sin()], -1)


def _rotated(x, cs):
    """[rows][heads][d] in 64 bits, turned by the table."""
    half = x.shape[-1] // 2
    l, r = x[..., :half].double(), x[..., half:].double()
    c, s = cs[:, None, :, 0].float().double(), cs[:, None, :, 1].float().double()
    return torch.cat([l * c - r * s, r * c + l * s], -1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "engine"):
        b = _Batch(case, seed)
        got = []
        for t in _layers(case, b, seed):
            args = (b.slots, case["kv"]), (case["page"], case["hkv"], case["d"])
            k = _appended(t["k"], t["new_k"], *args[0], t.get("ks"), *args[1])
            v = _appended(t["v"], t["new_v"], *args[0], t.get("vs"), *args[1])
            got.append(dict(o=_attend(b, t["q"], k, v, case["hq"], case["hkv"], case["d"]), k=None, v=None))
        return dict(status=None, slots=None, layers=got) if kind == "step" else dict(layers=got)
    if kind == "block":
        b, g = _Batch(case, seed), _gen(seed)
        hq, hkv, d, P = case["hq"], case["hkv"], case["d"], case["page"]
        tokens = b.pool_pages * P
        k, v = _plane(g, tokens, hkv, d, case["kv"]), _plane(g, tokens, hkv, d, case["kv"])
        x = _combined(case, b.rows, seed).reshape(b.rows, hq + 2 * hkv, d)
        cs = _rotation(b.positions, d)
        turned = _rotated(x[:, :hq + hkv], cs)
        query = turned[:, :hq]
        k = _appended(k, turned[:, hq:], b.slots, case["kv"], None, P, hkv, d)
        v = _appended(v, x[:, hq + hkv:], b.slots, case["kv"], None, P, hkv, d)
        o = _attend(b, query, k, v, hq, hkv, d)
        return dict(coefficients=cs, query=query, o=o, picked=o[torch.from_numpy(b.cu[1:] - 1).to(DEV)],
                    k=None, v=None)
    if kind == "rope":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        x = _combined(case, case["rows"], seed).reshape(case["rows"], hq + 2 * hkv, d)
        cs = _rotation(case["first"] + np.arange(case["rows"]), d)
        return dict(coefficients=cs, query=_rotated(x[:, :hq], cs), k=None, v=None)
    if kind == "quantize":
        g = _gen(seed)
        n, P, hkv, d = case["pages"], case["page"], case["hkv"], case["d"]
        ids = np.random.default_rng(seed).permutation(n + 5)[:n]
        got = []
        for _ in "kv":
            x = _randn(g, n * P, hkv, d).to(TORCH[case["src"]]).double().reshape(n, P, hkv, d)
            s = torch.ones((n + 5, hkv), dtype=torch.float64, device=DEV)
            s[torch.from_numpy(ids).to(DEV)] = x.abs().amax(dim=(1, 3)) / 448.0
            got.append(s.reshape(-1))
        return dict(k=None, v=None, ks=got[0], vs=got[1])
    return None  # tokens and bytes


def tolerance(case):
    kind = case["kind"]
    if kind in ("sample", "swap"):
        return "exact"
    if kind == "quantize":  # f32 scales; measured 4.6e-9
        return {"rel": 1e-6}
    if kind == "rope":  # measured 1.7e-3 with a bf16 query, 2.8e-8 with f32
        return {"rel": 7e-3 if case["q"] == "bf16" else 1e-6}
    # attention: the weights and the output are rounded to 16 bits.  Measured against exact(): 1.7e-3
    # to 2.9e-3 with bf16 weights or outputs, 2.3e-4 to 2.7e-4 with f16 weights and an f32 output
    out = case.get("out", case.get("q", "f32"))
    return {"rel": 1e-3, "max": 0.02} if out == "f32" and case["kv"] != "bf16" else {"rel": 1e-2, "max": 0.1}
