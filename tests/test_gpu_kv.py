"""GPU parity of packing, slot mapping, KV append and FP8 page quantisation: bit-exact
against the CPU oracle (through the C ABI)."""
import numpy as np
import pytest
import torch

import gpu_data as G
from gpu_data import BF16, F16, F32, FP8

pytestmark = pytest.mark.gpu


def _append_case(O, lia, wl, kv, src, page, use_slots, rows_per_seq=(1, 3, 40), seed=0):
    rng = np.random.default_rng(seed)
    g = wl.Geometry(hq=16, hkv=2, d=128, page_size=page, kv_dtype=kv)
    ctx = [50, 300, 1000]
    b = wl.custom(ctx, list(rows_per_seq), geom=g, seed=seed)
    n = b.n_rows
    W = g.hkv * g.d
    kf = rng.standard_normal((n, W)).astype(np.float32)
    vf = rng.standard_normal((n, W)).astype(np.float32)
    if src == BF16:
        ks, vs = O.from_f32(kf, BF16), O.from_f32(vf, BF16)
        kd, vd = G.to_dev(ks, torch.bfloat16), G.to_dev(vs, torch.bfloat16)
    elif src == F16:
        ks, vs = O.from_f32(kf, F16), O.from_f32(vf, F16)
        kd, vd = G.to_dev(ks, torch.float16), G.to_dev(vs, torch.float16)
    else:
        ks, vs = kf, vf
        kd, vd = G.to_dev(kf), G.to_dev(vf)
    tokens = b.pool_pages * page
    store = np.uint8 if kv == FP8 else np.uint16
    fill = rng.integers(0, 255 if kv == FP8 else 65535, tokens * W).astype(store)
    kc, vc = fill.copy(), fill[::-1].copy()
    k_scales = v_scales = None
    if kv == FP8:
        k_scales = rng.uniform(0.005, 0.02, b.pool_pages * g.hkv).astype(np.float32)
        v_scales = rng.uniform(0.005, 0.02, b.pool_pages * g.hkv).astype(np.float32)
        # pages never quantised (scale 0) take scale 1, which the append records
        k_scales[rng.random(k_scales.size) < 0.3] = 0.0
        v_scales[rng.random(v_scales.size) < 0.3] = 0.0
    layout_o = O.KVLayout(g.hkv, g.d, page, b.pool_pages, kv)
    layout_p = lia.KVLayout(g.hkv, g.d, page, b.pool_pages, kv)
    pos, seq, flat, slots = b.positions(), b.sequences(), b.flat_table(), b.slot_mapping()
    dkc = G.to_dev(kc, torch.uint8 if kv == FP8 else torch.int16)
    dvc = G.to_dev(vc, torch.uint8 if kv == FP8 else torch.int16)
    dks = G.to_dev(k_scales) if k_scales is not None else None
    dvs = G.to_dev(v_scales) if v_scales is not None else None
    O.kv_append(layout_o, pos, seq, flat, b.stride, ks, vs, kc, vc, src_dtype=src,
                slot_mapping=slots if use_slots else None, k_scales=k_scales, v_scales=v_scales)
    if use_slots:
        lia.kv_append(layout_p, kd, vd, dkc, dvc, slot_mapping=G.u32_dev(slots),
                      k_scales=dks, v_scales=dvs)
    else:
        lia.kv_append(layout_p, kd, vd, dkc, dvc, positions=G.u32_dev(pos), sequences=G.u32_dev(seq),
                      pages=G.u32_dev(flat), stride=b.stride, k_scales=dks, v_scales=dvs)
    torch.cuda.synchronize()
    gk = dkc.cpu().numpy().view(store)
    gv = dvc.cpu().numpy().view(store)
    assert np.array_equal(gk, kc) and np.array_equal(gv, vc)
    if kv == FP8:
        assert np.array_equal(dks.cpu().numpy(), k_scales) and np.array_equal(dvs.cpu().numpy(), v_scales)


@pytest.mark.parametrize("kv", [F16, BF16, FP8])
@pytest.mark.parametrize("src", [F32, BF16, F16])
@pytest.mark.parametrize("page", [16, 32])
def test_kv_append_bit_exact(O, lia, wl, kv, src, page):
    print(f"[case] append kv={kv} src={src} page={page}", flush=True)
    _append_case(O, lia, wl, kv, src, page, use_slots=False)
    _append_case(O, lia, wl, kv, src, page, use_slots=True, seed=1)


def test_kv_append_reference_fixture(O, lia):
    """llama_cache_paged addressing on the reference's rotary fixture rows
    (src/gpu/kernels/llama_position.rs:132-152): f16 pool, 32-token pages, stride 4096."""
    positions = np.array([0, 31, 32, 8191, 131071], np.uint32)
    sequences = np.array([0, 1, 0, 1, 0], np.uint32)
    tables = np.zeros(2 * 4096, np.uint32)
    for row, page in enumerate([5, 3, 2, 7, 1]):
        tables[sequences[row] * 4096 + positions[row] // 32] = page
    j = np.arange(5 * 256)
    k = ((j * 43 % 997) / 256.0 - 2.0).astype(np.float32).reshape(5, 256)
    v = ((j * 17 % 509) / 128.0 - 2.0).astype(np.float32).reshape(5, 256)
    ek = np.zeros(8 * 32 * 256, np.uint16)
    ev = np.zeros_like(ek)
    O.kv_append(O.KVLayout(2, 128, 32, 8, F16), positions, sequences, tables, 4096, k, v, ek, ev)
    dk = torch.zeros(ek.size, dtype=torch.int16, device="cuda")
    dv = torch.zeros_like(dk)
    lia.kv_append(lia.KVLayout(2, 128, 32, 8, F16), G.to_dev(k), G.to_dev(v), dk, dv,
                  positions=G.u32_dev(positions), sequences=G.u32_dev(sequences),
                  pages=G.u32_dev(tables), stride=4096)
    torch.cuda.synchronize()
    assert np.array_equal(dk.cpu().numpy().view(np.uint16), ek)
    assert np.array_equal(dv.cpu().numpy().view(np.uint16), ev)


def test_pack_device_matches_host(lia, wl, O):
    for cfg in (wl.config1(seed=2), wl.config3(seed=2), wl.config4(seed=2)):
        print(f"[case] pack_device {cfg.name}", flush=True)
        n = cfg.n_seqs
        rows = cfg.n_rows
        P = cfg.geom.page_size
        context = int(cfg.stride * P)
        dev_out = {k: torch.full((rows + (k == "cu"),), -7, dtype=torch.int32, device="cuda")
                   for k in ("cu", "positions", "sequences", "slots")}
        status = torch.full((1,), -7, dtype=torch.int32, device="cuda")
        lia.pack_device(G.u32_dev(np.arange(n)), G.u32_dev(cfg.q_len), G.u32_dev(cfg.cached),
                        G.u32_dev(cfg.flat_table()), cfg.stride, P, cfg.pool_pages, context, rows,
                        dev_out["cu"], dev_out["positions"], dev_out["sequences"], dev_out["slots"],
                        status)
        torch.cuda.synchronize()
        assert status.item() == 0
        host_rows = [(0, int(p), int(s)) for p, s in zip(cfg.positions(), cfg.sequences())]
        lim = lia.PagingLimits(max(n, 1), context, P, cfg.pool_pages, 1, max(rows, 1))
        packed = lia.pack_rows(lim, host_rows, [t.tolist() for t in cfg.tables])
        got = {k: v.cpu().numpy().view(np.uint32) for k, v in dev_out.items()}
        assert np.array_equal(got["positions"], packed["positions"])
        assert np.array_equal(got["sequences"], packed["sequences"])
        assert np.array_equal(got["slots"], packed["slot_mapping"])
        assert np.array_equal(got["cu"][:n + 1], packed["cu_seqlens"])


def test_pack_device_reports_missing_page(lia):
    pages = G.u32_dev(np.array([3, 0xFFFFFFFF], np.uint32))
    out = [torch.zeros(4, dtype=torch.int32, device="cuda") for _ in range(4)]
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    lia.pack_device(G.u32_dev([0]), G.u32_dev([2]), G.u32_dev([15]), pages, 2, 16, 8, 32, 4,
                    out[0], out[1], out[2], out[3], status)
    torch.cuda.synchronize()
    assert status.item() == 10  # -LIA_E_MISSING_PAGE


@pytest.mark.parametrize("order,expect", [((0, 1), 10), ((1, 0), 8)])
def test_pack_device_reports_first_failing_row(lia, order, expect):
    """Two failing sequences: the status is the error of the earlier row in packed order
    (sequence A: its second row needs a missing page; sequence B: position 40 >= context)."""
    pages = G.u32_dev(np.array([3, 0xFFFFFFFF, 4, 5], np.uint32))  # stride 2: rows 0 and 1
    seqs = {0: (0, 2, 15), 1: (1, 1, 40)}  # (table row, q_len, cached)
    slot, q_len, cached = zip(*[seqs[i] for i in order])
    out = [torch.zeros(8, dtype=torch.int32, device="cuda") for _ in range(4)]
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    lia.pack_device(G.u32_dev(slot), G.u32_dev(q_len), G.u32_dev(cached), pages, 2, 16, 8, 32, 8,
                    out[0], out[1], out[2], out[3], status)
    torch.cuda.synchronize()
    assert status.item() == expect  # 10: -LIA_E_MISSING_PAGE, 8: -LIA_E_POSITION


def test_kv_quantize_pages_bit_exact(O, lia):
    rng = np.random.default_rng(12)
    H, D, P, pool = 2, 128, 16, 40
    n = 9
    k = rng.standard_normal((n, P, H, D)).astype(np.float32) * 3
    v = rng.standard_normal((n, P, H, D)).astype(np.float32)
    v[3] = 0
    ids = rng.permutation(pool)[:n].astype(np.uint32)
    kc = np.zeros(pool * P * H * D, np.uint8)
    vc = np.zeros_like(kc)
    ks = np.zeros(pool * H, np.float32)
    vs = np.zeros_like(ks)
    O.kv_quantize_pages(O.KVLayout(H, D, P, pool, FP8), ids, k, v, kc, vc, ks, vs)
    dkc = torch.zeros(kc.size, dtype=torch.uint8, device="cuda")
    dvc = torch.zeros_like(dkc)
    dks = torch.zeros(ks.size, dtype=torch.float32, device="cuda")
    dvs = torch.zeros_like(dks)
    lia.kv_quantize_pages(lia.KVLayout(H, D, P, pool, FP8), G.u32_dev(ids), G.to_dev(k), G.to_dev(v),
                          dkc, dvc, dks, dvs)
    torch.cuda.synchronize()
    assert np.array_equal(dks.cpu().numpy(), ks) and np.array_equal(dvs.cpu().numpy(), vs)
    assert np.array_equal(dkc.cpu().numpy(), kc) and np.array_equal(dvc.cpu().numpy(), vc)


def test_engine_step_append_then_attend(lia, wl, O):
    """Engine mirror: stage (host packing + upload), append this step's K/V, attend."""
    g = wl.Geometry(hq=16, hkv=2, d=128, page_size=32, kv_dtype=BF16, q_dtype=BF16,
                    out_dtype=F32)
    eng = lia.Engine(16, 2, 128, pool_tokens=4096, layers=2, page_size=32, kv_dtype=BF16,
                     q_dtype=BF16, out_dtype=F32, prefill_batch=256)
    eng.configure_paging(4, 2048)
    rng = np.random.default_rng(13)
    pool_k = O.from_f32(rng.standard_normal((4096, 2, 128)).astype(np.float32), BF16)
    pool_v = O.from_f32(rng.standard_normal((4096, 2, 128)).astype(np.float32), BF16)
    eng.k[1].copy_(G.to_dev(pool_k, torch.int16).view(4096, 2, 128))
    eng.v[1].copy_(G.to_dev(pool_v, torch.int16).view(4096, 2, 128))
    tables = [[int(x) for x in rng.permutation(128)[:k]] for k in (10, 3)]
    tables[1] = [p for p in range(128) if p not in tables[0]][:3]
    rows = [(5, p, 0) for p in range(290, 300)] + [(7, 70, 1)]
    packed = eng.stage(rows, tables, outputs=[9, 10])
    n = len(rows)
    q = O.from_f32(rng.standard_normal((n, 16, 128)).astype(np.float32), BF16)
    k = O.from_f32(rng.standard_normal((n, 256)).astype(np.float32), BF16)
    v = O.from_f32(rng.standard_normal((n, 256)).astype(np.float32), BF16)
    out = eng.attention(1, G.to_dev(q, torch.bfloat16), G.to_dev(k, torch.bfloat16),
                        G.to_dev(v, torch.bfloat16))
    torch.cuda.synchronize()
    kc, vc = pool_k.reshape(-1).copy(), pool_v.reshape(-1).copy()
    O.kv_append(O.KVLayout(2, 128, 32, 128, BF16), packed["positions"], packed["sequences"],
                packed["flat"], packed["stride"], k, v, kc, vc, src_dtype=BF16)
    assert np.array_equal(eng.k[1].cpu().numpy().view(np.uint16).reshape(-1), kc)
    geom = O.geom(16, 2, 128, 32, packed["stride"], BF16)
    ref = O.attention_f64(geom, packed["positions"], packed["sequences"], packed["flat"],
                          O.to_f32(q, BF16), kc, vc)
    err = np.abs(out.cpu().numpy() - ref)
    assert err.max() < 2e-2 and err.mean() < 2e-3


def _append_plain(O, lia, hkv, d, kv, src, k, v, scales, offset=0):
    """rows of k and v appended to slots 3, 4, .. of a 16-token-page pool, here and by the oracle;
    offset: elements by which the source arrays start past their (aligned) allocation."""
    rows, W, P = k.shape[0], hkv * d, 16
    pool = -(-(rows + 3) // P)
    store = np.uint8 if kv == FP8 else np.uint16
    kc, vc = np.zeros(pool * P * W, store), np.full(pool * P * W, 9, store)
    ks = vs = None
    if kv == FP8:
        ks, vs = np.resize(scales, pool * hkv).astype(np.float32), np.resize(scales[::-1], pool * hkv).astype(np.float32)
    slots = np.arange(3, 3 + rows).astype(np.uint32)
    tdt = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[src]

    def dev(a):
        t = G.to_dev(np.concatenate([np.zeros(offset, a.dtype), a.reshape(-1)]))
        return (t if src == F32 else t.view(tdt))[offset:].view(rows, W)

    dkc, dvc = (G.to_dev(x.view(np.int16) if kv != FP8 else x).clone() for x in (kc, vc))
    dks, dvs = (None, None) if ks is None else (G.to_dev(ks).clone(), G.to_dev(vs).clone())
    with np.errstate(all="ignore"):
        O.kv_append(O.KVLayout(hkv, d, P, pool, kv), slots, slots * 0, np.arange(pool), pool, k, v, kc, vc,
                    src_dtype=src, slot_mapping=slots, k_scales=ks, v_scales=vs)
    lia.kv_append(lia.KVLayout(hkv, d, P, pool, kv), dev(k), dev(v), dkc, dvc, slot_mapping=G.u32_dev(slots),
                  k_scales=dks, v_scales=dvs)
    torch.cuda.synchronize()
    assert np.array_equal(dkc.cpu().numpy().view(store), kc) and np.array_equal(dvc.cpu().numpy().view(store), vc)
    if ks is not None:
        assert np.array_equal(dks.cpu().numpy(), ks) and np.array_equal(dvs.cpu().numpy(), vs)


SCALES = [1.0, 0.0, 0.0078125, 3.3e-3, 448.0, 1e-30, 1e-27, 8e-28, 1e30, 1.2e27, 1e-40, -0.5, 1.0 / 448.0, 0.7]


@pytest.mark.parametrize("kv", [F16, BF16, FP8])
@pytest.mark.parametrize("src", [F16, BF16])
def test_kv_append_every_16_bit_value(O, lia, kv, src):
    """Every 16-bit pattern (NaNs, infinities, subnormals and both zeros among them) into every pool
    type, on FP8 pools under scales at and past the ends of the fast quotient's range."""
    k = np.resize(np.arange(65536, dtype=np.uint32), 65536).astype(np.uint16).reshape(512, 128)
    for shift in range(0, len(SCALES) if kv == FP8 else 1, 4):
        _append_plain(O, lia, 2, 64, kv, src, k, k[::-1].copy(), SCALES[shift:] + SCALES[:shift])


@pytest.mark.parametrize("hkv,d,offset", [(1, 8, 0), (3, 24, 0), (2, 12, 0), (5, 4, 0), (2, 64, 1), (1, 128, 8)])
@pytest.mark.parametrize("kv,src", [(FP8, F32), (FP8, BF16), (BF16, F32), (F16, F16)])
def test_kv_append_edges(O, lia, hkv, d, offset, kv, src):
    """Row widths and alignments on both sides of the vector kernel's conditions, f32 values one ulp
    about the rounding boundaries of e4m3 quotients."""
    rng = np.random.default_rng(hkv * 100 + d)
    rows = 37
    scales = rng.uniform(1e-3, 2.0, 16).astype(np.float32)
    x = rng.standard_normal((2, rows, hkv * d)).astype(np.float32) * 100
    if kv == FP8 and src == F32:
        code = rng.integers(0, 1 << 12, x.shape)  # values (1 + m/16) 2^e: e4m3 values and their midpoints
        x = (((16 + code % 16) / 16.0) * 2.0 ** (code // 16 % 16 - 9) * rng.choice(scales, x.shape)).astype(np.float32)
        x = np.nextafter(x, np.float32(np.inf) * rng.choice([-1, 1], x.shape).astype(np.float32))
    if src != F32:
        x = O.from_f32(x, src)
    _append_plain(O, lia, hkv, d, kv, src, x[0], x[1], scales, offset)


@pytest.mark.parametrize("src", [F32, F16, BF16])
@pytest.mark.parametrize("hkv,d,page,offset", [(2, 128, 16, 0), (3, 64, 16, 0), (1, 128, 64, 0), (2, 64, 128, 0),
                                               (2, 128, 128, 0), (2, 24, 16, 0), (2, 8, 1, 0), (2, 64, 32, 1)])
def test_kv_quantize_pages_geometries(O, lia, src, hkv, d, page, offset):
    """Pages on both sides of the register-resident kernel's conditions (piece counts 1 to 1,024 and
    past them, rows that are no power of two, a source off its alignment), with zero pages, an
    infinity, NaNs, subnormal and very large pages: codes and scales bit for bit."""
    rng = np.random.default_rng(page + d)
    n, pool = 11, 17
    x = rng.standard_normal((2, n, page, hkv, d)).astype(np.float32)
    x[:, 1] = 0
    x[0, 2] = -0.0
    x[:, 3] *= 1e-38
    x[:, 4] *= 3e37 if src != F16 else 1e4
    x[0, 5, -1, 0, -1] = np.inf
    x[1, 6, 0, 0, ::3] = np.nan
    x[0, 7] *= 6e-8
    with np.errstate(all="ignore"):
        x = x if src == F32 else O.from_f32(x, src).reshape(x.shape)
    ids = rng.permutation(pool)[:n].astype(np.uint32)
    W = pool * page * hkv * d
    kc, vc, ks, vs = np.zeros(W, np.uint8), np.zeros(W, np.uint8), np.zeros(pool * hkv, np.float32), np.zeros(pool * hkv, np.float32)
    O.kv_quantize_pages(O.KVLayout(hkv, d, page, pool, FP8), ids, x[0], x[1], kc, vc, ks, vs, src_dtype=src)
    tdt = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[src]

    def dev(a):
        t = G.to_dev(np.concatenate([np.zeros(offset, a.dtype), a.reshape(-1)]))
        return (t if src == F32 else t.view(tdt))[offset:]

    got = [torch.zeros(W, dtype=torch.uint8, device="cuda") for _ in "kv"]
    sc = [torch.zeros(pool * hkv, device="cuda") for _ in "kv"]
    lia.kv_quantize_pages(lia.KVLayout(hkv, d, page, pool, FP8), G.u32_dev(ids), dev(x[0]), dev(x[1]), *got, *sc)
    torch.cuda.synchronize()
    for a, b in ((sc[0], ks), (sc[1], vs)):
        assert np.array_equal(a.cpu().numpy().view(np.uint32), b.view(np.uint32))
    assert np.array_equal(got[0].cpu().numpy(), kc) and np.array_equal(got[1].cpu().numpy(), vc)


@pytest.mark.parametrize("kv", [F16, BF16, FP8])
@pytest.mark.parametrize("src,offset", [(F16, 0), (BF16, 0), (BF16, 1), (F32, 0)])
def test_engine_attention_appends_and_attends(lia, O, kv, src, offset):
    """Engine.attention over rows of every type and alignment (appended by the attention launch where
    the pool's type and 16-byte alignment allow, else before it), two layers on one staged plan, then
    a second stage of another shape: pools bit for bit and outputs against the float64 oracle."""
    eng = lia.Engine(16, 2, 128, pool_tokens=2048, layers=2, page_size=32, kv_dtype=kv, q_dtype=F32,
                     out_dtype=F32, prefill_batch=256)
    eng.configure_paging(4, 1024)
    rng = np.random.default_rng(17)
    tables = [[int(x) for x in t] for t in np.split(rng.permutation(64), [16, 40])]
    pools = []
    for layer in range(2):
        kv_np = [O.from_f32(rng.standard_normal((2048, 2, 128)).astype(np.float32), kv) if kv != FP8
                 else rng.integers(0, 120, (2048, 2, 128)).astype(np.uint8) for _ in "kv"]
        for dst, a in zip((eng.k[layer], eng.v[layer]), kv_np):
            (dst if kv == FP8 else dst.view(torch.int16)).copy_(G.to_dev(a.view(np.int16) if kv != FP8 else a).view(2048, 2, 128))
        if kv == FP8:
            eng.k_scales[layer].fill_(0.01)
            eng.v_scales[layer].fill_(0.02)
        pools.append([a.reshape(-1).copy() for a in kv_np])
    tdt = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[src]
    scales = [np.full(64 * 2, x, np.float32) if kv == FP8 else None for x in (0.01, 0.02)]
    for rows in ([(1, p, 0) for p in range(100, 103)] + [(1, 500, 1)],
                 [(1, p, 2) for p in range(0, 70)] + [(1, 501, 1)]):
        packed = eng.stage(rows, tables, outputs=[0])
        n = len(rows)
        for layer in range(2):
            q = rng.standard_normal((n, 16, 128)).astype(np.float32)
            new = [rng.standard_normal((n, 256)).astype(np.float32) for _ in "kv"]
            new = new if src == F32 else [O.from_f32(x, src) for x in new]

            def dev(a):
                t = G.to_dev(np.concatenate([np.zeros(offset, a.dtype), a.reshape(-1)]))
                return (t if src == F32 else t.view(tdt))[offset:].view(n, 2, 128)

            out = eng.attention(layer, G.to_dev(q), dev(new[0]), dev(new[1]))
            torch.cuda.synchronize()
            kc, vc = pools[layer]
            O.kv_append(O.KVLayout(2, 128, 32, 64, kv), packed["positions"], packed["sequences"],
                        packed["flat"], packed["stride"], new[0], new[1], kc, vc, src_dtype=src,
                        k_scales=scales[0], v_scales=scales[1])
            got = [x if kv == FP8 else x.view(torch.int16) for x in (eng.k[layer], eng.v[layer])]
            store = np.uint8 if kv == FP8 else np.uint16
            assert np.array_equal(got[0].cpu().numpy().view(store).reshape(-1), kc)
            assert np.array_equal(got[1].cpu().numpy().view(store).reshape(-1), vc)
            ref = O.attention_f64(O.geom(16, 2, 128, 32, packed["stride"], kv), packed["positions"],
                                  packed["sequences"], packed["flat"], q, kc, vc, *scales)
            err = np.abs(out.cpu().numpy() - ref)
            assert err.max() < (5e-2 if kv == FP8 else 2e-2) and err.mean() < (5e-3 if kv == FP8 else 2e-3)


@pytest.mark.parametrize("kv", [F16, BF16])
@pytest.mark.parametrize("case", ["interleaved", "shared", "interleaved prefill", "shared prefill"])
def test_engine_attends_rows_the_step_appends(lia, O, kv, case):
    """Steps in which a cached key of one group is a row that the same step appends, with rows of the
    pool's type: one sequence in two groups, and a page that one sequence writes and another attends, as
    decode and as prefill batches.  The rows' slots hold garbage before; outputs against the float64
    oracle over the pool after the append."""
    eng = lia.Engine(16, 2, 128, pool_tokens=2048, layers=1, page_size=32, kv_dtype=kv, prefill_batch=256)
    eng.configure_paging(4, 1024)
    rng = np.random.default_rng(23)
    free = [int(p) for p in rng.permutation(64)]
    tables = [free[:8], free[8:28]]
    span = lambda s, a, b: [(1, p, s) for p in range(a, b)]  # noqa: E731
    if case == "interleaved":
        rows = span(0, 100, 101) + span(1, 500, 501) + span(0, 101, 102)
    elif case == "interleaved prefill":
        rows = span(0, 100, 140) + span(1, 500, 535) + span(0, 140, 200)
    else:  # sequence 1 attends page 3 of sequence 0 in its own place 1
        tables[1][1] = tables[0][3]
        rows = (span(0, 127, 128) + span(1, 500, 501) if case == "shared"
                else span(0, 90, 150) + span(1, 500, 540))
    packed = eng.stage(rows, tables, outputs=[0])
    n = len(rows)
    pool = [O.from_f32(rng.standard_normal((2048, 2, 128)).astype(np.float32), kv) for _ in "kv"]
    for a in pool:
        a[packed["slot_mapping"]] = O.from_f32(np.full((n, 2, 128), 50.0, np.float32), kv)
    for dst, a in zip((eng.k[0], eng.v[0]), pool):
        dst.view(torch.int16).copy_(G.to_dev(a.view(np.int16)))
    tdt = torch.float16 if kv == F16 else torch.bfloat16
    q = rng.standard_normal((n, 16, 128)).astype(np.float32)
    new = [O.from_f32(rng.standard_normal((n, 2, 128)).astype(np.float32), kv) for _ in "kv"]
    out = eng.attention(0, G.to_dev(q), *[G.to_dev(a, tdt) for a in new])
    torch.cuda.synchronize()
    for a, x in zip(pool, new):
        a[packed["slot_mapping"]] = x
    assert np.array_equal(eng.k[0].cpu().numpy().view(np.uint16), pool[0])
    assert np.array_equal(eng.v[0].cpu().numpy().view(np.uint16), pool[1])
    ref = O.attention_f64(O.geom(16, 2, 128, 32, packed["stride"], kv), packed["positions"], packed["sequences"],
                          packed["flat"], q, pool[0].reshape(-1), pool[1].reshape(-1))
    err = np.abs(out.cpu().numpy() - ref)
    assert err.max() < 2e-2 and err.mean() < 2e-3


def test_engine_layers_around_other_calls(lia):
    """A layer's output does not change when, after stage(), another batch runs on paging["workspace"]."""
    eng = lia.Engine(16, 2, 128, pool_tokens=4096, layers=1, page_size=32, prefill_batch=64)
    eng.configure_paging(4, 2048)
    g = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    for x in (eng.k[0], eng.v[0]):
        x.view(torch.float16).copy_(rand(4096, 2, 128))
    tables = [list(range(60)), list(range(60, 124))]
    rows = [(1, 1500, 0), (1, 2000, 1)]
    q, k, v = rand(2, 16, 128), rand(2, 2, 128).half(), rand(2, 2, 128).half()
    eng.stage(rows, tables, [0, 1])
    want = eng.attention(0, q, k, v).clone()
    w = eng.paging
    lia.paged_attention(eng.config, 1, w["cu_seqlens"], w["positions"], w["sequences"], w["pages"], q[:1],
                        eng.k[0], eng.v[0], torch.empty((1, 16, 128), device="cuda"), w["workspace"])
    assert torch.equal(eng.attention(0, q, k, v), want)


def test_engine_layer_replayed_for_later_steps(lia):
    """A captured layer, replayed after other steps of its shape were staged (private pages, a page that
    the step writes and attends, private pages of other contexts), equals the eager layer of each step,
    whose later layers the replay leaves alone."""
    eng = lia.Engine(16, 2, 128, pool_tokens=4096, layers=1, page_size=32, prefill_batch=64)
    eng.configure_paging(4, 2048)
    g = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    pool = [rand(4096, 2, 128).half() for _ in "kv"]
    q, k, v = rand(2, 16, 128), rand(2, 2, 128).half(), rand(2, 2, 128).half()
    out = torch.empty((2, 16, 128), device="cuda")

    def refill():
        for dst, src in zip((eng.k[0], eng.v[0]), pool):
            dst.view(torch.float16).copy_(src)

    private, shared = [list(range(60)), list(range(60, 124))], [list(range(60)), [*range(60, 70), 46, *range(70, 120)]]
    eng.stage([(1, 1500, 0), (1, 1900, 1)], private, [0, 1])
    eng.attention(0, q, k, v, out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        eng.attention(0, q, k, v, out)
    for tables, at in ((private, (1500, 1900)), (shared, (1500, 1900)), (private, (70, 333)), (shared, (1501, 700))):
        eng.stage([(1, at[0], 0), (1, at[1], 1)], tables, [0, 1])
        refill()
        want = eng.attention(0, q, k, v).clone()
        pools = eng.k[0].clone(), eng.v[0].clone()
        refill()
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        # the eager layer may read the new rows apart from the cached ones: f16 weights of other chunks,
        # each rounded by at most 2^-11
        assert (out - want).abs().max() <= 2e-3 * want.abs().max()
        assert torch.equal(eng.k[0], pools[0]) and torch.equal(eng.v[0], pools[1])
        refill()
        assert torch.equal(eng.attention(0, q, k, v), want)


def _pack_both(lia, q_len, cached, tables, P, pool):
    """The device's packing (both entry points' checks) and the host's, of one batch: their metadata,
    or their failure codes."""
    n, rows = len(q_len), int(sum(q_len))
    stride = max(len(t) for t in tables)
    context = stride * P
    flat = np.full(n * stride, 0xFFFFFFFF, np.uint32)
    for i, t in enumerate(tables):
        flat[i * stride:i * stride + len(t)] = t
    out = [torch.full((max(m, 1),), -7, dtype=torch.int32, device="cuda") for m in (n + 1, rows, rows, rows, 1)]
    lia.pack_device(G.u32_dev(np.arange(n)), G.u32_dev(q_len), G.u32_dev(cached), G.u32_dev(flat), stride, P, pool,
                    context, max(rows, 1), *out)
    torch.cuda.synchronize()
    status = int(out[4].item())
    if rows == 0:
        return status, None
    host_rows = [(0, int(c) + i, s) for s, (q, c) in enumerate(zip(q_len, cached)) for i in range(int(q))]
    try:
        packed = lia.pack_rows(lia.PagingLimits(n, context, P, pool, 1, rows), host_rows, [list(map(int, t)) for t in tables])
    except lia.LiaError as e:
        return status, -e.status
    got = [o.cpu().numpy().view(np.uint32) for o in out[:4]]
    assert status == 0
    assert np.array_equal(got[1], packed["positions"]) and np.array_equal(got[2], packed["sequences"])
    assert np.array_equal(got[3], packed["slot_mapping"])
    return 0, 0


@pytest.mark.parametrize("P,q_len", [(16, [5000, 3]), (16, [1] * 700), (16, [0, 1023, 0, 1, 1]), (64, [4097]),
                                     (16, [4090, 1, 1, 1, 1, 1, 1]), (1, [3000, 17]), (2, [5000]), (16, [0, 0])])
def test_pack_device_row_counts(lia, P, q_len):
    """Batches about the packing's limits (1,024 rows a pass, 4,096 a batch, the table of the runs'
    pages, pages of one and two tokens, no rows at all) equal the host's."""
    rng = np.random.default_rng(sum(q_len) + P)
    cached = rng.integers(0, 50, len(q_len))
    need = [-(-(int(q) + int(c)) // P) for q, c in zip(q_len, cached)]
    pool = max(sum(need), 1) + 3
    perm = rng.permutation(pool)
    tables = [x for x in np.split(perm[:sum(need)], np.cumsum(need)[:-1])]
    tables = [t if len(t) else perm[:1] for t in tables]
    status, want = _pack_both(lia, q_len, cached, tables, P, pool)
    assert status == (want or 0)


@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("other,want", [(6, 0), (5, 11), (3, 11)])
def test_pack_device_rows_sharing_a_page(lia, big, other, want):
    """Two sequences whose new rows lie in one physical page: accepted while their slots differ (rows
    3 to 5 of one and 6 on of the other), rejected at the first slot written twice; alone and behind
    4,500 rows."""
    P, pool = 16, 400
    q_len, cached, tables = [3, 2], [3, other], [[7], [7]]
    if big:
        q_len, cached, tables = [4500] + q_len, [0] + cached, [list(range(100, 100 + -(-4500 // P)))] + tables
    status, host = _pack_both(lia, q_len, cached, tables, P, pool)
    assert status == host == want


def test_pack_device_with_the_page_table_at_its_fullest(lia):
    """1,023 sequences of two rows that straddle a page each, and one of 14,353 rows: 2,944 runs, nearly
    all that the packing's rule lets into its table of 4,096 pages.  As the host packs them, and with a
    slot written twice."""
    P, q_len = 16, [2] * 1023 + [14353]
    cached = [15] * 1023 + [0]
    need = [2] * 1023 + [-(-14353 // P)]
    perm = np.random.default_rng(31).permutation(sum(need) + 3)
    tables = np.split(perm[:sum(need)], np.cumsum(need)[:-1])
    status, want = _pack_both(lia, q_len, cached, tables, P, len(perm))
    assert status == (want or 0) == 0
    tables[700][1] = tables[20][1]
    status, want = _pack_both(lia, q_len, cached, tables, P, len(perm))
    assert status == want == 11
