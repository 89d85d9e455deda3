"""The work that a user of dsv41_amd has it do, as cases that can be timed and compared: decode steps of an attention
layer (cache appends, lightning indexer, sparse attention), the attention layer's FP8 projections, the prefill
indexer and attention, a whole attention layer over a prompt, and the index-key snapshot converter.

Sizes are the benchmark's configurations (absorbed-MLA rows of 576 with 512 value columns, 64 index heads, ratio 4,
top-k 2048) and the reference geometry of the tests (rows of 512 with the rope inside, 32 index heads, top-k 512).
Decode steps run as serving runs them: a few layers' launches captured once in a HIP graph and replayed per token
(DecodeLayer is made to be captured); everything else is called eagerly."""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("deepseekv4.1-a100-custom_amd"))

DEV = "cuda:0"
H, DV, DI, WIN, RD, EPS = 64, 512, 128, 128, 64, 1e-6
DIM, QRANK, GROUPS, ORANK = 5120, 1280, 8, 1024  # the layer's widths at the projections' shapes
BF = torch.bfloat16

MLA = dict(d=576, hi=64, ratio=4, topk=2048)   # the benchmark's geometry
REF = dict(d=512, hi=32, ratio=2, topk=512)    # the reference geometry (rope inside the row)


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    ragged32 = ",".join(str(int(65536 * 2 ** (-i * 6 / 31))) for i in range(32))
    return [
        # one user, short context, eight layers of the token's graph: launches and latency
        dict(name="decode_1x8k", kind="decode", ctx="8191", rows=1, layers=8, **REF),
        # the headline decode configuration: four users at 128K
        dict(name="decode_4x128k", kind="decode", ctx="131072,131072,131072,131072", rows=1, layers=4, **MLA),
        # one user at a million tokens
        dict(name="decode_1x1m", kind="decode", ctx="1048576", rows=1, layers=2, **MLA),
        # speculative verify: eight users of very different contexts, 1 + 5 draft rows each
        dict(name="decode_drafts_8x6", kind="decode", ctx="524288,131072,131072,131072,65536,32768,8192,2048", rows=6,
             layers=1, **MLA),
        # a serving batch: 32 users with contexts between 1K and 64K
        dict(name="decode_32_ragged", kind="decode", ctx=ragged32, rows=1, layers=2, **REF),
        # the reference's own decode call sites, one by one and eager, on its bf16 index-key table
        dict(name="dropin_4x32k", kind="dropin", ctx="32767,32768,20001,9000", **REF),
        # one token through the layer's FP8 projections (replayed from the token's graph)
        dict(name="proj_1", kind="proj", m=1),
        # a prefill chunk through the same projections
        dict(name="proj_2048", kind="proj", m=2048),
        # the prefill indexer of a 2K chunk after 64K tokens
        dict(name="index_2k_64k", kind="index", s=2048, prior=65536, keys="e4m3", blocks=0, **MLA),
        # the prefill attention of the same chunk
        dict(name="attn_2k_64k", kind="attn", s=2048, prior=65536, **MLA),
        # a whole attention layer over a fresh prompt, FP8 weights
        dict(name="layer_3000", kind="layer", b=1, s=3000, hi=32, ratio=4, topk=512),
        # restoring a prefix snapshot: the bf16 index-key table to e4m3 + scales, and back
        dict(name="snapshot_256k", kind="snapshot", rows=262144),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "dropin", "proj", "proj", "index", "attn", "layer", "snapshot"])
    geo = dict(rng.choice([MLA, REF]))
    if kind == "decode":
        rows = rng.choice([1, 1, 1, 2, 4, 6])
        slots = _log(rng, 1, 32 if rows == 1 else 8)
        top = _log(rng, 600, min(1048576, 2097152 // slots))
        ctx = [top] + [_log(rng, 600, top) if top > 600 else top for _ in range(slots - 1)]
        return dict(kind=kind, ctx=",".join(map(str, ctx)), rows=rows, layers=rng.choice([1, 2]), **geo)
    if kind == "dropin":
        slots = _log(rng, 1, 8)
        return dict(kind=kind, ctx=",".join(str(_log(rng, 600, 65536)) for _ in range(slots)), **geo)
    if kind == "proj":
        return dict(kind=kind, m=_log(rng, 1, 2048))
    if kind in ("index", "attn"):
        s = _log(rng, 17, 2048)
        prior = rng.choice([0, _log(rng, 100, 65536)])
        c = dict(kind=kind, s=max(s, 4 * geo["ratio"]), prior=prior, **geo)
        if geo["ratio"] == 2 and prior > 32768:
            c["prior"] = prior // 2
        if kind == "index":  # a context that has more compressed rows than are selected
            c["prior"] = _log(rng, geo["topk"] * geo["ratio"] * 1.25, 65536 if geo["ratio"] == 4 else 32768)
            c.update(keys=rng.choice(["e4m3", "e4m3", "bf16"]), blocks=rng.choice([0, 0, 16]))
        return c
    if kind == "layer":
        return dict(kind=kind, b=rng.choice([1, 1, 2]), s=_log(rng, 64, 1500), hi=32, ratio=rng.choice([2, 4]), topk=512)
    return dict(kind=kind, rows=_log(rng, 1000, 262144))


# ------------------------------------------------------------------------------------------------ number formats
def _ceil_log2(a):
    m, e = torch.frexp(a)
    return e - (m == 0.5).to(e.dtype)


def _pow2(e):
    return torch.ldexp(torch.ones_like(e, dtype=torch.float32), e)


def _e4m3(v):
    return v.clamp(-448, 448).to(torch.float8_e4m3fn)


def _e2m1(v):
    a = v.abs()
    r = torch.where(a < 2, torch.round(a * 2) / 2, torch.where(a < 4, torch.round(a), torch.round(a / 2) * 2))
    return torch.copysign(r.clamp(max=6), v)


def _fq8(x, block=32):
    """e4m3 values with a power-of-two scale per block (bf16 in, bf16 out)."""
    g = x.float().reshape(-1, block)
    s = _pow2(_ceil_log2(g.abs().amax(-1, keepdim=True).clamp_min(1e-4) / 448))
    return (_e4m3(g / s).float() * s).reshape(x.shape).to(BF)


def _fq4(x, block=32, e4m3_scale=False):
    """E2M1 values with a power-of-two (or e4m3) scale per block (bf16 in, bf16 out)."""
    g = x.float().reshape(-1, block)
    amax = g.abs().amax(-1, keepdim=True)
    if e4m3_scale:
        s = _e4m3(amax.clamp_min(6 * 2.0 ** -9) / 6).float()
    else:
        s = _pow2(_ceil_log2(amax.clamp_min(6 * 2.0 ** -126) / 6))
    return (_e2m1((g / s).clamp(-6, 6)) * s).reshape(x.shape).to(BF)


def _encode_keys(k):
    """bf16 rows -> (e4m3 rows, fp32 power-of-two scale per row)."""
    kf = k.float()
    s = _pow2(_ceil_log2(kf.abs().amax(-1, keepdim=True).clamp_min(1e-30) / 448).clamp_min(-126))
    return _e4m3(kf / s), s[..., 0]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape, scale=1.0, dt=BF):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dt)


def _rope_tables(n):
    ang = torch.outer(torch.arange(n, dtype=torch.float64, device=DEV),
                      1.0 / (10000.0 ** (torch.arange(0, RD, 2, dtype=torch.float64, device=DEV) / RD)))
    return torch.cos(ang).float(), torch.sin(ang).float()


def _index_keys(g, *shape):
    """Index keys as the caches hold them: the FP4 grid, a few outlier channels."""
    k = torch.randn(*shape, DI, generator=g, device=DEV) * 0.1
    k[..., [3, 40, 77, 120]] *= 8
    return _fq4(k)


def _w8(g, n, k):
    """An FP8 block-scaled weight: e4m3 bytes [n, k] (natural order) and E8M0 scales [ceil(n / 32), k / 32]."""
    w = torch.randn(n, k, generator=g, device=DEV) * k ** -0.5
    e = _ceil_log2(w.view(n // 32, 32, k // 32, 32).abs().amax((1, 3)) / 448)
    s = _pow2(e).repeat_interleave(32, 0).repeat_interleave(32, 1)
    return _e4m3(w / s).view(torch.uint8), (e + 127).to(torch.uint8)


def _w8_64(pair):
    w, s = pair
    sc = torch.ldexp(torch.ones(s.shape, dtype=torch.float64, device=DEV), s.to(torch.int32) - 127)
    return w.view(torch.float8_e4m3fn).double() * sc.repeat_interleave(32, 0).repeat_interleave(32, 1)


def _contexts(case):
    return [int(c) for c in case["ctx"].split(",")]


# ------------------------------------------------------------------------------------------------ inputs
def _decode_inputs(case, seed, bf16_keys=False):
    g = _gen(seed)
    ctx, rows, d, hi, ratio = _contexts(case), case.get("rows", 1), case["d"], case["hi"], case["ratio"]
    S, R = len(ctx), len(ctx) * rows
    cap = max(max(ctx) // ratio, case["topk"]) + 1  # and the spare row
    layers = []
    for _ in range(case.get("layers", 1)):
        kbf = _index_keys(g, S, cap)
        k8, ks = (None, None) if bf16_keys else _encode_keys(kbf)
        layers.append(dict(ring=_randn(g, S, WIN, d), ckv=_fq4(_randn(g, S, cap, d), 16, True),
                           kbf=kbf if bf16_keys else None, k8=k8, ks=ks))
    step = dict(q=_randn(g, R, 1, H, d), q_idx=_fq4(_randn(g, R, 1, hi, DI)),
                w_idx=_randn(g, R, hi, scale=DI ** -0.5 * hi ** -0.5), kv_raw=_randn(g, R, d),
                latent=_randn(g, R, 1, d), k_raw=_randn(g, R, DI),
                kv_norm=(torch.rand(d, generator=g, device=DEV) + 0.5).to(BF),
                k_norm=(torch.rand(DI, generator=g, device=DEV) + 0.5).to(BF),
                sink=_randn(g, H, dt=torch.float32))
    pos = [c - rows + j for c in ctx for j in range(rows)]
    step["pos"] = torch.tensor(pos, device=DEV)
    step["seq"] = torch.tensor([s for s in range(S) for _ in range(rows)], device=DEV)
    step["pmax"] = torch.tensor([c - 1 for c in ctx for _ in range(rows)], device=DEV)
    step["cos"], step["sin"] = _rope_tables(max(ctx) + 1)
    return layers, step


def _chunk_inputs(case, seed):
    g = _gen(seed)
    s, prior, d, hi, ratio = case["s"], case["prior"], case["d"], case["hi"], case["ratio"]
    T = (prior + s) // ratio
    if case["kind"] == "index":
        kbf = _index_keys(g, 1, T)
        k8, ks = _encode_keys(kbf)
        return dict(q=_fq4(_randn(g, 1, s, hi, DI)), w=_randn(g, 1, s, hi, scale=DI ** -0.5 * hi ** -0.5), kbf=kbf,
                    k8=k8, ks=ks)
    hist = min(prior, WIN - 1)
    kk = min(case["topk"], T)
    n_win = hist + s
    qq = hist + torch.arange(s, device=DEV).unsqueeze(1)
    width = min(WIN, n_win)
    widx = (qq - WIN + 1).clamp_min(0) + torch.arange(width, device=DEV)
    widx = torch.where(widx <= qq, widx, -1)
    # the selection: kk of the row's causal compressed rows at random, ascending, -1 past them
    cl = (prior + torch.arange(s, device=DEV) + 1) // ratio
    sc = torch.rand(s, T, generator=g, device=DEV)
    sc.masked_fill_(torch.arange(T, device=DEV) >= cl.unsqueeze(1), -1.0)
    val, sel = sc.topk(kk, -1)
    sel = torch.where(val < 0, T, sel).sort(-1).values
    sel = torch.where(sel < T, sel + n_win, -1)
    idx = torch.cat([widx, sel], -1).to(torch.int32).unsqueeze(0)
    return dict(q=_randn(g, 1, s, H, d), win=_fq8(_randn(g, 1, n_win, d)), ckv=_fq4(_randn(g, 1, T, d), 16, True),
                sink=_randn(g, H, dt=torch.float32), idx=idx)


PROJ = (("wq_a", QRANK, DIM), ("wq_b", H * DV, QRANK), ("wkv", DV, DIM), ("wo_a", GROUPS * ORANK, H * DV // GROUPS),
        ("wo_b", DIM, GROUPS * ORANK))


def _proj_inputs(case, seed):
    g = _gen(seed)
    m = case["m"]
    w = {name: _w8(g, n, k) for name, n, k in PROJ}
    x = dict(x=_randn(g, m, DIM), qr=_randn(g, m, QRANK), o=_randn(g, m, H * DV), oa=_randn(g, m, GROUPS * ORANK),
             norm=(torch.rand(QRANK, generator=g, device=DEV) + 0.5).to(BF))
    return w, x


def _layer_inputs(case, seed):
    g = _gen(seed)
    hi = case["hi"]
    w8 = {name: _w8(g, n, k) for name, n, k in PROJ + (("i_wq_b", hi * DI, QRANK),)}
    w = dict(q_norm_w=(torch.rand(QRANK, generator=g, device=DEV) + 0.5).to(BF),
             kv_norm_w=(torch.rand(DV, generator=g, device=DEV) + 0.5).to(BF),
             c_norm_w=(torch.rand(DV, generator=g, device=DEV) + 0.5).to(BF),
             i_k_norm_w=(torch.rand(DI, generator=g, device=DEV) + 0.5).to(BF),
             attn_sink=_randn(g, H, dt=torch.float32), c_wkv=_randn(g, DV, DIM, scale=DIM ** -0.5, dt=torch.float32),
             c_wgate=_randn(g, DV, DIM, scale=DIM ** -0.5, dt=torch.float32),
             i_weights_proj=_randn(g, hi, DIM, scale=DIM ** -0.5), i_wk=_randn(g, DI, DV, scale=DV ** -0.5))
    return w8, w, _randn(g, case["b"], case["s"], DIM)


# ------------------------------------------------------------------------------------------------ prepare and run
def _capture(step):
    """A HIP graph of step(), captured the way a serving loop does: warmed on the capture stream, then recorded."""
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    side.wait_stream(main)
    with torch.cuda.stream(side):
        step()
    main.wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = step()
    return graph, out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        from dsv41_amd.decode import DecodeLayer
        tabs, st = _decode_inputs(case, seed)
        layers = [DecodeLayer(t["ring"], t["ckv"], t["k8"], t["ks"], st["sink"], st["cos"], st["sin"], case["ratio"],
                              case["topk"], rd=RD, dv=DV, eps=EPS) for t in tabs]
        cl = torch.div(st["pos"] + 1, case["ratio"], rounding_mode="floor")

        def step():
            out = []
            for lay in layers:
                new = (st["kv_raw"], st["kv_norm"], st["latent"], st["k_raw"], st["k_norm"], st["pos"], st["seq"],
                       st["q_idx"], st["w_idx"])
                if case["rows"] == 1:
                    idx = lay.appends_select(*new, cl)
                else:
                    lay.appends(*new)
                    idx = lay.select(st["q_idx"], st["w_idx"], st["pos"], st["seq"], cl)
                out.append((lay.attend(st["q"], idx, st["pos"], st["seq"], st["pmax"], plim=st["pos"]), idx))
            return out

        graph, out = _capture(step)
        return dict(kind=kind, graph=graph, out=out, tabs=tabs, st=st, layers=layers, step=step)
    if kind == "dropin":
        tabs, st = _decode_inputs(case, seed, bf16_keys=True)
        st["cl"] = (st["pos"] + 1) // case["ratio"]
        closes = (st["pos"] + 1) % case["ratio"] == 0
        st["row"] = torch.where(closes, st["cl"] - 1, tabs[0]["ckv"].shape[1] - 1)
        return dict(kind=kind, case=case, st=st, **tabs[0])
    if kind == "proj":
        from dsv41_amd.w8 import W8
        w, x = _proj_inputs(case, seed)
        s = dict(kind=kind, m=case["m"], w={k: W8(*v) for k, v in w.items()}, **x)
        if case["m"] <= 8:
            s["graph"], s["out"] = _capture(lambda: _projections(s))
        return s
    if kind == "layer":
        from dsv41_amd.attention import SparseAttention
        from dsv41_amd.w8 import W8
        w8, w, x = _layer_inputs(case, seed)
        cos, sin = _rope_tables(case["s"] + 1)
        layer = SparseAttention(dict(w, **{k: W8(*v) for k, v in w8.items()}), n_heads=H, head_dim=DV,
                                rope_head_dim=RD, window=WIN, ratio=case["ratio"], index_n_heads=case["hi"],
                                index_topk_k=case["topk"], cos=cos, sin=sin, slots=case["b"],
                                cap=case["s"] // case["ratio"] + 1, n_groups=GROUPS, o_lora_rank=ORANK)
        return dict(kind=kind, layer=layer, x=x)
    if kind == "snapshot":
        return dict(kind=kind, kbf=_index_keys(_gen(seed), case["rows"]))
    return dict(kind=kind, case=case, **_chunk_inputs(case, seed))


def _projections(s):
    from dsv41_amd.attention import linear_fp8
    from dsv41_amd.fused import norm_quant
    from dsv41_amd.w8 import fp8_gemm_tc, fp8_gemv_m1, fp8_gemv_m1_pre
    w, m = s["w"], s["m"]
    o = s["o"].view(m * GROUPS, -1)
    if m == 1:  # the GEMVs with their activation prologue
        pre = lambda x, n, norm, mode: fp8_gemv_m1_pre(x, w[n].w8, w[n].s8, norm, EPS, mode)  # noqa: E731
        return dict(wq_a=pre(s["x"], "wq_a", None, 2), wq_b=pre(s["qr"], "wq_b", s["norm"], 1),
                    wkv=pre(s["x"], "wkv", None, 2), wo_a=fp8_gemv_m1(o, w["wo_a"].w8, w["wo_a"].s8, group_cols=ORANK),
                    wo_b=pre(s["oa"], "wo_b", None, 2))
    qr = norm_quant(s["qr"], s["norm"], EPS)
    return dict(wq_a=linear_fp8(s["x"], w["wq_a"]), wq_b=fp8_gemm_tc(qr, w["wq_b"].w8, w["wq_b"].s8),
                wkv=linear_fp8(s["x"], w["wkv"]), wo_a=fp8_gemm_tc(o, w["wo_a"].w8, w["wo_a"].s8, group_cols=ORANK),
                wo_b=linear_fp8(s["oa"], w["wo_b"]))


def run(s):
    kind = s["kind"]
    if kind == "decode":
        s["graph"].replay()
        # (the caches' last row takes the writes of steps that close no group: it holds nothing)
        return dict(o=[o for o, _ in s["out"]], idx=[i for _, i in s["out"]],
                    tabs=[dict(ring=t["ring"], ckv=t["ckv"][:, :-1], k8=t["k8"].view(torch.uint8)[:, :-1],
                               ks=t["ks"][:, :-1]) for t in s["tabs"]])
    if kind == "dropin":
        from dsv41_amd import cache
        from dsv41_amd.fused2 import kv_write, sattn2
        from dsv41_amd.fused3 import index_score, topk_indices
        c, st = s["case"], s["st"]
        kv_write(st["kv_raw"], st["kv_norm"], st["cos"], st["sin"], st["pos"], s["ring"], RD, EPS, st["seq"])
        cache.append_compressed_decode(s["ckv"], st["latent"], st["pos"], st["seq"], st["row"], c["ratio"], st["cos"],
                                       st["sin"], RD)
        cache.append_index_k_decode(s["kbf"], st["k_raw"], st["k_norm"], EPS, st["pos"], st["seq"], st["row"],
                                    c["ratio"], st["cos"], st["sin"], RD)
        score = index_score(st["q_idx"], s["kbf"], st["w_idx"], st["seq"], st["cl"])
        idx = topk_indices(score, c["topk"], st["cl"])
        o = sattn2(st["q"], s["ring"], s["ckv"], idx, st["pos"], st["sink"], st["cos"], st["sin"],
                   RD if c["d"] == DV else 0, c["d"] ** -0.5, st["seq"], st["pmax"], d_v=DV)
        return dict(o=o, idx=idx, score=score, ring=s["ring"], ckv=s["ckv"][:, :-1], kbf=s["kbf"][:, :-1])
    if kind == "proj":
        if "graph" not in s:
            return _projections(s)
        s["graph"].replay()
        return s["out"]
    if kind == "index":
        from dsv41_amd.indexer import index_topk
        c = s["case"]
        e4m3 = c["keys"] == "e4m3"
        return index_topk(s["q"], s["w"], s["k8"] if e4m3 else s["kbf"], c["prior"], c["ratio"], c["topk"],
                          c["s"] + min(c["prior"], WIN - 1), k_scale=s["ks"] if e4m3 else None,
                          candidate_source=(c["blocks"], 64) if c["blocks"] else None)
    if kind == "attn":
        from dsv41_amd.kernels import sparse_attn
        return sparse_attn(s["q"], s["win"], s["sink"], s["idx"], s["case"]["d"] ** -0.5, d_v=DV, kv2=s["ckv"])
    if kind == "layer":
        lay = s["layer"]
        out = lay(s["x"], 0)
        return dict(out=out, ring=lay.ring, ckv=lay.ckv, index_k=lay.index_k, k8=lay.k8, ks=lay.ks,
                    ring_kv=lay.ring_kv, ring_score=lay.ring_score)
    from dsv41_amd.cache import index_keys_to_bf16, index_keys_to_e4m3
    k8, ks = index_keys_to_e4m3(s["kbf"])
    return dict(k8=k8.view(torch.uint8), ks=ks, back=index_keys_to_bf16(k8, ks))


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    kind = case["kind"]
    if kind in ("decode", "dropin"):
        rows, d, hi, k, ratio = case.get("rows", 1), case["d"], case["hi"], case["topk"], case["ratio"]
        key = DI + 4 if kind == "decode" else 2 * DI
        by = fl = 0
        for c in _contexts(case):
            n = c // ratio
            union = n * (1 - (1 - min(1.0, k / n)) ** rows)  # rows' selections overlap as random ones do
            by += n * key + (union + WIN) * d * 2 + rows * 2 * (d + d + DI)
            by += rows * (H * d * 2 + H * DV * 2 + hi * DI * 2 + hi * 2 + 4 * k)
            fl += rows * (2 * n * hi * DI + 2 * (min(k, n) + WIN) * H * (d + DV))
        if kind == "dropin":  # its scores come back
            by += 4 * len(_contexts(case)) * (max(max(_contexts(case)) // ratio, k) + 1)
        return dict(bytes=by * case.get("layers", 1), flops=fl * case.get("layers", 1))
    if kind == "proj":
        m = case["m"]
        by = sum(n * k + n * k // 1024 for _, n, k in PROJ) + 2 * m * (sum(n for _, n, _ in PROJ) + DIM + QRANK
                                                                     + H * DV + GROUPS * ORANK)
        return dict(bytes=by, flops=sum(2 * m * n * k for _, n, k in PROJ))
    if kind in ("index", "attn"):
        s, prior, d, hi, ratio = case["s"], case["prior"], case["d"], case["hi"], case["ratio"]
        T = (prior + s) // ratio
        cls = [(prior + i + 1) // ratio for i in range(s)]
        kk = min(case["topk"], T)
        if kind == "index":
            key = DI + 4 if case["keys"] == "e4m3" else 2 * DI
            by = T * key + s * (hi * (DI + 1) * 2 + 4 * kk) + (s * T if case["blocks"] else 0)
            return dict(bytes=by, flops=sum(2 * hi * DI * c for c in cls))
        by = s * H * 2 * (d + DV) + (T + min(prior, WIN - 1) + s) * d * 2 + 4 * s * (WIN + kk)
        return dict(bytes=by, flops=sum(2 * (min(c, kk) + min(WIN, prior + i + 1)) * H * (d + DV)
                                        for i, c in enumerate(cls)))
    if kind == "layer":
        b, s, hi, ratio = case["b"], case["s"], case["hi"], case["ratio"]
        shapes = PROJ + (("i_wq_b", hi * DI, QRANK),)
        fl = sum(2 * s * n * k for _, n, k in shapes) + 2 * s * DIM * (2 * DV + hi) + 2 * (s // ratio) * DV * DI
        for i in range(s):
            c = (i + 1) // ratio
            fl += 2 * hi * DI * c + 4 * (min(c, case["topk"]) + min(WIN, i + 1)) * H * DV
        by = sum(n * k + n * k // 1024 for _, n, k in shapes) + 8 * DV * DIM + 2 * hi * DIM + b * s * DIM * 4
        by += b * (s // ratio) * (2 * DV + 3 * DI + 4) + b * WIN * DV * 2
        return dict(bytes=by, flops=b * fl)
    return dict(bytes=case["rows"] * (DI * 2 + DI + 4) * 2, flops=0)


def tolerance(case):
    kind = case["kind"]
    if kind == "snapshot":
        return "exact"
    if kind == "attn":  # bf16 probabilities and results
        return dict(rel=8e-3, max=0.1)
    if kind == "proj":  # bf16 results
        return dict(rel=5e-3, max=0.05)
    if kind == "index":  # positions whose scores the order of a 32-bit sum can swap; the list is ascending
        return dict(rel=1e-5, differ=0.01)
    if kind == "layer":  # fp8 and fp4 grids round the earlier results' last bits to whole steps
        return dict(rel=0.03, max=0.99, differ=0.01)
    return dict(rel=0.015, max=0.9, differ=0.01)  # a swapped position moves a row's mean by one of its 2176 values


# ------------------------------------------------------------------------------------------------ in 64 bits
def _norm64(x, w):
    x = x.double()
    return (x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()).to(BF)


def _rope64(x, cos, sin, pos, inverse=False):
    """The last RD columns of x [..., d] rotated at pos (broadcast over x's leading axes), rounded to bf16."""
    c, s = cos[pos].double(), sin[pos].double()
    s = -s if inverse else s
    y = x.clone()
    t = x[..., -RD:].double()
    r, i = t[..., 0::2], t[..., 1::2]
    y[..., -RD:] = torch.stack([r * c - i * s, r * s + i * c], -1).flatten(-2).to(y.dtype)
    return y


def _attend64(q, rows, valid, sink, scale):
    """q [n, H, d], rows [n, t, d], valid [n, t] -> [n, H, DV] (the sink in the denominator only), in 64 bits."""
    q, rows = q.double(), rows.double()
    lg = torch.matmul(q, rows.transpose(1, 2).contiguous()) * scale
    lg.masked_fill_(~valid.unsqueeze(1), -math.inf)
    m = torch.maximum(lg.amax(-1), sink.double()).unsqueeze(-1)
    p = torch.exp(lg - m)
    den = p.sum(-1, keepdim=True) + torch.exp(sink.double().unsqueeze(-1) - m)
    return torch.matmul(p, rows[..., :DV].contiguous()) / den


def _scores64(q, w, keys):
    """sum_h w_h relu(q_h . key): q [n, hi, DI], w [n, hi], keys [T, DI] -> [n, T] in 64 bits."""
    n, hi, _ = q.shape
    sc = torch.matmul(q.double().reshape(n * hi, DI), keys.double().t().contiguous()).clamp_min_(0).view(n, hi, -1)
    return (sc * w.double().unsqueeze(-1)).sum(1)


def _decode_exact(case, seed, dropin):
    tabs, st = _decode_inputs(case, seed, bf16_keys=dropin)
    d, ratio, k = case["d"], case["ratio"], case["topk"]
    pos, seq, cos, sin = st["pos"], st["seq"], st["cos"], st["sin"]
    R = pos.numel()
    cl = (pos + 1) // ratio
    shut = ((pos + 1) % ratio == 0).nonzero()[:, 0]
    slot = torch.arange(WIN, device=DEV)
    res = []
    for t in tabs:
        ring, ckv = t["ring"], t["ckv"]
        ring[seq, pos % WIN] = _fq8(_rope64(_norm64(st["kv_raw"], st["kv_norm"]), cos, sin, pos))
        first = pos + 1 - ratio
        ckv[seq[shut], cl[shut] - 1] = _fq4(_rope64(st["latent"][shut, 0], cos, sin, first[shut]), 16, True)
        new = _fq4(_rope64(_norm64(st["k_raw"][shut], st["k_norm"]), cos, sin, first[shut]))
        if dropin:
            t["kbf"][seq[shut], cl[shut] - 1] = new
        else:
            n8, ns = _encode_keys(new)
            t["k8"].view(torch.uint8)[seq[shut], cl[shut] - 1] = n8.view(torch.uint8)
            t["ks"][seq[shut], cl[shut] - 1] = ns
        o = torch.empty(R, 1, H, DV, dtype=torch.float64, device=DEV)
        score = torch.full((R, ckv.shape[1]), -math.inf, dtype=torch.float64, device=DEV)
        for r in range(R):
            s, c = int(seq[r]), int(cl[r])
            keys = t["kbf"][s, :c] if dropin else t["k8"][s, :c].double() * t["ks"][s, :c, None].double()
            score[r, :c] = _scores64(st["q_idx"][r], st["w_idx"][r:r + 1], keys)[0]
            sel = score[r, :c].topk(min(k, c)).indices
            held = st["pmax"][r] - (st["pmax"][r] - slot) % WIN
            ok = (held >= 0) & (held <= pos[r]) & (pos[r] - held < WIN)
            rows = torch.cat([ring[s], ckv[s, sel]])
            ok = torch.cat([ok, torch.ones_like(sel, dtype=torch.bool)])
            o[r, 0] = _attend64(st["q"][r], rows[None], ok[None], st["sink"], d ** -0.5)[0]
        if d == DV:
            o = _rope64(o, cos, sin, pos.view(R, 1, 1), inverse=True)
        res.append((o, score))
    if dropin:
        return dict(o=res[0][0], idx=None, score=res[0][1], ring=tabs[0]["ring"], ckv=tabs[0]["ckv"][:, :-1],
                    kbf=tabs[0]["kbf"][:, :-1])
    return dict(o=[o for o, _ in res], idx=[None] * len(res),
                tabs=[dict(ring=t["ring"], ckv=t["ckv"][:, :-1], k8=None, ks=t["ks"][:, :-1]) for t in tabs])


def _lin64(x, w):
    return torch.matmul(x.double(), w.double().t().contiguous())


def _proj_exact(case, seed):
    w8, x = _proj_inputs(case, seed)
    w = {k: _w8_64(v) for k, v in w8.items()}
    o = x["o"].view(-1, GROUPS, H * DV // GROUPS)
    oa = torch.cat([_lin64(o[:, i], w["wo_a"][i * ORANK:(i + 1) * ORANK]) for i in range(GROUPS)], -1)
    return dict(wq_a=_lin64(_fq8(x["x"]), w["wq_a"]), wq_b=_lin64(_fq8(_norm64(x["qr"], x["norm"])), w["wq_b"]),
                wkv=_lin64(_fq8(x["x"]), w["wkv"]), wo_a=oa, wo_b=_lin64(_fq8(x["oa"]), w["wo_b"]))


def _gather_attend(q, kv, idx, sink, scale, step=48):
    """q [s, H, d], kv [n, d], idx [s, t] (-1 = none) -> [s, H, DV], in 64 bits."""
    return torch.cat([_attend64(q[i:i + step], kv[idx[i:i + step].clamp_min(0).long()], idx[i:i + step] >= 0, sink,
                                scale) for i in range(0, q.shape[0], step)])


def _select64(q, w, keys, cl, k):
    """Per query the k best of keys[:cl] by the 64-bit scores, ascending, -1 past them: [s, k]."""
    T = keys.shape[0]
    t = torch.arange(T, device=DEV)
    out = []
    for i in range(0, q.shape[0], 16):
        sc = _scores64(q[i:i + 16], w[i:i + 16], keys).masked_fill_(t >= cl[i:i + 16, None], -math.inf)
        val, sel = sc.topk(k, -1)
        sel = torch.where(torch.isinf(val), T, sel).sort(-1).values
        out.append(torch.where(sel < T, sel, -1))
    return torch.cat(out)


def _layer_exact(case, seed):
    w8, w, x = _layer_inputs(case, seed)
    w = dict(w, **{k: _w8_64(v) for k, v in w8.items()})
    b, s, hi, ratio, k = case["b"], case["s"], case["hi"], case["ratio"], case["topk"]
    cos, sin = _rope_tables(s + 1)
    at = torch.arange(s, device=DEV)
    T = s // ratio
    kk = min(k, T)
    lin8 = lambda v, n: _lin64(_fq8(v), w[n]).to(BF)  # noqa: E731
    out = []
    ring = torch.zeros(b, WIN, DV, dtype=BF, device=DEV)
    ckv = torch.zeros(b, T + 1, DV, dtype=BF, device=DEV)
    index_k = torch.zeros(b, T + 1, DI, dtype=BF, device=DEV)
    rk = torch.zeros(b, 8, DV, dtype=torch.float64, device=DEV)
    rs = torch.full((b, 8, DV), -math.inf, dtype=torch.float64, device=DEV)
    widx = (at[:, None] - WIN + 1).clamp_min(0) + torch.arange(min(WIN, s), device=DEV)
    widx = torch.where(widx <= at[:, None], widx, -1)
    for i in range(b):
        qr = _norm64(lin8(x[i], "wq_a"), w["q_norm_w"])
        q = _rope64(lin8(qr, "wq_b").view(s, H, DV), cos, sin, at[:, None])
        win = _fq8(_rope64(_norm64(lin8(x[i], "wkv"), w["kv_norm_w"]), cos, sin, at))
        ring[i, at[-WIN:] % WIN] = win[-WIN:]
        kv, gate = _lin64(x[i], w["c_wkv"]), _lin64(x[i], w["c_wgate"])
        rk[i, at[-8:] % 8], rs[i, at[-8:] % 8] = kv[-8:], gate[-8:]
        n = T * ratio
        pool = (kv[:n].view(T, ratio, -1) * torch.softmax(gate[:n].view(T, ratio, -1), 1)).sum(1).to(BF)
        lat = _norm64(pool, w["c_norm_w"])
        key = _fq4(_rope64(_norm64(_lin64(lat, w["i_wk"]).to(BF), w["i_k_norm_w"]), cos, sin, at[:n:ratio]))
        index_k[i, :T] = key
        ckv[i, :T] = _fq4(_rope64(lat, cos, sin, at[:n:ratio]), 16, True)
        qi = _fq4(_rope64(lin8(qr, "i_wq_b").view(s, hi, DI), cos, sin, at[:, None]))
        wi = (_lin64(x[i], w["i_weights_proj"]).to(BF).float() * (DI ** -0.5 * hi ** -0.5)).to(BF)
        sel = _select64(qi, wi, key, (at + 1) // ratio, kk)
        idx = torch.cat([widx, torch.where(sel >= 0, sel + s, -1)], -1)
        o = _gather_attend(q, torch.cat([win, ckv[i, :T]]), idx, w["attn_sink"], DV ** -0.5, 96).to(BF)
        o = _rope64(o, cos, sin, at[:, None], inverse=True).reshape(s, GROUPS, -1)
        oa = torch.cat([_lin64(o[:, j], w["wo_a"][j * ORANK:(j + 1) * ORANK]) for j in range(GROUPS)], -1).to(BF)
        out.append(_lin64(_fq8(oa), w["wo_b"]))
    return dict(out=torch.stack(out), ring=ring, ckv=ckv, index_k=index_k, k8=None, ks=None, ring_kv=rk, ring_score=rs)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "dropin"):
        return _decode_exact(case, seed, kind == "dropin")
    if kind == "proj":
        return _proj_exact(case, seed)
    if kind == "attn":
        x = _chunk_inputs(case, seed)
        return _gather_attend(x["q"][0], torch.cat([x["win"][0], x["ckv"][0]]), x["idx"][0], x["sink"],
                              case["d"] ** -0.5)[None]
    if kind == "layer":
        return _layer_exact(case, seed)
    return None  # positions and stored bytes: whole values, compared as they are
