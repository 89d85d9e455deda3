"""GPU parity of the shapes the unit cases do not reach: the attention's many-row kernels (16-255 query rows: the
64-head kernel with key splits and its combine, in both head geometries), the full C3 prefill chunk, the one-launch
decode indexer against the oracle directly, and the reference's own indexer geometry (32 index heads, ratio 2,
top-k 512, dsv41/decode.py:252, README.md:402).

Bars as in test_gpu_parity.py: top-k bit-exact given identical scores, scores within 1e-2 relative, attention max
|err| <= 2e-2 and mean <= 2e-3, quantised cache rows bit-exact up to rare one-step fp8 flips."""
import numpy as np
import pytest
import torch

from oracle import dsv41_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ATT_MAX, ATT_MEAN = 2e-2, 2e-3


def bf(x):
    return torch.from_numpy(np.ascontiguousarray(O.bf16(x))).to(torch.bfloat16).to(DEV)


def f32(x):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(x, np.float32))).to(DEV)


def i64(x):
    return torch.tensor(np.asarray(x, np.int64), device=DEV)


def host(t):
    return t.float().cpu().numpy()


def attn_close(got, want, tag=""):
    err = np.abs(got - want)
    print(f"[{tag}] max {err.max():.3e} mean {err.mean():.3e}", flush=True)
    assert err.max() <= ATT_MAX, (tag, err.max())
    assert err.mean() <= ATT_MEAN, (tag, err.mean())


def _fp8_close(got, want, tag):
    diff = got != want
    print(f"[{tag}] mismatching elements {diff.sum()} ({diff.mean():.2e})", flush=True)
    assert diff.mean() <= 2e-3, tag
    if diff.any():
        rel = np.abs(got[diff] - want[diff]) / np.maximum(np.abs(want[diff]), 1e-30)
        assert rel.max() <= 0.34, (tag, rel.max())


def _rope_tables(rd, n):
    ang = torch.outer(torch.arange(n, dtype=torch.float32),
                      1.0 / (10000.0 ** (torch.arange(0, rd, 2, dtype=torch.float32) / rd)))
    return torch.cos(ang), torch.sin(ang)


# ------------------------------------------------------------------------------------------ many-row attention
@pytest.mark.parametrize("dqk,R,k,n,nsplit", [(576, 32, 2048, 6000, 0), (576, 48, 300, 250, 0), (512, 24, 512, 9000, 0),
                                              (512, 16, 512, 700, 1), (512, 40, 130, 4000, 3), (512, 300, 100, 99, 0),
                                              (512, 16, 4100, 6000, 0), (576, 16, 4100, 6000, 0), (512, 17, 900, 1500, 12),
                                              (512, 16, 2000, 2500, 67), (576, 16, 2000, 2500, 67), (256, 16, 700, 900, 0),
                                              (128, 24, 500, 700, 3), (64, 16, 500, 600, 10), (64, 33, 130, 600, 0)])
def test_sattn2_many_rows_unit_scale(dqk, R, k, n, nsplit):
    """The 64-head kernel, with (up to 512) and without (576) the inverse rope of the result, up to 67 splits (its
    combine takes 8 at once, up to 32 and more in three ways), at values of unit size against a float64 softmax, three
    launches bit-equal: gathers still in flight when the output is staged would show in single elements.  Rows end in
    empty entries as short contexts do.
    Bound per output row: bf16 probabilities, partials and result round by at most 2^-8, in the 2-norm by under 2^-8.5
    each (independent): sqrt(3) 2^-8.5 < 2^-7."""
    import dsv41_amd
    g = torch.Generator(device=DEV).manual_seed(7)
    H, dv, win = 64, min(dqk, 512), 128
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    q, ring, ckv = rn(R, 1, H, dqk), rn(R, win, dqk), rn(R, n, dqk)
    sink = torch.randn(H, generator=g, device=DEV)
    idx = torch.rand(R, n, generator=g, device=DEV).argsort(-1)[:, :k].to(torch.int32)
    if k > n:
        idx = torch.cat([idx, torch.full((R, k - n), -1, device=DEV, dtype=torch.int32)], -1)
    for r in range(R):  # ever shorter contexts: -1 tails
        idx[r, k - (r * k) // (R + 4):] = -1
    pos = torch.arange(R, device=DEV) + 5000
    seq = torch.arange(R, device=DEV)
    cos, sin = (x.to(DEV) for x in _rope_tables(64, 8192))
    rd = 0 if dqk == 576 else 64
    got = [dsv41_amd.sattn2(q, ring, ckv, idx.unsqueeze(1), pos, sink, cos, sin, rd, dqk ** -0.5, seq, pos, d_v=dv,
                            nsplit=nsplit) for _ in range(3)]
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    for r in range(R):
        sel = idx[r][idx[r] >= 0].long()
        rows = torch.cat([ring[r], ckv[r, sel]]).double()
        lg = q[r, 0].double() @ rows.t() * dqk ** -0.5
        e = torch.exp(lg - lg.amax(-1, keepdim=True))
        want = e @ rows[:, :dv] / (e.sum(-1, keepdim=True) + torch.exp(sink.double()[:, None] - lg.amax(-1, keepdim=True)))
        if rd:  # inverse rope on the last rd columns
            c, s = cos[pos[r]].double(), -sin[pos[r]].double()
            a, b = want[:, -rd::2].clone(), want[:, -rd + 1::2].clone()
            want[:, -rd::2], want[:, -rd + 1::2] = a * c - b * s, a * s + b * c
        rel = (got[0][r, 0].double() - want).norm(dim=-1) / want.norm(dim=-1)
        assert rel.max() < 2 ** -7, (r, float(rel.max()))


@pytest.mark.parametrize("nsplit", [0, 3, 1])
def test_sattn2_mla_48_rows_ragged_drafts(nsplit):
    """C5's attention shape (dsv41/fused2.py:334-446): 8 ragged slots x (1 + 5 MTP drafts) = 48 rows, absorbed MLA
    576/512, draft rows causal among themselves through plim, top-k 2048 capped by each row's compressed length.
    48 rows run the 64-head kernel; nsplit 0 (the library's plan: key splits + the combine kernel), 3 (forced
    splits) and 1 (no split) share one workspace."""
    import dsv41_amd
    from dsv41_amd._lib import lib
    r = np.random.default_rng(40)
    H, dqk, dv, win, k = 64, 576, 512, 128, 2048
    ctx = [32768, 8192, 8192, 8192, 4096, 2048, 512, 64]
    S, D = len(ctx), 6
    n_cap = max(ctx) // 4 + 1
    B = S * D
    q = O.bf16(r.standard_normal((B, 1, H, dqk)).astype(np.float32))
    sink = r.standard_normal(H).astype(np.float32)
    ring = O.bf16(r.standard_normal((S, win, dqk)).astype(np.float32) * 0.1)
    ckv = O.bf16(r.standard_normal((S, n_cap, dqk)).astype(np.float32) * 0.1)
    pos, seq, pmax = [], [], []
    for s, c in enumerate(ctx):
        for j in range(D):
            pos.append(c - D + j)
            seq.append(s)
            pmax.append(c - 1)
    idx = np.full((B, 1, k), -1, np.int32)
    for b in range(B):
        cl = (pos[b] + 1) // 4
        nv = min(k, cl)
        idx[b, 0, :nv] = np.sort(r.choice(cl, nv, replace=False))
    zero = np.zeros((1, 1), np.float32)
    want = O.sattn2(q, ring, ckv, idx, pos, seq, pmax, pos, sink, zero, zero, 0, dqk ** -0.5, dv=dv)
    nbytes = max(lib().dsv41_attn_workspace_bytes(B, H, win + k, dv, n) for n in (0, 3, 1))
    ws = torch.zeros(max(nbytes, 4) // 4, dtype=torch.float32, device=DEV)
    for rep in range(2):
        o = dsv41_amd.sattn2(bf(q), bf(ring), bf(ckv), torch.from_numpy(idx).to(DEV), i64(pos), f32(sink), f32(zero),
                             f32(zero), 0, dqk ** -0.5, i64(seq), i64(pmax), plim=i64(pos), d_v=dv, nsplit=nsplit,
                             ws=ws)
        attn_close(host(o), want, f"sattn2 mla 48 rows nsplit {nsplit} rep {rep}")


@pytest.mark.parametrize("R,nsplit", [(16, 0), (32, 0), (32, 4), (64, 0)])
def test_sattn2_reference_geometry_many_rows(R, nsplit):
    """The reference's geometry (head_dim 512, in-row rope on the last 64 columns, inverse rope on the output,
    dsv41/fused2.py:434-446) at 16-64 decode slots (run_16slots.sh / run_64slots.sh): the 64-head split kernel +
    its combine (key splits)."""
    import dsv41_amd
    r = np.random.default_rng(41 + R)
    H, hd, win, rd, n_c, t = 64, 512, 128, 64, 4097, 512
    cos, sin = O.rope_tables(rd, 8192, 0, 10000.0, 1.0, 32, 1)
    S = R
    q = O.bf16(r.standard_normal((R, 1, H, hd)).astype(np.float32))
    sink = r.standard_normal(H).astype(np.float32)
    ring = O.bf16(r.standard_normal((S, win, hd)).astype(np.float32))
    ckv = O.bf16(r.standard_normal((S, n_c, hd)).astype(np.float32))
    pos = r.integers(30, 8000, R).tolist()
    seq = list(range(R))
    idx = np.full((R, 1, t), -1, np.int32)
    for b in range(R):
        cl = min((pos[b] + 1) // 2, n_c)
        nv = min(t - 37, cl)
        idx[b, 0, :nv] = np.sort(r.choice(cl, nv, replace=False))
    o = dsv41_amd.sattn2(bf(q), bf(ring), bf(ckv), torch.from_numpy(idx).to(DEV), i64(pos), f32(sink), f32(cos),
                         f32(sin), rd, hd ** -0.5, i64(seq), i64(pos), nsplit=nsplit)
    want = O.sattn2(q, ring, ckv, idx, pos, seq, pos, None, sink, cos, sin, rd, hd ** -0.5)
    attn_close(host(o), want, f"sattn2 ref geometry R={R} nsplit {nsplit}")


# ------------------------------------------------------------------------------------------ C3 at full size
def test_prefill_c3_full_size():
    """The C3 chunk (2048 queries after 65536 tokens, 16896 compressed rows, top-k 2048, 128 window + 2048 indices
    per query), as the benchmark runs it: index_topk into the compressed columns of the [window | compressed] index
    buffer, then sparse_attn over the window rows and the compressed table read in place.
    Every row: indices ascending, below the causal limit, -1 only as a tail, bit-exact re-selection by the oracle
    from the kernel's own scores.  64 sampled rows: scores within 1e-2 of the oracle, the selection agreeing with
    the oracle's own, and the attention output against the oracle."""
    from dsv41_amd.indexer import index_topk
    from dsv41_amd.kernels import sparse_attn
    from dsv41_amd.workloads import DI, DQK, DV, H, PREFILL, WIN, make_prefill_inputs
    cfg = PREFILL["C3"]
    x = make_prefill_inputs(cfg, DEV)
    S, T, k = cfg.chunk, cfg.n_c, cfg.topk
    sink = (torch.randn(H, generator=torch.Generator().manual_seed(3))).to(DEV)
    idx_buf = torch.full((1, S, WIN + k), 7777, dtype=torch.int32, device=DEV)
    widx = x["widx"]
    off = x["win"].shape[1]
    _, score = index_topk(x["q_idx"], x["w_idx"], x["k8"], cfg.prior, cfg.ratio, k, off, k_scale=x["ks"],
                          return_score=True, out=idx_buf[:, :, WIN:])
    idx_buf[:, :, :WIN] = widx
    o = sparse_attn(x["q"], x["win"], sink, idx_buf, DQK ** -0.5, d_v=DV, kv2=x["ckv"])
    torch.cuda.synchronize()
    sel = idx_buf[0, :, WIN:].cpu().numpy()
    sc = score[0].cpu().numpy()
    cls = (cfg.prior + np.arange(S) + 1) // cfg.ratio
    comp = np.where(sel >= 0, sel - off, -1)
    for i in range(0, S, 256):
        print(f"[c3] rows {i}..{i + 255}", flush=True)
        for j in range(i, i + 256):
            v = comp[j][comp[j] >= 0]
            assert np.all(np.diff(v) > 0), j
            assert v.size == 0 or v[-1] < cls[j], j
            nv = v.size
            assert np.all(comp[j, nv:] == -1), j  # -1 only as a tail
        resel = O.topk_indices(sc[i:i + 256], k, cls[i:i + 256])
        np.testing.assert_array_equal(comp[i:i + 256], resel, err_msg=f"rows {i}..")
    rows = np.random.default_rng(5).choice(S, 64, replace=False)
    rows.sort()
    qi = host(x["q_idx"])[0, rows]
    wi = host(x["w_idx"])[0, rows]
    kk = host(x["k8"])[0] * x["ks"].cpu().numpy()[0][:, None]
    want_sc = np.zeros((64, T), np.float32)
    for h in range(H):
        want_sc += wi[:, h:h + 1] * np.maximum(qi[:, h] @ kk.T, 0)
    want_sc = np.where(np.arange(T)[None] < cls[rows][:, None], want_sc, -np.inf).astype(np.float32)
    fin = np.isfinite(want_sc)
    got_sc = sc[rows]
    assert np.array_equal(np.isfinite(got_sc) | ~fin, np.ones_like(fin))  # finite wherever the oracle is
    for n, j in enumerate(rows):
        m = fin[n]
        err = np.abs(got_sc[n][m] - want_sc[n][m]).max() / np.abs(want_sc[n][m]).max()
        assert err <= 1e-2, (j, err)
    agree = (O.topk_indices(want_sc, k, cls[rows]) == comp[rows]).mean()
    print(f"[c3] selection agreement with the oracle on 64 rows: {agree:.5f}", flush=True)
    assert agree >= 0.999
    kv_all = np.concatenate([host(x["win"])[0], host(x["ckv"])[0]])[None]
    idx_rows = idx_buf[0, rows].cpu().numpy()[None]
    want_o = O.sparse_attn(host(x["q"])[:, rows], kv_all, sink.cpu().numpy(), idx_rows, DQK ** -0.5, dv=DV)
    attn_close(host(o)[:, rows], want_o, "c3 attention 64 rows")


# ------------------------------------------------------------------------------------------ one-launch indexer
def _decode_geometry(dev, ctx, Dw, HI, ratio, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    from dsv41_amd.workloads import encode_e4m3_rows, fp4_round
    S = len(ctx)
    cap = max(c // ratio for c in ctx) + 8
    ring = (torch.randn(S, 128, Dw, generator=g, device=dev) * 0.1).to(torch.bfloat16)
    ckv = (torch.randn(S, cap, Dw, generator=g, device=dev) * 0.1).to(torch.bfloat16)
    kk = torch.randn(S, cap, 128, generator=g, device=dev) * 0.1
    kk[..., [3, 40, 77, 120]] *= 8
    kbf = fp4_round(kk)
    k8, ks = encode_e4m3_rows(kbf)
    return dict(ring=ring, ckv=ckv, kbf=kbf, k8=k8, ks=ks, g=g, cap=cap)


@pytest.mark.parametrize("geom", ["mla", "reference"])
def test_decode_select_against_oracle(geom):
    """dsv41_decode_select (DecodeLayer.appends_select: the step's cache appends, index-query preparation, scores and
    top-k in one launch) against the oracle directly, over a closing and a non-closing step: the ring row
    (O.kv_write), the compressed row (O.compress_row) and the index-key row (O.index_key_row) written, the kernel's
    scores within 1e-2 of O.index_score over the updated keys, the indices bit-exact against O.topk_indices of the
    kernel's scores and agreeing >= 0.999 with O.topk_indices of the oracle's scores.
    mla: 576-wide rows, 64 index heads, ratio 4, k 2048; reference: 512-wide rows, 32 index heads, ratio 2, k 512."""
    from dsv41_amd.decode import DecodeLayer
    if geom == "mla":
        Dw, HI, ratio, k, ctx = 576, 64, 4, 2048, [65536, 8192, 40000, 12]
    else:
        Dw, HI, ratio, k, ctx = 512, 32, 2, 512, [30000, 4096, 1001, 9]
    from dsv41_amd.workloads import fp4_round
    rd = 64
    d = _decode_geometry(DEV, ctx, Dw, HI, ratio, 50 + HI)
    g = d["g"]
    cos_t, sin_t = _rope_tables(rd, max(ctx) + 16)
    cos, sin = cos_t.to(DEV), sin_t.to(DEV)
    sink = torch.randn(64, generator=g, device=DEV)
    L = DecodeLayer(d["ring"].clone(), d["ckv"].clone(), d["k8"].clone(), d["ks"].clone(), sink, cos, sin, ratio, k,
                    rd=rd, dv=Dw if Dw == 512 else 512)
    sel = L.selector(len(ctx), DEV)
    assert sel.one_launch
    sel.keep_scores = True
    B = len(ctx)
    seq = i64(list(range(B)))
    kvn = (torch.rand(Dw, generator=g, device=DEV) + 0.5).to(torch.bfloat16)
    kn = (torch.rand(128, generator=g, device=DEV) + 0.5).to(torch.bfloat16)
    cosn, sinn = cos_t.numpy(), sin_t.numpy()
    for step in range(2):
        # step 0: positions close their compression group; step 1: they do not (spare row)
        pos_l = [c - 1 + step for c in ctx]
        pos = i64(pos_l)
        kv_raw = torch.randn(B, Dw, generator=g, device=DEV).to(torch.bfloat16)
        latent = torch.randn(B, 1, Dw, generator=g, device=DEV).to(torch.bfloat16)
        k_raw = (torch.randn(B, 128, generator=g, device=DEV) * 2).to(torch.bfloat16)
        q_idx = fp4_round(torch.randn(B, 1, HI, 128, generator=g, device=DEV))
        w_idx = (torch.randn(B, HI, generator=g, device=DEV) * (128 ** -0.5 * HI ** -0.5)).to(torch.bfloat16)
        ring0, ckv0 = host(L.ring), host(L.ckv)
        k80, ks0 = L.k8.float().cpu().numpy(), L.ks.cpu().numpy()
        cl_l = [(p + 1) // ratio for p in pos_l]
        print(f"[decode_select {geom}] step {step} pos {pos_l}", flush=True)
        idx = L.appends_select(kv_raw, kvn, latent, k_raw, kn, pos, seq, q_idx, w_idx, cl=i64(cl_l)).clone()
        torch.cuda.synchronize()
        assert int(sel.fws[-4].item()) == 0, "row barrier wait gave up"
        # cache rows against the oracle's append arithmetic
        want_ring = O.kv_write(host(kv_raw), host(kvn), cosn, sinn, pos_l, list(range(B)), ring0, rd, 1e-6)
        _fp8_close(host(L.ring), want_ring, f"{geom} ring step {step}")
        want_c, want_k = ckv0.copy(), k80 * ks0[..., None]
        for b in range(B):
            row = cl_l[b] - 1 if (pos_l[b] + 1) % ratio == 0 else L.ckv.shape[1] - 1
            p0 = np.int64(pos_l[b] + 1 - ratio)
            want_c[b, row] = O.compress_row(host(latent)[b, 0], cosn, sinn, p0, rd)
            want_k[b, row] = O.index_key_row(host(k_raw)[b], host(kn), cosn, sinn, p0, rd, 1e-6)
        _fp8_close(host(L.ckv), want_c, f"{geom} compressed step {step}")
        got_k = L.k8.float().cpu().numpy() * L.ks.cpu().numpy()[..., None]
        _fp8_close(got_k, want_k, f"{geom} index keys step {step}")
        # scores and selection
        sc = sel.score.cpu().numpy()
        want_sc = O.index_score(host(q_idx), L.k8.float().cpu().numpy(), host(w_idx), list(range(B)), cl_l,
                                k_scale=L.ks.cpu().numpy())
        for b in range(B):
            c = cl_l[b]
            err = np.abs(sc[b, :c] - want_sc[b, :c]).max() / np.abs(want_sc[b, :c]).max()
            assert err <= 1e-2, (geom, step, b, err)
        got = idx.cpu().numpy()[:, 0]
        np.testing.assert_array_equal(got, O.topk_indices(sc, k, cl_l), err_msg=f"{geom} step {step}")
        agree = (got == O.topk_indices(want_sc, k, cl_l)).mean()
        print(f"[decode_select {geom}] step {step} agreement with the oracle {agree:.5f}", flush=True)
        assert agree >= 0.999


# ------------------------------------------------------------------------------------------ reference geometry
def test_index_topk_reference_geometry():
    """Indexer.__call__ prefill selection (dsv41/model.py:766-893) at the reference's geometry: 32 index heads,
    ratio 2, top-k 512, bf16 and e4m3 keys; plus the prefill appends at ratio 2 (dsv41/model.py:1300-1348,
    :696-732) against the oracle's rows."""
    import dsv41_amd
    from dsv41_amd import cache as C
    r = np.random.default_rng(60)
    b, s, H, D, start, ratio, topk, offset = 1, 200, 32, 128, 1500, 2, 512, 131
    T = (start + s) // ratio
    q = O.bf16(O.fake_quant_fp4(O.bf16(r.standard_normal((b, s, H, D)).astype(np.float32)), 32))
    w = O.bf16(r.standard_normal((b, s, H)).astype(np.float32) * (D ** -0.5 * H ** -0.5))
    keys = O.bf16(O.fake_quant_fp4(O.bf16(r.standard_normal((b, T + 3, D)).astype(np.float32) * 0.1), 32))
    q8, s8 = O.key_encode_fp8(keys)
    want = O.indexer_prefill(q, w, keys, start, ratio, topk, offset)
    got, score = dsv41_amd.index_topk(bf(q), bf(w), bf(keys), start, ratio, topk, offset, return_score=True)
    got8 = dsv41_amd.index_topk(bf(q), bf(w), torch.from_numpy(q8).to(torch.float8_e4m3fn).to(DEV), start, ratio,
                                topk, offset, k_scale=f32(s8[..., 0]))
    sc = score.cpu().numpy()[0]
    cls = (start + np.arange(s) + 1) // ratio
    resel = O.topk_indices(sc, min(topk, T), cls)
    np.testing.assert_array_equal(got.cpu().numpy()[0], np.where(resel >= 0, resel + offset, -1))
    np.testing.assert_array_equal(got.cpu().numpy(), got8.cpu().numpy())
    agree = (got.cpu().numpy() == want).mean()
    print(f"[index_topk ref geometry] agreement with oracle {agree:.5f}", flush=True)
    assert agree >= 0.999
    # prefill appends at ratio 2: compressed rows (512 wide) and index keys (bf16 + e4m3 copy)
    rd, n_new, st = 64, s // ratio, start
    cos, sin = O.rope_tables(rd, 4096, 0, 10000.0, 1.0, 32, 1)
    lat = O.bf16(r.standard_normal((1, n_new, 512)).astype(np.float32))
    kraw = O.bf16(r.standard_normal((1, n_new, 128)).astype(np.float32) * 2)
    kn = O.bf16(r.random(128).astype(np.float32) + 0.5)
    cap = T + 4
    ckv = torch.zeros(1, cap, 512, dtype=torch.bfloat16, device=DEV)
    kb = torch.zeros(1, cap, 128, dtype=torch.bfloat16, device=DEV)
    k8t = torch.zeros(1, cap, 128, dtype=torch.uint8, device=DEV)
    kst = torch.zeros(1, cap, dtype=torch.float32, device=DEV)
    C.write_compress_kv(ckv, bf(lat), st, ratio, f32(cos), f32(sin), rd)
    C.write_index_k(kb, bf(kraw), bf(kn), 1e-6, st, ratio, f32(cos), f32(sin), rd, k8=k8t, k_scale=kst)
    wc = np.zeros((1, cap, 512), np.float32)
    wk = np.zeros((1, cap, 128), np.float32)
    for i in range(n_new):
        p = np.int64(st - st % ratio + i * ratio)
        wc[0, st // ratio + i] = O.compress_row(lat[0, i], cos, sin, p, rd)
        wk[0, st // ratio + i] = O.index_key_row(kraw[0, i], kn, cos, sin, p, rd, 1e-6)
    _fp8_close(host(ckv), wc, "ratio-2 compressed append")
    _fp8_close(host(kb), wk, "ratio-2 index-key append")
    dec = k8t.view(torch.float8_e4m3fn).float().cpu().numpy() * kst.cpu().numpy()[..., None]
    np.testing.assert_array_equal(dec, host(kb))


def test_decode_selector_reference_geometry():
    """index_score + topk_indices of the graph decode (dsv41/decode.py:284-294) at 32 index heads and k 512 on the
    multi-launch path (rows past the one-launch limit: 600 positions over 8 rows is one launch, 200000 is not)."""
    from dsv41_amd.fused3 import DecodeSelector
    from dsv41_amd.workloads import encode_e4m3_rows, fp4_round
    g = torch.Generator(device=DEV).manual_seed(61)
    for n, cls in ((601, [600, 600, 17, 512, 1, 300, 599, 2]), (200001, [200000, 77777])):
        R = len(cls)
        keys = fp4_round(torch.randn(R, n, 128, generator=g, device=DEV) * 0.1)
        k8, ks = encode_e4m3_rows(keys)
        q = fp4_round(torch.randn(R, 1, 32, 128, generator=g, device=DEV))
        w = (torch.randn(R, 32, generator=g, device=DEV) * 0.03).to(torch.bfloat16)
        seq = i64(list(range(R)))
        sel = DecodeSelector(R, n, 512, DEV, keep_scores=True, max_cl=n - 1)
        print(f"[selector ref geometry] n {n} one_launch {sel.one_launch}", flush=True)
        idx = sel(q, k8, w, seq, i64(cls), k_scale=ks)
        torch.cuda.synchronize()
        sc = sel.score.cpu().numpy()
        np.testing.assert_array_equal(idx.cpu().numpy()[:, 0], O.topk_indices(sc, 512, cls))
        want = O.index_score(host(q), k8.float().cpu().numpy(), host(w), list(range(R)), cls,
                             k_scale=ks.cpu().numpy())
        for b, c in enumerate(cls):
            err = np.abs(sc[b, :c] - want[b, :c]).max() / max(np.abs(want[b, :c]).max(), 1e-30)
            assert err <= 1e-2, (n, b, err)
