"""The passes that work on the stream formats in place (C-stream order, A layout, attention tiles) against the oracle,
and against the general forms that first bring the operands to row-major order."""

import numpy as np
import pytest
import torch

from oracle import attn as A
from oracle import bfp16 as F
from oracle import gemm as G
from oracle import ln as LN
from rlbfp import forward, layouts, ops, run_attn, run_ln, run_qkv

pytestmark = pytest.mark.gpu


def tt(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda").to(dtype)


@pytest.mark.parametrize("M,D,S,branch,norm", [
    (512, 1024, 0, "packed", "layer"), (512, 2048, 3, "bf16", "rms"), (1024, 3072, 1, "none", "layer"),
    (512, 4096, 5, "packed", "rms"), (512, 5120, 0, "bf16", "layer"), (512, 6144, 2, "packed", "layer"),
    (512, 7168, 4, "none", "rms"), (512, 8192, 1, "packed", "layer")])
def test_ln_stream(dev, M, D, S, branch, norm):
    """Every width the kernel has a variant for, each branch format: x' bit-exact; y equal to the oracle's in 99.9% of
    values (float32 against float64 sums, so a value at a rounding tie may take either side) and within 1e-2."""
    rng = np.random.default_rng(M + D + S)
    x = F.bf16_round((rng.standard_normal((M, D)) * 3).astype(np.float32))
    x[:, 7] += 32
    x = F.bf16_round(x)
    br = F.bf16_round(rng.standard_normal((M, D)).astype(np.float32))
    p = LN.ln_params(np.tanh(rng.standard_normal((2, D))), 1 + 0.3 * rng.standard_normal((2, D)))
    xs = run_ln.ln_pack_x(tt(x))
    brs = {"none": None, "bf16": run_ln.ln_pack_x(tt(br)), "packed": run_ln.ln_pack_br(tt(br))}[branch]
    ref_br = {"none": np.zeros_like(br), "bf16": br, "packed": F.quantize_rows(br)}[branch]
    art = f"{'vlm-rms' if norm == 'rms' else 'glue-ln'}-m{M}-s{S}"
    pt = tt(p, torch.bfloat16).reshape(-1)
    xo, ao = torch.full_like(xs, 7.0), torch.full((M * D // 8 * 9,), 7, dtype=torch.uint8, device="cuda")
    run_ln.ln_fused(art, xs, brs, pt, xo, ao)
    xp, y = run_ln.ln_unpack(xo, ao, M)
    xr, yr = LN.ln_mod_ref(x, ref_br, p, split_row=S * 128, norm=norm)
    np.testing.assert_array_equal(xp.cpu().numpy(), xr)
    y = y.cpu().numpy()
    assert G.rel_err(y, yr) <= 1e-2
    assert (y == F.quantize_rows(yr.astype(np.float32))).mean() > 0.999
    # x' in place
    run_ln.ln_fused(art, xs, brs, pt, xs, torch.zeros_like(ao))
    assert torch.equal(xs, xo)


def test_ln_stream_general_form(dev):
    """Buffers that the stream kernel does not take in place (an output over the branch, an unaligned address) go
    through the general form, with the same x' and A up to ties."""
    M, D = 512, 1024
    rng = np.random.default_rng(5)
    x, br = tt(rng.standard_normal((M, D)) * 2, torch.bfloat16), tt(rng.standard_normal((M, D)))
    p = run_ln.ln_params(tt(np.tanh(rng.standard_normal((2, D)))), tt(1 + 0.1 * rng.standard_normal((2, D))))
    xs, brs = run_ln.ln_pack_x(x), run_ln.ln_pack_br(br)
    xo, ao = torch.zeros_like(xs), forward.v9(M * D)
    assert run_ln._stream_form(xs, brs, p, xo, ao, M, D)
    run_ln.ln_fused("glue-ln-m512-s1", xs, brs, p, xo, ao)
    over = brs.clone()
    off = torch.zeros(M * D + 1, dtype=torch.bfloat16, device="cuda")[1:]
    off.copy_(xs)
    for X, B, A in ((xs, over, over), (off, brs, torch.zeros_like(ao))):
        assert not run_ln._stream_form(X, B, p, xo, A, M, D)
        x2 = torch.zeros_like(xs)
        run_ln.ln_fused("glue-ln-m512-s1", X, B, p, x2, A)
        assert torch.equal(x2, xo)
        assert (layouts.from_bfp16(A) == layouts.from_bfp16(ao)).float().mean() > 0.999


# ---- attention on packed tiles ------------------------------------------------------------------------------------

def tiles(rng, heads, t, kv=False):
    """Random Q ([head][tile]) or KV ([head][tile][K | V]) tiles and their decoded values (heads, 64 t, 128)."""
    mk = lambda: rng.standard_normal((heads, 64 * t, 128)).astype(np.float32)
    rows = lambda x, h, i: x[h, 64 * i:64 * i + 64]
    if not kv:
        q = mk() * A.C_LOG2
        raw = [F.to_bfp16(F.a_layout(rows(q, h, i), 64, 128)) for h in range(heads) for i in range(t)]
        return tt(np.concatenate(raw), torch.uint8), F.quantize_rows(q.reshape(-1, 128)).reshape(q.shape)
    k, v = mk(), mk()
    raw = []
    for h in range(heads):
        for i in range(t):
            raw += [F.to_bfp16(F.b_layout(np.ascontiguousarray(rows(k, h, i).T), 128, 64)),
                    F.to_bfp16(F.b_layout(rows(v, h, i), 64, 128))]
    vq = F.quantize_rows(np.ascontiguousarray(v.transpose(0, 2, 1)).reshape(-1, 64 * t)).reshape(heads, 128, 64 * t)
    return tt(np.concatenate(raw), torch.uint8), (F.quantize_rows(k.reshape(-1, 128)).reshape(k.shape),
                                                  np.ascontiguousarray(vq.transpose(0, 2, 1)))


@pytest.mark.parametrize("hq,hkv,qa,q0,qn,nq,kv", [
    (2, 2, 2, 0, 2, 128, [(3, 0, 3)]), (3, 1, 5, 1, 3, 256, [(4, 2, 1), (7, 3, 4)]), (1, 2, 1, 0, 1, 128, [(1, 0, 1)])])
def test_attn_tiles(dev, hq, hkv, qa, q0, qn, nq, kv):
    """Tile ranges of one or two K / V buffers, query rows past the range: the exact values."""
    rng = np.random.default_rng(hq + nq)
    qb, qv = tiles(rng, hq, qa)
    bufs = [tiles(rng, hkv, t, kv=True) for t, _, _ in kv]
    q, k, vt = ops.attn_tiles(qb, hq, qa, q0, qn, nq, [(b[0], *g) for b, g in zip(bufs, kv)], hkv)
    ref_q = np.zeros((hq, nq, 128), np.float32)
    ref_q[:, :64 * qn] = qv[:, 64 * q0:64 * (q0 + qn)]
    cut = lambda x, g: x[:, 64 * g[1]:64 * (g[1] + g[2])]
    np.testing.assert_array_equal(q.float().cpu().numpy(), ref_q)
    np.testing.assert_array_equal(k.float().cpu().numpy(), np.concatenate([cut(b[1][0], g) for b, g in zip(bufs, kv)], 1))
    np.testing.assert_array_equal(vt.float().cpu().numpy().transpose(0, 2, 1),
                                  np.concatenate([cut(b[1][1], g) for b, g in zip(bufs, kv)], 1))


def check_o(got, ref):
    """Packed O against float64: 1e-2 of the largest value (P in bf16, O in bfp16), correlation above 0.9999."""
    assert G.rel_err(got, ref) <= 1e-2 and G.corr(got, ref) > 0.9999


@pytest.mark.parametrize("H,OH,H0,nqt,nk,pad", [(2, 2, 0, 4, 5, 13), (1, 3, 1, 2, 33, 64), (3, 4, 1, 6, 2, 0),
                                                (65, 65, 0, 16, 2, 1)])
def test_attn_artifact(dev, H, OH, H0, nqt, nk, pad):
    """Whole tasks and tasks split along the keys, 4- and 8-wave workgroups, an O wider than the heads, padded keys (a
    whole tile of them too): against float64 and against the general form; other columns of O stay."""
    rng = np.random.default_rng(H + nk)
    qb, qv = tiles(rng, H, nqt)
    kb, (kd, vd) = tiles(rng, H, nk, kv=True)
    meta = {"family": "attn32o", "H": H, "QN": nqt, "NK": 64 * nk, "NKV": 64 * nk - pad, "OA": 1, "OHEADS": OH, "H0": H0}
    M = 64 * nqt
    o = torch.full((M * OH * 128 // 8 * 9,), 5, dtype=torch.uint8, device="cuda")
    run_attn.run_artifact(meta, [qb, kb, o])
    full = layouts.from_bfp16_a_layout(o, M, OH * 128)
    got = full.cpu().numpy().reshape(M, OH, 128).transpose(1, 0, 2)
    hs = list(range(H)) if H < 8 else [0, 31, 64]
    check_o(got[[H0 + h for h in hs]], A.attention_ref(qv[hs], kd[hs], vd[hs], nkv=64 * nk - pad))
    rest = torch.full_like(o, 5)
    untouched = layouts.from_bfp16_a_layout(rest, M, OH * 128).reshape(M, OH, 128)
    keep = [h for h in range(OH) if not H0 <= h < H0 + H]
    assert torch.equal(full.reshape(M, OH, 128)[:, keep], untouched[:, keep])
    # the general form re-encodes bf16 values, which only blocks led by -128 change
    q, k, vt = ops.attn_tiles(qb, H, nqt, 0, nqt, M, [(kb, nk, 0, nk)], H)
    o16 = ops.attention(q, k, vt, nkv=64 * nk - pad, quantize_out=True)
    same = full.reshape(M, OH * 128)[:, H0 * 128:(H0 + H) * 128] == o16.float()
    assert same.all()


@pytest.mark.parametrize("hq,hkv,M,nqt", [(4, 2, 256, 3), (8, 1, 512, 8), (32, 8, 1536, 17), (64, 64, 1280, 20)])
def test_causal_artifact(dev, hq, hkv, M, nqt):
    """Grouped-query heads, an odd number of query tiles, rows past them left alone, more tasks than workgroups."""
    rng = np.random.default_rng(hq + nqt)
    T, n = M // 64, 64 * nqt
    qb, qv = tiles(rng, hq, T)
    kb, (kd, vd) = tiles(rng, hkv, T, kv=True)
    o = torch.full((M * hq * 128 // 8 * 9,), 5, dtype=torch.uint8, device="cuda")
    run_attn.run_artifact({"family": "causal", "M": M, "NQT": nqt}, [qb, kb, o])
    full = layouts.from_bfp16_a_layout(o, M, hq * 128)
    got = full.cpu().numpy().reshape(M, hq, 128).transpose(1, 0, 2)
    g = hq // hkv
    for h in (0, hq // 2, hq - 1):
        ref = A.attention_ref(qv[h:h + 1, :n], kd[h // g:h // g + 1, :n], vd[h // g:h // g + 1, :n], lim=np.arange(n))
        check_o(got[h:h + 1, :n], ref)
        # query 0 sees key 0 only: O is that V row (blocks of 8 keys) rounded to blocks of 8 dims
        np.testing.assert_array_equal(got[h, :1], F.quantize_rows(vd[h // g, :1]))
    keep = layouts.from_bfp16_a_layout(torch.full_like(o, 5), M, hq * 128)
    assert torch.equal(full[n:], keep[n:])


@pytest.mark.parametrize("H,NQ,NK,split", [(2, 256, 1024, True), (3, 384, 640, False), (300, 256, 128, True)])
def test_limits_clip(dev, H, NQ, NK, split):
    """Limits that let a workgroup skip key blocks (sorted, and below zero: a query that sees nothing gives 0)."""
    rng = np.random.default_rng(H)
    mk = lambda n: F.bf16_round(rng.standard_normal((H, n, 128)).astype(np.float32))
    q, k, v = F.bf16_round(mk(NQ) * np.float32(A.C_LOG2)), mk(NK), mk(NK)
    lim = np.sort(rng.integers(-40, NK, NQ)).astype(np.int32)
    lim[:130] = -1
    o = ops.attention(tt(q, torch.bfloat16), tt(k, torch.bfloat16),
                      tt(v.transpose(0, 2, 1), torch.bfloat16), nkv=NK - 7, lim=tt(lim, torch.int32), split=split)
    got = o.float().cpu().numpy().reshape(NQ, H, 128).transpose(1, 0, 2)
    assert (got[:, :130] == 0).all()
    hs = [0, H // 2, H - 1]
    check_o(got[hs], A.attention_ref(q[hs], k[hs], v[hs], nkv=NK - 7, lim=lim))


# ---- QKV post on the C stream and the rotary table ----------------------------------------------------------------

@pytest.mark.parametrize("M,hq,hkv", [(512, 8, 8), (1024, 4, 2), (512, 6, 1), (1536, 32, 8)])
@pytest.mark.parametrize("packed", [True, False])
def test_qkv_stream(dev, monkeypatch, M, hq, hkv, packed):
    """The tiles equal those of the general form (C and the table to row-major order, then rl_qkv_post) byte for byte:
    the same float32 arithmetic on the same values; blocks of zeros and of extreme exponents among them."""
    rng = np.random.default_rng(M + hq)
    n = 128 * (hq + 2 * hkv)
    C = (rng.standard_normal((M, n)) * 2).astype(np.float32)
    C[64:80] = 0.0
    C[100:108] *= np.float32(2.0 ** -124)
    C[200:208, ::3] *= np.float32(2.0 ** 60)
    cin = ops.quantize(tt(C), order="c_atb")[0] if packed else layouts.c_layout_atb_values(tt(C, torch.bfloat16))
    ang = tt(rng.uniform(-np.pi, np.pi, (M, 64)))
    w = tt(1 + 0.1 * rng.standard_normal((2, 128)))
    tabs = run_qkv.qkv_tables(torch.cos(ang), torch.sin(ang), w[0] * float(A.C_LOG2), w[1]).reshape(-1)
    outs = []
    for general in (False, True):
        q = torch.full((hq * (M // 64) * 9216,), 3, dtype=torch.uint8, device="cuda")
        kv = torch.full((hkv * (M // 64) * 2 * 9216,), 3, dtype=torch.uint8, device="cuda")
        assert run_qkv._stream_form(cin, tabs, q, kv, M, M // 64, hq, hkv)
        if general:
            monkeypatch.setattr(run_qkv, "_stream_form", lambda *a: False)
        run_qkv.qkv_post_run("glue", cin, tabs, q, kv)
        outs.append((q, kv))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("M,D,rows,dtype", [(512, 1024, 512, torch.float32), (1024, 3072, 777, torch.bfloat16),
                                            (512, 8192, 1, torch.float32), (512, 2048, 0, torch.bfloat16)])
def test_stream_pack(dev, M, D, rows, dtype):
    """Both directions, with and without a column order, short inputs padded with zero rows: the exact values."""
    rng = np.random.default_rng(M + rows)
    x = rng.standard_normal((rows, D)).astype(np.float32)
    perm = rng.permutation(D)
    xb = np.zeros((M, D), np.float32)
    xb[:rows] = F.bf16_round(x) if rows else x
    for p in (None, perm):
        pt = None if p is None else tt(p, torch.int64)
        s = ops.stream_pack(tt(x, dtype), M, D, perm=pt)
        want = F.c_layout_atb(xb if p is None else np.ascontiguousarray(xb[:, p]))
        np.testing.assert_array_equal(s.float().cpu().numpy(), want)
        for dt in (torch.float32, torch.bfloat16):
            back = ops.stream_unpack(s, M, D, perm=pt, dtype=dt)
            assert back.dtype == dt
            np.testing.assert_array_equal(back.float().cpu().numpy(), xb)
    b = layouts.c_layout_atb_values(tt(xb, torch.bfloat16))
    np.testing.assert_array_equal(b.float().cpu().numpy(), F.c_layout_atb(xb))
    assert torch.equal(b.float(), layouts.c_layout_atb_values(tt(xb)))
    assert torch.equal(layouts.c_unlayout_atb_values(b, M, D).float(), layouts.c_unlayout_atb_values(b.float(), M, D))


@pytest.mark.parametrize("H,N", [(24, 4352), (24, 1152)])
def test_attention_deterministic_on_cold_caches(dev, H, N):
    """The same bits on every launch, with K, V and Q pushed out of the caches before each: the waves of a workgroup then
    run far apart, and a key block that is overwritten before all of them have read it shows."""
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn((H, N, 128), generator=g, device="cuda").bfloat16() for _ in range(3))
    vt = v.transpose(1, 2).contiguous()
    q = q * float(A.C_LOG2)
    big = torch.zeros(1 << 28, dtype=torch.uint8, device="cuda")
    ref = ops.attention(q, k, vt, split=False)
    for i in range(12):
        big.add_(1)
        assert torch.equal(ops.attention(q, k, vt, split=False), ref), i


@pytest.mark.parametrize("M,D,branch,packed", [(6600, 3072, "none", False), (3300, 3072, "bf16", True),
                                               (4300, 3008, "packed", False), (3250, 4096, "packed", True),
                                               (2600, 4096, "bf16", False), (1300, 8192, "bf16", True),
                                               (1650, 8192, "packed", False)])
def test_ln_x_past_the_caches(dev, M, D, branch, packed):
    """x' stored past the caches (more than 40 MB read): the same bits as from two halves, which are below that line and
    store it through the caches."""
    g = torch.Generator(device=dev).manual_seed(M + D)
    x, b = (torch.randn(M, D, device=dev, generator=g).to(torch.bfloat16) for _ in range(2))
    params = torch.randn(2, 2 * D, device=dev, generator=g).to(torch.bfloat16)
    br = lambda r: {"none": None, "bf16": b[r], "packed": ops.quantize(b[r].contiguous())[0]}[branch]
    run = lambda r: ops.ln_modulate(x[r], params, branch=br(r), norm="layer", packed=packed, deq=True)
    whole, h = run(slice(0, M)), M // 2
    lo, hi = run(slice(0, h)), run(slice(h, M))
    assert torch.equal(whole[0], torch.cat([lo[0], hi[0]]))
    assert torch.equal(whole[2], torch.cat([lo[2], hi[2]]))
    if packed:
        assert torch.equal(whole[1].reshape(-1), torch.cat([lo[1].reshape(-1), hi[1].reshape(-1)]))
