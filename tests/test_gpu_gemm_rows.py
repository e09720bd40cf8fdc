"""The few-row GEMM kernels (M <= 128: one 128-column tile per workgroup, and the register-only kernel of short K)
against the emulation with every epilogue, at the edges of their row fragments, column sets and K pieces; whole-K calls
bit for bit against the same rows inside a taller GEMM, which runs the 4- or 8-wave kernels."""

import numpy as np
import pytest
import torch

from oracle import bfp16 as F
from oracle import gemm as G
from rlbfp import ops

pytestmark = pytest.mark.gpu


def t(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dtype)


def case(M, K, N, act, seed):
    rng = np.random.default_rng(seed)
    if act == "swiglu":
        packed = F.pack_b(F.interleave_up(G.linear_weight(rng, N // 2, K), G.linear_weight(rng, N // 2, K)))
    else:
        packed = F.pack_b(G.linear_weight(rng, N, K).T)
    return rng, F.quantize_rows(G.activations(rng, M, K)), packed


EPILOGUES = ["none", "bias", "gelu_tanh", "swiglu", "swiglu_bias_q", "gate"]
CODE = {"gelu_tanh": G.ACT_GELU_TANH, "swiglu": G.ACT_SWIGLU, None: G.ACT_NONE}


@pytest.mark.parametrize("ep", EPILOGUES)
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("M,K,N", [
    (1, 1024, 256), (17, 1088, 384), (16, 8192, 128), (33, 2048, 1024), (48, 4096, 512), (64, 1984, 640),
    (64, 2048, 4224), (65, 4096, 256), (81, 1536, 1152), (97, 6144, 256), (128, 4160, 384), (5, 512, 8448),
    (40, 64, 256), (113, 192, 128), (20, 1024, 17408)])
def test_few_rows(dev, M, K, N, split, ep):
    act = "gelu_tanh" if ep == "gelu_tanh" else "swiglu" if ep.startswith("swiglu") else None
    rng, Aq, packed = case(M, K, N, act, M + K + N)
    nout = N // 2 if act == "swiglu" else N
    kw, ref = {"act": act}, {"act": CODE[act]}
    if ep in ("bias", "gelu_tanh", "swiglu_bias_q"):
        bias = (rng.standard_normal(N) * 0.3).astype(np.float32)
        kw["bias"], ref["bias"] = t(bias), bias
    if ep == "swiglu_bias_q":
        kw["quantize_out"] = ref["quantize_out"] = True
    if ep == "gate":
        gate = rng.standard_normal((2, nout)).astype(np.float32)
        res = F.bf16_round(rng.standard_normal((M, nout)).astype(np.float32))
        kw.update(gate=t(gate), gate_split_row=M // 2, residual=t(res, torch.bfloat16))
        ref.update(gate=gate, gate_split_row=M // 2, residual=res)
    a, b = t(Aq, torch.bfloat16), t(packed, torch.uint8)
    out = torch.full((M + 1, nout), 7.0, dtype=torch.bfloat16, device="cuda")
    got = ops.gemm(a, b, N, K, split=split, out=out[:M], **kw)
    assert (out[M] == 7.0).all()                       # nothing past the last row
    want = G.gemm_ref(Aq, F.decode_b(packed, K, N), **ref)
    g = got.float().cpu().numpy()
    # a re-quantized value at a tie of its block may take either side: one step of 2^-6 of the block's largest value
    assert G.rel_err(g, want) <= (2e-2 if ep == "swiglu_bias_q" else 1e-2)
    if ep != "swiglu_bias_q":
        d = np.abs(g.astype(np.float64) - want)
        assert (d <= 2 * np.abs(want) * 2.0 ** -8 + 1e-5 * np.abs(want).max()).mean() > 0.999
    if not split:
        # the same rows among 300 (the rows beyond repeat them)
        rows = np.arange(300) % M
        tall = dict(kw)
        if ep == "gate":
            tall.update(residual=t(res[rows], torch.bfloat16))
        assert torch.equal(got, ops.gemm(t(Aq[rows], torch.bfloat16), b, N, K, split=False, **tall)[:M])


@pytest.mark.parametrize("act", [None, "swiglu"])
def test_few_rows_packed_out(dev, act):
    """A packed output of 128 rows: the pieces run here, the reduce launch writes the blocks."""
    M, K, N = 128, 8192, 1024
    rng, Aq, packed = case(M, K, N, act, 3)
    assert ops.gemm_workspace_bytes(M, N, K) > 0
    a, b = t(Aq, torch.bfloat16), t(packed, torch.uint8)
    nout = N // 2 if act else N
    pk = torch.empty(M * nout // 8 * 9, dtype=torch.uint8, device="cuda")
    ops.gemm(a, b, N, K, act=act, packed_out=pk, packed_order="a_layout")
    y = ops.gemm(a, b, N, K, act=act)
    assert torch.equal(pk, ops.quantize(y, order="a_layout")[0])


def test_few_rows_strided_a(dev):
    """A with a row stride above K, and a C with one above N."""
    M, K, N = 70, 4096, 256
    rng, Aq, packed = case(M, K, N, None, 8)
    wide = torch.full((M, K + 72), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, :K] = t(Aq, torch.bfloat16)
    for rows in (M, 9):
        c = torch.full((rows, N + 16), 3.0, dtype=torch.bfloat16, device="cuda")
        for split in (True, False):
            ops.gemm(wide[:rows, :K], t(packed, torch.uint8), N, K, split=split, out=c[:, :N])
            assert G.rel_err(c[:, :N].float().cpu().numpy(), G.gemm_ref(Aq[:rows], F.decode_b(packed, K, N))) <= 1e-2
            assert (c[:, N:] == 3.0).all()
