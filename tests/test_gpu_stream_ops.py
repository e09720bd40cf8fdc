"""The passes that work on the stream formats in place (C-stream order, A layout, attention tiles) against the oracle,
and against the general forms that first bring the operands to row-major order."""

import numpy as np
import pytest
import torch

from oracle import bfp16 as F
from oracle import gemm as G
from oracle import ln as LN
from rlbfp import forward, layouts, ops, run_ln

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
