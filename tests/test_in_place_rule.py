"""Which tensors a kernel may work on in place of torch operations: not those whose operations something records."""

import numpy as np
import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode

from oracle import bfp16 as F
from rlbfp import layouts, ops, vlm_run


def test_plain():
    t = torch.zeros(8)
    seen = []
    assert ops.plain(t)
    assert not ops.plain(t.clone().requires_grad_()) and not ops.plain(torch.nn.Parameter(t))
    see = lambda x: (seen.append(ops.plain(x)), x * 2)[1]
    torch.vmap(see)(torch.zeros(2, 8))
    torch.func.jvp(see, (t,), (t,))
    with torch.autograd.forward_ad.dual_level():
        see(torch.autograd.forward_ad.make_dual(t, t))
    torch.jit.trace(see, t, check_trace=False)
    with FlopCounterMode(display=False):
        see(t)
    assert len(seen) >= 5 and not any(seen)
    assert ops.plain(t)


def test_load_x_without_a_gpu_buffer():
    """A channel order that is not on the GPU goes through torch operations."""
    m, d, rows = 512, 1024, 77
    rng = np.random.default_rng(0)
    lm = object.__new__(vlm_run.LM)
    hp = rng.permutation(d)
    lm.m, lm.d, lm.hp, lm.hp_kernel, lm.x, lm.br_zero = m, d, torch.from_numpy(hp), True, [None] * 3, None
    x = F.bf16_round(rng.standard_normal((rows, d)).astype(np.float32))
    lm.load_x(x)
    want = np.zeros((m, d), np.float32)
    want[:rows] = x[:, hp]
    np.testing.assert_array_equal(lm.x[0].float().numpy(), F.c_layout_atb(want))


@pytest.mark.gpu
def test_layout_gradients(dev):
    """The C-stream layouts of a tensor that needs gradients, and under vmap: as the same values in float32 give them."""
    M, N = 512, 1024
    x = torch.randn(M, N, device=dev).to(torch.bfloat16)
    w = torch.randn(M * N, device=dev).to(torch.bfloat16)
    for f, a in ((layouts.c_layout_atb_values, x), (lambda s: layouts.c_unlayout_atb_values(s, M, N), x.reshape(-1))):
        grads = []
        for dt in (torch.bfloat16, torch.float32):
            leaf = a.detach().to(dt).requires_grad_()
            y = f(leaf)
            (y.reshape(-1) * w.to(dt)).sum().backward()
            grads.append(leaf.grad.float())
        assert torch.equal(*grads)
    both = torch.stack([x, -x])
    assert torch.equal(torch.vmap(layouts.c_layout_atb_values)(both)[1], layouts.c_layout_atb_values(-x))
