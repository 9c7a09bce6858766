"""The warm-start network's GELU and its derivative on the GPU, read out of the training
kernels: with one output weight of 1 and an output gradient of 1, dz2 is gelu'(z2) in FP32,
and the forward trace holds z beside the BF16 activation.

gelu'(x) = 0.5 (1 + erf) + x phi in FP32 is within 2.1e-7 of the exact value: erf's last two
places (1.2e-7) and the rounding of 1 + erf <= 2 (1.2e-7 / 2), both halved (0.9e-7); x phi <=
0.242 within four roundings (0.6e-7); the rounding of a result up to 1.13 (0.6e-7).

A saved network evaluates to the bits it was trained with, so the activations are the erf form
evaluated in that order, not merely a close value.
"""

import ctypes as ct

import numpy as np
import pytest

from test_mlp import mo, random_params


def points(count, seed):
    """Values over the range that the activations meet, the saturated ends and zero among them."""
    rng = np.random.default_rng(seed)
    x = np.concatenate([np.linspace(-12.0, 12.0, count // 2), rng.standard_normal(count - count // 2) * 2.0])
    x[:4] = (0.0, -0.0, 1.0e-30, -1.0e-30)
    return x.astype(np.float32)


@pytest.mark.gpu
def test_derivative_error_against_64_bits(gpu):
    import torch
    from metalrobo import native as nat
    from metalrobo import warmstart as ws

    n = 512
    m = ws.WarmStartMLP(seed=0)
    for t in (*m.master.values(), *m.bf16.values()):
        t.zero_()
    m.bf16["w3"][0] = 1.0
    z = points(n * 256, 1).reshape(n, 256)
    b = m._buffers(n)
    for k in ("xq", "h1", "h2", "z1"):
        b[k].zero_()
    b["z2"].copy_(torch.from_numpy(z))
    b["dy"].zero_()
    b["dy"][:, 0] = 1.0
    p = lambda t: ct.c_void_p(t.data_ptr())  # noqa: E731
    w, tr, g = m.weights(), m._trace(b), b["grads"]
    grads = nat.MlpGradsC(*(p(g[k]) for k in ("w1", "b1", "w2", "b2", "w3", "b3")))
    m._b.check(m._b.lib.mr_mlp_backward(ct.byref(w), ct.byref(tr), p(b["dy"]), n, p(b["dz2"]), p(b["dz1"]),
                                        ct.byref(grads), None))
    torch.cuda.synchronize()
    error = np.abs(b["dz2"].cpu().numpy().astype(np.float64) - mo.gelu_grad(z))
    assert error.max() <= 2.1e-7, (error.max(), z.reshape(-1)[error.argmax()])


@pytest.mark.gpu
def test_activations_are_the_erf_form_s_bits(gpu):
    import torch
    from test_mlp_tiles import _model

    x = (2.0 * np.random.default_rng(5).standard_normal((4000, 8))).astype(np.float32)
    m = _model(random_params(6), torch)
    m.forward(torch.from_numpy(x).cuda(), trace=True)
    torch.cuda.synchronize()
    for k in ("1", "2"):
        z = m._bufs["z" + k]
        expect = (0.5 * z * (1.0 + torch.erf(z * 0.7071067811865476))).to(torch.bfloat16)
        assert torch.equal(m._bufs["h" + k].view(torch.int16), expect.view(torch.int16)), k
