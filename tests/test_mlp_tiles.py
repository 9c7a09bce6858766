"""Row counts at the edges of the warm-start MLP kernels against the CPU
restatement in oracle/mlp_oracle.py: one row, one short of a 16-row tile, a full
tile and one more, a full 32-row chunk and one more, one more than the 16 x 32
rows one pass of the weight-gradient waves covers and than the four passes they
load at a time, and more 16-row tiles than the forward grid has workgroups; the
fused Adam launch against one launch per tensor, and the largest tensors Adam takes.

Tolerances as in test_mlp.py: gradients from the kernel's own trace within 2e-3
of their scale (BF16 operands), activations within one BF16 rounding.
"""

import ctypes as ct

import numpy as np
import pytest

from test_mlp import mo, random_params


def _model(p, torch):
    from metalrobo import warmstart as ws

    m = ws.WarmStartMLP(seed=0)
    m.load_state({k: np.asarray(v) for k, v in p.items()})
    return m


def _close(got, ref, rel):
    scale = max(np.abs(ref).max(), 1e-12)
    assert np.abs(got - ref).max() <= rel * scale, np.abs(got - ref).max() / scale


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 513, 2049, 512 * 16 + 5])
def test_forward_and_gradients_at_tile_edges(gpu, n):
    import torch

    p = random_params(21)
    rng = np.random.default_rng(n)
    x = (2.0 * rng.standard_normal((n, 8))).astype(np.float32)
    t = rng.standard_normal((n, 3)).astype(np.float32)
    m = _model(p, torch)
    xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    y0 = m.forward(xd).clone()
    _, g = m.loss_and_grads(xd, td)
    torch.cuda.synchronize()
    b = m._bufs
    assert torch.equal(y0, b["y"])
    ref = mo.forward(p, x)
    for k in ("z1", "z2"):
        _close(b[k].cpu().numpy(), ref[k], 2e-3)
    _close(y0.cpu().numpy(), ref["y_hat"], 2e-3)
    tr = {k: b[k].float().cpu().numpy().astype(np.float64) for k in ("xq", "z1", "h1", "z2", "h2")}
    ref_g, ref_dz2, ref_dz1 = mo.backward(p, tr, b["dy"].cpu().numpy().astype(np.float64))
    _close(b["dz2"].cpu().numpy(), ref_dz2, 2e-3)
    _close(b["dz1"].cpu().numpy(), ref_dz1, 2e-3)
    for k in ("w1", "b1", "w2", "b2", "w3", "b3"):
        _close(g[k].cpu().numpy(), ref_g[k], 2e-3)


@pytest.mark.gpu
def test_adam_on_many_tensors_equals_one_at_a_time(gpu):
    """Nine tensors (two launches) with lengths around the 256 values of a workgroup."""
    import torch
    from metalrobo import native as nat

    b = nat.load()
    gen = torch.Generator().manual_seed(3)
    lengths = (1, 255, 256, 257, 3, 1000, 64, 512, 513)
    base = [[torch.rand(n, generator=gen).cuda() for _ in range(4)] for n in lengths]
    one = [[v.clone() for v in q] for q in base]
    many = [[v.clone() for v in q] for q in base]
    half = [[torch.zeros(n, dtype=torch.bfloat16, device="cuda") for n in lengths] for _ in range(2)]
    p = lambda v: ct.c_void_p(v.data_ptr())
    hyper = (1e-3, 0.9, 0.999, 1e-8, 3, None)
    tensors = (nat.MlpAdamTensorC * len(lengths))()
    for k, n in enumerate(lengths):
        w, g, m1, m2 = one[k]
        b.check(b.lib.mr_mlp_adam(p(w), p(half[0][k]), p(g), p(m1), p(m2), n, *hyper))
        w, g, m1, m2 = many[k]
        tensors[k] = nat.MlpAdamTensorC(w.data_ptr(), half[1][k].data_ptr(), g.data_ptr(), m1.data_ptr(),
                                        m2.data_ptr(), n, 0)
    b.check(b.lib.mr_mlp_adam_tensors(tensors, len(lengths), *hyper))
    torch.cuda.synchronize()
    for k in range(len(lengths)):
        assert torch.equal(half[0][k], half[1][k])
        assert all(torch.equal(u, v) for u, v in zip(one[k], many[k])), lengths[k]
        assert not torch.equal(many[k][0], base[k][0])


@pytest.mark.parametrize("count", [2**31 - 1, 2**31, 2**31 + 1, 2**32 - 1])
def test_adam_takes_every_count(count):
    """A learning rate out of range is refused after the counts have been accepted; nothing is launched."""
    from metalrobo import native as nat

    b = nat.load()
    p = ct.c_void_p(64)
    with pytest.raises(nat.MetalRoboError, match="hyper-parameters"):
        b.check(b.lib.mr_mlp_adam(p, None, p, p, p, count, -1.0, 0.9, 0.999, 1e-8, 1, None))
    with pytest.raises(nat.MetalRoboError, match="count and step"):
        b.check(b.lib.mr_mlp_adam(p, None, p, p, p, count, 1e-3, 0.9, 0.999, 1e-8, 0, None))


@pytest.mark.gpu
def test_adam_on_more_than_2_to_the_31_values(gpu):
    """One tensor in two parts: values on both sides of the joint, and the last ones, as in a tensor of their own."""
    import torch
    from metalrobo import native as nat

    n = 2**31 + 300
    if torch.cuda.mem_get_info()[0] < 6 * 4 * n:
        pytest.skip("needs 52 GB of device memory")
    b = nat.load()
    at = torch.tensor([0, 255, 256, 2**31 - 1, 2**31, 2**31 + 255, 2**31 + 256, n - 1], device="cuda")
    gen = torch.Generator().manual_seed(4)
    small = [torch.rand(len(at), generator=gen).cuda() for _ in range(4)]
    half = [torch.zeros(k, dtype=torch.bfloat16, device="cuda") for k in (len(at), n)]
    large = [torch.zeros(n, device="cuda") for _ in range(4)]
    for u, v in zip(large, small):
        u[at] = v
    p = lambda v: ct.c_void_p(v.data_ptr())  # noqa: E731
    print("adam on", n, "values", flush=True)
    for (w, g, m1, m2), h in ((small, half[0]), (large, half[1])):
        b.check(b.lib.mr_mlp_adam(p(w), p(h), p(g), p(m1), p(m2), w.numel(), 1e-3, 0.9, 0.999, 1e-8, 2, None))
    torch.cuda.synchronize()
    assert torch.equal(half[1][at], half[0]) and half[0].count_nonzero() == len(at)
    assert all(torch.equal(u[at], v) for u, v in zip(large, small))
