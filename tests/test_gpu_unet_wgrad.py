"""The predictor's backward pass against a 64-bit restatement with the same BF16 rounding points, from the
engine's own activations, on grids where the weight gradient's split can go wrong: rows of one, two and a
broken number of 8-point blocks on the three levels (extents 8 to 36, so 2 to 9 points per row on the
coarsest), every layer and tap by itself.

Bound: given the activations, the two sides differ by FP32 summation (about 1e-6) and by the BF16
gradients that this flips by one unit (2^-8 relative, on about 1 value in 1000), at most ten layers deep:
sqrt(1e-3) 2^-8 sqrt(10) = 4e-4 of a layer's norm, more on single taps; 5e-3 is allowed (measured: 1e-7
at the last layer to 3e-3 on the worst tap of the first).  A wrong neighbour, a lost block of
points or a padding value that counts changes a tap by 10% or more at these sizes."""
import numpy as np
import pytest
import torch

from tests import unet_ref

pytestmark = pytest.mark.gpu

TAPS = [(z, y, x) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
# act index of each conv layer's output and of its inputs (-1: the packed input)
OUT = [0, 1, 3, 4, 6, 7, 8, 9, 10, 11]
SRC = [(-1, None), (0, None), (2, None), (3, None), (5, None), (6, None), (7, 4), (8, None), (9, 1), (10, None)]


def bf(t):
    return t.float().to(torch.bfloat16).double()


def up(t):
    return t.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)


def pool_sum(t):
    a, b, c, m = t.shape
    return t.reshape(a // 2, 2, b // 2, 2, c // 2, 2, m).sum(dim=(1, 3, 5))


def backward(w, acts, out, target, shape):
    """Flat parameter gradient from the activations {index: (z, y, x, c) float64}."""
    layers, off = [], 0
    for co, c1, c2, u, lv in unet_ref.SPEC:
        n = 27 * co * (c1 + c2)
        layers.append((w[off : off + n].reshape(27, co, c1 + c2), off))
        off += n + co
    head = w[off : off + 17]
    grad = torch.zeros(w.numel(), dtype=torch.float64)
    dout = (2.0 * (out.float() - target.float()) / out.numel()).double().reshape(shape)
    grad[off : off + 16] = torch.einsum("zyx,zyxc->c", dout, acts[11])
    grad[off + 16] = dout.sum()
    g = bf(dout[..., None] * head[:16] * (acts[11] > 0))
    skip = {}
    for li in range(9, -1, -1):
        co, c1, c2, u, lv = unet_ref.SPEC[li]
        W, o = layers[li]
        W = bf(W)
        s1, s2 = SRC[li]
        x = up(acts[s1]) if u else acts[s1]
        if s2 is not None:
            x = torch.cat([x, acts[s2]], 3)
        ci = c1 + c2
        fx = torch.zeros(x.shape, dtype=torch.float64)
        for t, d in enumerate(TAPS):
            xs = torch.roll(x, (-d[0], -d[1], -d[2]), (0, 1, 2)).reshape(-1, ci)
            grad[o + t * co * ci : o + (t + 1) * co * ci] = (g.reshape(-1, co).T @ xs).reshape(-1)
            fx += torch.roll(g, d, (0, 1, 2)) @ W[t]
        grad[o + 27 * co * ci : o + 27 * co * ci + co] = g.reshape(-1, co).sum(0)
        if li == 0:
            break
        if u:  # [up(coarse), skip]
            skip[li] = fx[..., c1:]
            g = bf(pool_sum(fx[..., :c1]) * (acts[s1] > 0))
        elif li in (2, 4):  # through the pool, plus the skip part
            k, dst = (8, 1) if li == 2 else (6, 4)
            g = bf((up(fx) / 8.0 + skip[k]) * (acts[dst] > 0))
        else:
            g = bf(fx * (acts[OUT[li - 1]] > 0))
    return grad


@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 12, 20), (12, 8, 28), (16, 20, 32), (12, 16, 36), (36, 8, 12)])
def test_backward(shape):
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    from salmon2_amd.unet import UNet

    nz, ny, nx = shape
    print(f"[gpu] unet backward {nx}x{ny}x{nz}", flush=True)
    net = UNet(nx, ny, nz, seed=5, stream=torch.cuda.current_stream())
    rng = np.random.default_rng(11)
    n = nx * ny * nz
    x = torch.from_numpy(rng.standard_normal((n, 4)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
    out = torch.zeros(n, dtype=torch.float32, device="cuda")
    net.forward(x, out)
    for _ in range(2):  # gradients add up over samples
        net.train_sample(x, t)
    torch.cuda.synchronize()
    got = torch.from_numpy(net.get_grads()).double() / 2
    acts = {}
    for i in range(-1, 12):
        lv = 0 if i < 0 else UNet.ACT_SHAPES[i][1]
        acts[i] = torch.from_numpy(net.activation(i)).double().reshape(nz >> lv, ny >> lv, nx >> lv, -1)
    w = torch.from_numpy(net.get_params()).double()
    ref = backward(w, acts, out.cpu(), t.cpu(), shape)
    off, worst = 0, 0.0
    for co, c1, c2, u, lv in unet_ref.SPEC:
        for m in 27 * [co * (c1 + c2)] + [co]:
            a, b = got[off : off + m], ref[off : off + m]
            worst = max(worst, float((a - b).norm() / b.norm()))
            off += m
    worst = max(worst, float((got[off:] - ref[off:]).norm() / ref[off:].norm()))
    print(f"[parity] unet backward {shape}: worst layer and tap {worst:.2e}", flush=True)
    assert worst <= 5e-3
    net.close()
