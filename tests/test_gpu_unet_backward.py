"""The backward convolutions at FP32 precision: a network whose activations are
small integers, exact in BF16 (two weights of +-1 per output channel, the
prolonged inputs unused), so that the gradients are FP32 sums alone and have
to agree with an FP64 reference to FP32 rounding (sums of up to 1e5 terms;
6e-8 sqrt(1e5) = 2e-5 bounds their relative error), layer by layer.  Grids
below and above the 32768-node switch, no dimension a multiple of a tile."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import serac_amd as sx

pytestmark = pytest.mark.gpu


def integer_weights(rng):
    parts = []
    for ca, cb, co in sx.UNet.LAYERS:
        w = np.zeros((27, ca + cb, co), dtype=np.float32)
        for c in range(co):
            first = ca if cb else 0  # decoder layers read their skip
            for _ in range(2):
                w[rng.integers(27), rng.integers(first, ca + cb), c] = rng.choice([-1.0, 1.0])
        parts += [w.ravel(), np.zeros(co, dtype=np.float32)]
    return np.concatenate(parts)


def reference_gradients(p, x, t, dims, relu):
    leaf = torch.tensor(p, dtype=torch.float64, requires_grad=True)
    act = torch.relu if relu else (lambda v: v)
    ws, off = [], 0
    for ca, cb, co in sx.UNet.LAYERS:
        n = 27 * (ca + cb) * co
        ws.append((leaf[off:off + n].reshape(3, 3, 3, ca + cb, co).permute(4, 3, 0, 1, 2), leaf[off + n:off + n + co]))
        off += n + co

    def conv(v, k, stride=1):
        return F.conv3d(v, ws[k][0], ws[k][1], stride=stride, padding=1)

    def up(v, like):
        return F.interpolate(v, size=like.shape[2:], mode="trilinear", align_corners=True)

    def vol(a):
        return torch.tensor(a.reshape(dims[2], dims[1], dims[0], 3).transpose(3, 0, 1, 2)[None], dtype=torch.float64)

    b0 = act(conv(act(conv(vol(x), 0)), 1))
    b1 = act(conv(act(conv(b0, 2, 2)), 3))
    b2 = act(conv(act(conv(b1, 4, 2)), 5))
    b3 = act(conv(act(conv(b2, 6, 2)), 7))
    c2 = act(conv(torch.cat([up(b3, b2), b2], 1), 8))
    c1 = act(conv(torch.cat([up(c2, b1), b1], 1), 9))
    c0 = act(conv(torch.cat([up(c1, b0), b0], 1), 10))
    loss = (conv(c0, 11) - vol(t)).square().sum() / vol(t).square().sum()
    loss.backward()
    return leaf.grad.numpy()


@pytest.mark.parametrize("dims", [(9, 9, 9), (17, 9, 25), (41, 33, 33)])
@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("mfma", [True, False])
def test_gradients_at_fp32_precision(gpu_lib, dims, relu, mfma):
    rng = np.random.default_rng(7)
    net = sx.UNet(*dims, seed=1)
    if not relu:
        net.set_activation(sx.capi.SX_UNET_IDENTITY, seed=1)
    net.set_mfma(mfma)
    p = integer_weights(rng)
    net.set_params(p)
    x = rng.integers(-1, 2, (net.nvox, 3)).astype(np.float32)
    t = rng.standard_normal((net.nvox, 3)).astype(np.float32)
    net.backward(x, t)
    g, ref = net.grads(), reference_gradients(p, x, t, dims, relu)
    off = 0
    for k, (ca, cb, co) in enumerate(sx.UNet.LAYERS):
        for n in (27 * (ca + cb) * co, co):
            a, b = g[off:off + n], ref[off:off + n]
            assert np.linalg.norm(a - b) <= 2e-5 * np.linalg.norm(b), (k, n)
            off += n


@pytest.mark.parametrize("mfma", [True, False])
@pytest.mark.parametrize("through", ["weights", "data"])
@pytest.mark.parametrize("g", [1e-33, 3e-20, 0.7, 3.39e38, 3.4e38])
def test_one_gradient_value_over_the_float_range(gpu_lib, mfma, through, g):
    """dL/dy is one number of FP32's range (the planes' sum is exact from 2^-110 up), everything else small powers of
    two or zero: the head's weight gradients are that number at its 27 taps, or half of it reaches the layer below."""
    dims = (9, 9, 9)
    net = sx.UNet(*dims, seed=1)
    net.set_activation(sx.capi.SX_UNET_IDENTITY, seed=1)
    net.set_mfma(mfma)
    offs = np.cumsum([0] + [n for ca, cb, co in sx.UNet.LAYERS for n in (27 * (ca + cb) * co, co)])
    p = np.zeros(net.nparam, dtype=np.float32)
    if through == "weights":
        p[offs[21]] = 1.0  # layer 10's bias, channel 0: the head's input is 1, its output 0
    else:
        p[offs[22] + (13 * 16) * 3 + 1] = -0.5  # the head's centre weight, channel 0 -> 1; its input is 0
    net.set_params(p)
    t = np.zeros((net.nvox, 3), dtype=np.float32)
    t[4 * 81 + 4 * 9 + 4, 1] = v = np.float32(2.0 / g)
    net.backward(np.zeros((net.nvox, 3), dtype=np.float32), t)
    want = np.float32(-np.float64(v) * (2.0 / (np.float64(v) * np.float64(v))))
    assert abs(want / g + 1.0) < 1e-5
    ref = np.zeros(net.nparam, dtype=np.float32)
    ref[offs[23] + 1] = want
    if through == "weights":
        ref[offs[22]:offs[23]].reshape(27, 16, 3)[:, 0, 1] = want
    else:
        ref[offs[21]] = np.float32(-0.5) * want
    assert np.array_equal(net.grads(), ref)


def test_work_memory_comes_with_the_first_matrix_core_backward(gpu_lib):
    """65^3 nodes: networks that are evaluated, or trained on the vector units, go without its 109 MB."""
    rng = np.random.default_rng(3)
    net = sx.UNet(65, 65, 65, seed=1)
    x = sx.DeviceVector.from_numpy(rng.standard_normal(net.nvox * 3), dtype=np.float32)
    t = sx.DeviceVector.from_numpy(rng.standard_normal(net.nvox * 3), dtype=np.float32)
    net.set_mfma(False)
    free = []
    for mfma in (False, True, True):
        net.set_mfma(mfma)
        net.forward(x)
        free.append(torch.cuda.mem_get_info()[0])
        net.backward(x, t)
        free.append(torch.cuda.mem_get_info()[0])
    assert abs(free[1] - free[0]) < 16 << 20 and abs(free[2] - free[1]) < 16 << 20
    assert free[2] - free[3] > 80 << 20
    assert abs(free[5] - free[3]) < 16 << 20
