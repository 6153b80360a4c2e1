'''A training step whose products and kernel gradients all run on the bf16 matrix cores, against the same step in 64 bits: its gradients are no
further off than through the fp32 kernels.'''
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import vkjax_amd
from vkjax_amd import kernels as K
from vkjax_amd import minijax as mj

lax, jnp, nn = mj.lax, mj.numpy, mj.nn
WEIGHTS = [(1, 1, 64, 96), (3, 3, 96, 64), (1, 1, 64, 128), (3, 3, 128, 64), (1, 1, 64, 128)]
STRIDES = (1, 1, 1, 2, 1)


def loss(weights, x, target):
    y = x
    for w, stride in zip(weights, STRIDES):
        pad = w.shape[0] // 2
        z = lax.conv_general_dilated(y, w, (stride, stride), ((pad, pad), (pad, pad)), dimension_numbers=('NHWC', 'HWIO', 'NHWC'))
        y = nn.relu(z + y) if z.shape == y.shape else nn.relu(z)
    d = y - target
    return jnp.mean(d * d)


def loss64(weights, x, target):
    y = x
    for w, stride in zip(weights, STRIDES):
        z = F.conv2d(y.permute(0, 3, 1, 2), w.permute(3, 2, 0, 1), stride=stride, padding=w.shape[0] // 2).permute(0, 2, 3, 1)
        y = F.relu(z + y) if z.shape == y.shape else F.relu(z)
    return ((y - target) ** 2).mean()


@pytest.mark.gpu
@pytest.mark.parametrize('seed', (0, 1))
def test_gradients_are_no_further_from_64_bits(seed):
    rng = np.random.RandomState(seed)
    weights = [(rng.standard_normal(s) * np.sqrt(2.0 / np.prod(s[:3]))).astype(np.float32) for s in WEIGHTS]
    x, target = rng.standard_normal((3, 15, 14, 64)).astype(np.float32), rng.standard_normal((3, 8, 7, 128)).astype(np.float32)
    w64   = [torch.tensor(w, dtype=torch.float64, requires_grad=True) for w in weights]
    value = loss64(w64, torch.tensor(x, dtype=torch.float64), torch.tensor(target, dtype=torch.float64))
    value.backward()
    exact = [w.grad.numpy() for w in w64]
    def step(**choice):
        with K.overrides(**choice):
            fn = vkjax_amd.wrap(mj.value_and_grad(loss), frontend='minijax')
            v, grads = fn(weights, x, target)
        kernels  = [l.kernel for l in list(fn._jaxpr_interpreters.values())[0].launches]
        products = [k for k in kernels if k.startswith(('conv_gemm', 'wgrad'))]
        assert abs(v - value.item()) <= 1e-5 * value.item()
        return products, np.sqrt(sum(np.sum((g - e) ** 2) for g, e in zip(grads, exact)) / sum(np.sum(e ** 2) for e in exact))
    products, fp32 = step(conv_split=False, wgrad_split=False)
    assert not any('split' in k for k in products)
    for tile, wgrad_tile in (('128x128', '128x128'), ('128x64', '64x64')):
        products, error = step(conv_split=tile, wgrad_split=wgrad_tile)
        print(f'seed {seed}, tiles {tile}, {wgrad_tile}: {error:.2e}, fp32 products {fp32:.2e}', flush=True)
        assert all('split' in k for k in products), products
        assert error <= fp32
