"""The kernels that multiply fp32 operands as two terms of IEEE half (x3p_*, x3_win_*, x3w_*): the powers of two that bring inputs
and filters into a half's range, the second attempt with another one, and the results that are computed again in fp32."""
import numpy as np
import pytest
import torch

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph

pytestmark = pytest.mark.gpu

NAMES = [name for name in rt.conv_variant_names() if name.startswith(('x3p_', 'x3_win_', 'x3w_'))]
SHAPE, OC, BATCH = (35, 9, 11), 37, 3
FAN = SHAPE[0] * 9


@pytest.fixture(autouse=True)
def default_options():
    rt.set_option('autotune', 0)
    yield
    for key, value in (('autotune', 1), ('conv_variant', -1), ('conv_split_k', 0), ('split_k_reduce', 'xcd')):
        rt.set_option(key, value)


def network():
    ios.reset_name()
    holder = ios.placeholder(SHAPE)
    block = Block(holder.node, None, [], None)
    ios.conv2d(block, [[holder]], OC, (3, 3), (1, 1), (1, 1), act='identity', is_exit=True)
    graph = Graph('two', holder.node, [block])
    graph.init_weights(3, 'he_normal')
    graph.sequential_schedule()
    conv = list(graph.conv_nodes())[0]
    conv.bias = np.zeros(OC, np.float32)
    return graph, conv


def check(graph, conv, x, what, split, reduce='xcd'):
    """Every output to within the rounding of an fp32 sum of its own products, wherever its inputs lie in the range."""
    rt.set_option('conv_split_k', split)
    rt.set_option('split_k_reduce', reduce)
    got = rt.graph_inference(graph, len(x), x).astype(np.float64)
    x64, w64 = torch.from_numpy(x).double(), torch.from_numpy(conv.weight).double()
    want = torch.nn.functional.conv2d(x64, w64, None, 1, 1).numpy()
    size = torch.nn.functional.conv2d(x64.abs(), w64.abs(), None, 1, 1).numpy()
    # two roundings of an operand and one of a product are 2^-22 of it; a sum of FAN products in fp32 (in chunks of 16) is off by at
    # most FAN / 16 * 3 + 8 roundings of 2^-24 of their magnitudes; results below 2^-126 are rounded to multiples of 2^-149
    bound = size * (2.0 ** -22 + (FAN / 16 * 3 + 8) * 2.0 ** -24) + 2.0 ** -148
    worst = np.nanmax(np.abs(got - want) - bound)
    assert (np.abs(got - want) <= bound).all(), f'{what} split {split} {reduce}: {worst}'


@pytest.mark.parametrize('name', NAMES)
def test_magnitudes(name):
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    graph, conv = network()
    rng = np.random.default_rng(5)
    x = rng.standard_normal((BATCH, *SHAPE), dtype=np.float32)
    weight = conv.weight.copy()
    for e in (-100, -60, -12, -8, 0, 17, 19, 20, 25, 26, 40, 100):   # largest inputs on both sides of every limit
        check(graph, conv, np.ldexp(x, e).astype(np.float32), f'inputs times 2^{e}', 1)
    check(graph, conv, np.ldexp(x, 22).astype(np.float32), 'a second attempt', 3)
    check(graph, conv, np.ldexp(x, 40).astype(np.float32), 'far from 1', 3, 'kernel')
    # filters of every channel on another scale
    conv.weight = np.ldexp(weight, rng.integers(-90, 60, (OC, 1, 1, 1))).astype(np.float32)
    check(graph, conv, x, 'filters', 1)
    check(graph, conv, x, 'filters', 3, 'inline')
    conv.weight = np.zeros_like(weight)
    check(graph, conv, x, 'no filters', 1)
    conv.weight = weight
    # values on both sides of powers of two and of the largest half
    for value in (65504.0 * 16, 65505.0 * 16, 2.0 ** 26, np.nextafter(np.float32(2.0 ** 26), np.float32(0)), 2.0 ** -7, np.nextafter(np.float32(2.0 ** -7), np.float32(0))):
        check(graph, conv, np.clip(x * np.float32(1e30), -value, value).astype(np.float32), f'largest input {value}', 1)
    check(graph, conv, np.zeros_like(x), 'zeros', 2)


@pytest.mark.parametrize('name', NAMES)
def test_a_large_value_spares_the_others(name):
    """One image in the plain range, one with a value beyond it, one with an infinity: the outputs that do not see them are exact to
    the limits above, those that do are what fp32 gives."""
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    graph, conv = network()
    x = np.random.default_rng(6).standard_normal((BATCH, *SHAPE), dtype=np.float32)
    x[1, 20, 2, 3] = 3e20
    check(graph, conv, x, 'a large value', 1)
    check(graph, conv, x, 'a large value', 2)
    plain = x.copy()
    plain[1, 20, 2, 3] = 0
    for value, split in ((np.inf, 1), (np.inf, 2), (np.nan, 1), (np.nan, 2)):
        x[1, 20, 2, 3] = value
        rt.set_option('conv_split_k', split)
        got = rt.graph_inference(graph, BATCH, x)
        seen = np.zeros(got.shape, bool)
        seen[1, :, 1:4, 2:5] = True
        assert not np.isfinite(got[seen]).any()
        want = torch.nn.functional.conv2d(torch.from_numpy(plain).double(), torch.from_numpy(conv.weight).double(), None, 1, 1).numpy()
        np.testing.assert_allclose(got[~seen], want[~seen], rtol=1e-5, atol=1e-5)
        if value == np.inf:
            with np.errstate(invalid='ignore'):
                np.testing.assert_array_equal(np.signbit(got[seen]), np.signbit(torch.nn.functional.conv2d(torch.from_numpy(x), torch.from_numpy(conv.weight), None, 1, 1).numpy()[seen]))
