"""fp32 convolutions on operands whose magnitudes differ: every output is as good as a sum of its own products in fp32, whatever lies
beside it in its tile, in its batch or in its own sum.  All configurations that multiply fp32 operands as two terms of IEEE half, in
every form of their kernels."""
import numpy as np
import pytest
import torch

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph

pytestmark = pytest.mark.gpu

NAMES = [name for name in rt.conv_variant_names() if name.startswith(('x3p_', 'x3_win_', 'x3w_'))]

# in_shape, out channels, kernel, stride, padding, batch
FORMS = {
    '3x3': ((35, 9, 11), 37, (3, 3), (1, 1), (1, 1), 3),
    '1x1': ((75, 7, 9), 37, (1, 1), (1, 1), (0, 0), 3),
    '1x1 strided': ((75, 7, 9), 37, (1, 1), (2, 2), (0, 0), 3),
    '1x7': ((35, 9, 11), 37, (1, 7), (1, 1), (0, 3), 3),
    '5x5': ((19, 9, 11), 37, (5, 5), (1, 1), (2, 2), 2),
    '3x3 strided': ((35, 9, 11), 37, (3, 3), (2, 2), (0, 1), 3),
}


@pytest.fixture(autouse=True)
def default_options():
    rt.set_option('autotune', 0)
    yield
    for key, value in (('autotune', 1), ('executor', 'fused'), ('conv_variant', -1), ('conv_split_k', 0), ('split_k_reduce', 'xcd')):
        rt.set_option(key, value)


def network(form, groups=1):
    in_shape, oc, kernel, stride, pad, _ = form
    ios.reset_name()
    holder = ios.placeholder((in_shape[0] * groups, *in_shape[1:]))
    block = Block(holder.node, None, [], None)
    ios.conv2d(block, [[holder]], oc * groups, kernel, stride, pad, groups=groups, act='identity', is_exit=True)
    graph = Graph('mixed', holder.node, [block])
    graph.init_weights(3, 'he_normal')
    graph.sequential_schedule()
    conv = list(graph.conv_nodes())[0]
    conv.bias = np.zeros(oc * groups, np.float32)
    return graph, conv


def compare(got, conv, x, form, groups, what):
    _, _, kernel, stride, pad, _ = form
    x64, w64 = torch.from_numpy(x).double(), torch.from_numpy(conv.weight).double()
    want = torch.nn.functional.conv2d(x64, w64, None, stride, pad, 1, groups).numpy()
    size = torch.nn.functional.conv2d(x64.abs(), w64.abs(), None, stride, pad, 1, groups).numpy()
    # The operands of a product are off by 2^-23 each and the product of their lower terms (2^-22) is left out; the sum of FAN products in
    # fp32, in chunks of 16, is off by at most FAN / 16 * 3 + 8 roundings of 2^-24 of their magnitudes; results below 2^-126 are
    # rounded to multiples of 2^-149
    fan = conv.weight[0].size
    bound = size * (2.0 ** -21 + (fan / 16 * 3 + 8) * 2.0 ** -24) + 2.0 ** -148
    off = np.abs(got.astype(np.float64) - want)
    assert (off <= bound).all(), f'{what}: {np.nanmax(off / np.maximum(bound, 1e-300)):.3g} times the bound, {(~(off <= bound)).mean():.2%} of the outputs'


def check(graph, conv, x, form, what, groups=1):
    for split, reduce in ((1, 'xcd'), (2, 'inline'), (3, 'kernel')):
        rt.set_option('conv_split_k', split)
        rt.set_option('split_k_reduce', reduce)
        compare(rt.graph_inference(graph, len(x), x), conv, x, form, groups, f'{what} split {split} {reduce}')


def normal(form, seed, groups=1):
    return np.random.default_rng(seed).standard_normal((form[5], form[0][0] * groups, *form[0][1:]), dtype=np.float32)


@pytest.mark.parametrize('form', FORMS)
@pytest.mark.parametrize('name', NAMES)
def test_mixed(name, form):
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    form = FORMS[form]
    graph, conv = network(form)
    weight = conv.weight
    rng = np.random.default_rng(9)
    x = normal(form, 5)
    # pixels, from one to the next
    for low in (-10, -20, -40, -70):
        check(graph, conv, np.ldexp(x, rng.integers(low, 1, (form[5], 1, *form[0][1:]))).astype(np.float32), form, f'pixels from 2^{low} on')
    # images
    mixed = x.copy()
    mixed[0] *= np.float32(1e-6)
    mixed[1] *= np.float32(1e-4)
    check(graph, conv, mixed, form, 'images of 1e-6, 1e-4 and 1')
    mixed[-1, 3, 2, 2] = 6e7
    check(graph, conv, mixed, form, 'and one value of 6e7')
    # channels of the input, undone by the filters
    exponents = rng.integers(-40, 41, (form[0][0], 1, 1))
    conv.weight = np.ldexp(weight, -exponents).astype(np.float32)
    check(graph, conv, np.ldexp(x, exponents).astype(np.float32), form, 'channels and filters against each other')
    # one large channel that meets filters of zero: small ones must not lose a digit to it
    for e in (-12, -30, -60):
        conv.weight = weight.copy()
        conv.weight[:, 1] = 0
        mixed = np.ldexp(x, e).astype(np.float32)
        mixed[:, 1] = x[:, 1]
        check(graph, conv, mixed, form, f'channels of 2^{e} beside one of 1')
    # one large filter that meets inputs of zero
    for e in (-10, -20, -28, -45):
        conv.weight = np.ldexp(weight, e).astype(np.float32)
        conv.weight[:, 1] = weight[:, 1]
        mixed = x.copy()
        mixed[:, 1] = 0
        check(graph, conv, mixed, form, f'filters of 2^{e} beside one of 1')
    # every value its own magnitude
    conv.weight = np.ldexp(weight, rng.integers(-30, 1, weight.shape)).astype(np.float32)
    check(graph, conv, np.ldexp(x, rng.integers(-30, 1, x.shape)).astype(np.float32), form, 'any values')
    # small filters on small inputs, results of ordinary size from large ones
    for f, e in ((-20, -100), (-100, 20), (60, -100), (-60, 90), (-100, 120)):
        conv.weight = np.ldexp(weight, f).astype(np.float32)
        check(graph, conv, np.ldexp(x, e).astype(np.float32), form, f'filters of 2^{f} on inputs of 2^{e}')


@pytest.mark.parametrize('name', NAMES)
def test_groups(name):
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    form = FORMS['3x3']
    graph, conv = network(form, groups=2)
    x = normal(form, 6, 2)
    check(graph, conv, x, form, 'ordinary values', 2)
    for e in (-40, 22, 40):
        mixed = x.copy()
        mixed[:, 35:] = np.ldexp(x[:, 35:], e)
        check(graph, conv, mixed, form, f'a group of 2^{e}', 2)


@pytest.mark.parametrize('name', NAMES)
def test_infinite_values(name):
    """An infinite input or filter gives what fp32 gives, on the outputs that it meets and no others."""
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    form = FORMS['3x3']
    graph, conv = network(form)
    weight = conv.weight
    for what in ('input', 'filter'):
        for split in (1, 2):
            rt.set_option('conv_split_k', split)
            x = normal(form, 7)
            conv.weight = weight.copy()
            if what == 'input': x[1, 20, 2, 3] = np.inf
            else: conv.weight[5, 20, 1, 1] = -np.inf
            got = rt.graph_inference(graph, len(x), x)
            with np.errstate(invalid='ignore'):
                want = torch.nn.functional.conv2d(torch.from_numpy(x), torch.from_numpy(conv.weight), None, 1, 1).numpy()
            infinite = np.isinf(want)
            assert infinite.any()
            np.testing.assert_array_equal(got[infinite], want[infinite])
            plain = np.isfinite(want)
            np.testing.assert_allclose(got[plain], want[plain], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize('name', NAMES)
@pytest.mark.parametrize('folded', [False, True])
def test_residual_and_folded_relu(name, folded):
    """The residual form of the kernels (a convolution plus another one's output), and the ReLU of the producer in their loader."""
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    ios.reset_name()
    holder = ios.placeholder((67, 9, 11))
    block = Block(holder.node, None, [], None)
    if folded:
        ios.relu_conv(block, [[holder]], 40, (3, 3), (1, 1), (1, 1), is_exit=True)
    else:
        side = ios.conv2d(block, [[holder]], 40, (1, 1), act='identity')
        main = ios.conv2d(block, [[holder]], 40, (3, 3), (1, 1), (1, 1), act='identity')
        ios.addition(block, [[main, side]], is_exit=True)
    graph = Graph('residual', holder.node, [block])
    graph.init_weights(3, 'he_normal')
    graph.sequential_schedule()
    convs = list(graph.conv_nodes())
    for conv in convs:
        conv.bias = np.zeros(40, np.float32)
    if not folded:
        assert any(op.get('residual') for op in rt.plan_describe(graph, 3))
    rng = np.random.default_rng(3)
    x = np.ldexp(rng.standard_normal((3, 67, 9, 11), dtype=np.float32), rng.integers(-40, 1, (3, 1, 9, 11))).astype(np.float32)
    x64 = torch.from_numpy(x).double()
    if folded:
        x64 = x64.clamp(min=0)
    want, size = 0.0, 0.0
    for conv in convs:
        w64, pad = torch.from_numpy(conv.weight).double(), conv.weight.shape[2] // 2
        want = want + torch.nn.functional.conv2d(x64, w64, None, 1, pad).numpy()
        size = size + torch.nn.functional.conv2d(x64.abs(), w64.abs(), None, 1, pad).numpy()
    bound = size * (2.0 ** -21 + (67 * 9 / 16 * 3 + 10) * 2.0 ** -24) + 2.0 ** -148   # (see compare)
    for split in (1, 2):
        rt.set_option('conv_split_k', split)
        off = np.abs(rt.graph_inference(graph, 3, x).astype(np.float64) - want)
        assert (off <= bound).all(), f'split {split}: {(off / bound).max():.3g} times the bound'


# the configurations of that family: up to two 32 x 32 tiles and eight wavefronts
@pytest.mark.parametrize('name', ['x3w_m32n32_w8', 'x3w_m32n32_w4', 'x3w_m64n32_w8', 'x3w_m64n32_w4', 'x3w_m32n64_w4', 'x3w_m32n64_w8', 'x3w_m64n32_w2'])
def test_parallel_stage(name):
    """Two branches in one launch of the wide-register kernel family."""
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    rt.set_option('executor', 'fused')
    ios.reset_name()
    holder = ios.placeholder((67, 9, 11))
    block = Block(holder.node, None, [], None)
    one = ios.conv2d(block, [[holder]], 40, (1, 1), act='identity')
    three = ios.conv2d(block, [[holder]], 33, (3, 3), (1, 1), (1, 1), act='identity')
    ios.identity(block, [[one], [three]], is_exit=True)
    graph = Graph('parallel', holder.node, [block])
    graph.init_weights(3, 'he_normal')
    graph.greedy_schedule(4)
    convs = list(graph.conv_nodes())
    for conv in convs: conv.bias = np.zeros(conv.weight.shape[0], np.float32)
    rng = np.random.default_rng(4)
    by_size = {conv.weight.shape[2]: conv for conv in convs}
    plain = rng.standard_normal((3, 67, 9, 11), dtype=np.float32)
    for e in (None, -12, 22, 40, 110):
        shift = rng.integers(-40, 1, (3, 1, 9, 11)) if e is None else e
        x = np.ldexp(plain, shift).astype(np.float32)
        got = rt.graph_inference(graph, 3, x)
        compare(got[:, :40], by_size[1], x, ((67, 9, 11), 40, (1, 1), (1, 1), (0, 0), 3), 1, f'1x1 {e}')
        compare(got[:, 40:], by_size[3], x, ((67, 9, 11), 33, (3, 3), (1, 1), (1, 1), 3), 1, f'3x3 {e}')
