"""Inputs that need neither a ReLU nor channels masked take forms of the staged two-term kernels of their own (whole stages of channels for
1 x 1 filters, whole quads for others), with the limits, the second attempt and the fp32 results in code of their own: operands whose
magnitudes differ, infinities and NaN through these forms, by themselves and in shared launches."""
import numpy as np
import pytest
import torch

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph
from test_mixed_magnitudes import check, compare, network, normal

pytestmark = pytest.mark.gpu

PIPE = [name for name in rt.conv_variant_names() if name.startswith('x3p_')]
WINDOW = [name for name in rt.conv_variant_names() if name.startswith('x3_win_')]

# in_shape, out channels, kernel, stride, padding, batch
FORMS = {
    '1x1': ((128, 7, 9), 37, (1, 1), (1, 1), (0, 0), 3),
    '1x1 strided': ((64, 7, 9), 37, (1, 1), (2, 2), (0, 0), 3),
    '3x3': ((36, 9, 11), 37, (3, 3), (1, 1), (1, 1), 3),
    '3x3 strided': ((32, 9, 11), 37, (3, 3), (2, 2), (0, 1), 3),
    '1x7': ((64, 9, 11), 37, (1, 7), (1, 1), (0, 3), 3),
    '5x5': ((20, 9, 11), 37, (5, 5), (1, 1), (2, 2), 2),
}


@pytest.fixture(autouse=True)
def default_options():
    rt.set_option('autotune', 0)
    yield
    for key, value in (('autotune', 1), ('executor', 'fused'), ('conv_variant', -1), ('conv_split_k', 0), ('split_k_reduce', 'xcd')):
        rt.set_option(key, value)


def infinite_as_fp32_has_it(got, conv, x, form):
    """What meets the value is what fp32 gives, everything else an ordinary result."""
    with np.errstate(invalid='ignore'):
        want = torch.nn.functional.conv2d(torch.from_numpy(x), torch.from_numpy(conv.weight), None, form[3], form[4]).numpy()
    plain = np.isfinite(want)
    assert not plain.all()
    infinite = np.isinf(want)
    np.testing.assert_array_equal(got[infinite], want[infinite])
    assert np.isnan(got[np.isnan(want)]).all()
    np.testing.assert_allclose(got[plain], want[plain], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize('form', FORMS)
@pytest.mark.parametrize('name', PIPE + WINDOW)
def test_magnitudes(name, form):
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    form = FORMS[form]
    graph, conv = network(form)
    weight = conv.weight
    rng = np.random.default_rng(9)
    x = normal(form, 5)
    # one factor for all: the plain range, both sides of it, a second attempt, far from one
    for e in (0, -40, 17, 22, 40, 100):
        check(graph, conv, np.ldexp(x, e).astype(np.float32), form, f'inputs times 2^{e}')
    # from pixel to pixel, and late channels that no first stage shows
    check(graph, conv, np.ldexp(x, rng.integers(-40, 1, (form[5], 1, *form[0][1:]))).astype(np.float32), form, 'pixels from 2^-40 on')
    late = x.copy()
    late[:, -5] = np.ldexp(late[:, -5], 22)
    check(graph, conv, late, form, 'a late channel of 2^22')
    late[-1, -1, 2, 2] = 3e20
    check(graph, conv, late, form, 'and one late value of 3e20')
    # small ones must not lose a digit to a large channel that meets filters of zero
    conv.weight = weight.copy()
    conv.weight[:, 1] = 0
    mixed = np.ldexp(x, -30).astype(np.float32)
    mixed[:, 1] = x[:, 1]
    check(graph, conv, mixed, form, 'channels of 2^-30 beside one of 1')
    conv.weight = np.ldexp(weight, rng.integers(-30, 1, weight.shape)).astype(np.float32)
    check(graph, conv, np.ldexp(x, rng.integers(-30, 1, x.shape)).astype(np.float32), form, 'any values')


@pytest.mark.parametrize('form', ['1x1', '3x3', '1x7'])
@pytest.mark.parametrize('name', PIPE + WINDOW)
def test_infinities_and_nan(name, form):
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    form = FORMS[form]
    graph, conv = network(form)
    for channel in (1, form[0][0] - 2):
        for value in (np.inf, -np.inf, np.nan):
            for split in (1, 2):
                rt.set_option('conv_split_k', split)
                x = normal(form, 7)
                x[1, channel, 2, 3] = value
                infinite_as_fp32_has_it(rt.graph_inference(graph, len(x), x), conv, x, form)


def shared(channels, kernels):
    ios.reset_name()
    holder = ios.placeholder((channels, 9, 11))
    block = Block(holder.node, None, [], None)
    parts = [ios.conv2d(block, [[holder]], oc, kernel, (1, 1), (kernel[0] // 2, kernel[1] // 2), act='identity') for oc, kernel in zip((37, 70, 8), kernels)]
    ios.identity(block, [[v] for v in parts], is_exit=True)
    graph = Graph('shared', holder.node, [block])
    graph.init_weights(3, 'he_normal')
    graph.sequential_schedule()
    convs = list(graph.conv_nodes())
    for conv in convs: conv.bias = np.zeros(conv.weight.shape[0], np.float32)
    return graph, convs


@pytest.mark.parametrize('name,channels,kernels', [(name, 128, [(1, 1)] * 3) for name in PIPE] +
                         [(name, 36, kernels) for name in PIPE + WINDOW for kernels in ([(1, 7), (7, 1)], [(3, 3), (1, 3), (5, 5)])])
def test_shared_launches(name, channels, kernels):
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    rt.set_option('conv_split_k', 1)
    graph, convs = shared(channels, kernels)
    rng = np.random.default_rng(11)
    x = rng.standard_normal((3, channels, 9, 11), dtype=np.float32)
    late = x.copy()
    late[:, -5] = np.ldexp(late[:, -5], 22)
    infinite = x.copy()
    infinite[1, -2, 2, 3] = np.inf
    with rt.Session(graph, 3) as session:
        session.load_weights()
        assert sum('batch' in op for op in session.describe()) == len(kernels)
        for what, values in [(f'2^{e}', np.ldexp(x, e).astype(np.float32)) for e in (0, 22, 40, -40)] + [('a late channel', late), (None, infinite)] + \
                [('pixels', np.ldexp(x, rng.integers(-40, 1, (3, 1, 9, 11))).astype(np.float32))]:
            session.set_input(values)
            session.run()
            got, first = session.output(), 0
            for conv, kernel in zip(convs, kernels):
                oc = conv.weight.shape[0]
                form = ((channels, 9, 11), oc, kernel, (1, 1), (kernel[0] // 2, kernel[1] // 2), 3)
                if what is None: infinite_as_fp32_has_it(got[:, first:first + oc], conv, values, form)
                else: compare(got[:, first:first + oc], conv, values, form, 1, f'{what} {kernel}')
                first += oc
