"""ReLU gives 0 for NaN, whatever the planner folds it into (reference: NOT_PROPAGATE_NAN); other values keep their bits."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph
from test_gpu_parity import assert_close, ios_oracle

pytestmark = pytest.mark.gpu

NAMES = [(name, {'wb_': 'bf16', 'wh_': 'fp16'}.get(name[:3], 'fp32')) for name in rt.conv_variant_names()]


@pytest.fixture(autouse=True)
def default_options():
    rt.set_option('autotune', 0)
    yield
    for key, value in (('autotune', 1), ('conv_variant', -1), ('conv_split_k', 0), ('precision', 'fp32'), ('thin_conv_min_pixels', 1 << 18)):
        rt.set_option(key, value)


def network(shape, operators):
    ios.reset_name()
    holder = ios.placeholder(shape)
    block = Block(holder.node, None, [], None)
    operators(block, holder)
    graph = Graph('nan', holder.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    graph.sequential_schedule()
    return graph


def with_nans(shape, batch, share=0.02):
    rng = np.random.default_rng(7)
    x = rng.standard_normal((batch, *shape), dtype=np.float32)
    where = rng.random(x.shape)
    x[where < share] = np.float32(np.nan)
    x[where < share / 2] = np.array([0xffc00000], np.uint32).view(np.float32)[0]   # the other sign
    x[(where > 1 - share / 2)] = np.float32(0)
    return x


def run(graph, x):
    with rt.Session(graph, len(x)) as session:
        session.load_weights()
        session.set_input(x)
        session.run()
        return session.output()


def check_behind(graph, x, exact=True):
    """ReLU is the last operator: NaNs of the values it works on are zeros of the result."""
    got = run(graph, x)
    with np.errstate(invalid='ignore'):
        want = ios_oracle.run(graph, x)
    assert np.isnan(want).any() and not np.isnan(want).all()
    assert np.isfinite(got).all() and (got[np.isnan(want)] == 0).all() and (got >= 0).all()
    if exact:
        assert_close(got, np.nan_to_num(want, nan=0.0), 'values that are numbers')


def check_in_front(graph, x, exact=True):
    """ReLU is the first operator: the rest of the network sees zeros."""
    got = run(graph, x)
    assert np.isfinite(got).all()
    if exact:
        assert_close(got, ios_oracle.run(graph, np.nan_to_num(x, nan=0.0)), 'behind the ReLU')


@pytest.mark.parametrize('name,precision', NAMES, ids=[n[0] for n in NAMES])
def test_matrix_path(name, precision):
    rt.set_option('precision', precision)
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    shape = (20, 9, 11)
    graph = network(shape, lambda b, v: ios.conv2d(b, [[v]], 33, (3, 3), (1, 1), (1, 1), act='relu', is_exit=True))
    check_behind(graph, with_nans(shape, 2, 0.002), precision == 'fp32')
    graph = network(shape, lambda b, v: ios.relu_conv(b, [[v]], 33, (3, 3), (1, 1), (1, 1), is_exit=True))
    assert [op['conv']['pre_relu'] for op in rt.plan_describe(graph, 2)] == [1]
    check_in_front(graph, with_nans(shape, 2), precision == 'fp32')
    # without ReLU, NaNs are NaNs
    graph = network(shape, lambda b, v: ios.conv2d(b, [[v]], 33, (3, 3), (1, 1), (1, 1), act='identity', is_exit=True))
    x = with_nans(shape, 2, 0.002)
    with np.errstate(invalid='ignore'):
        assert np.array_equal(np.isnan(run(graph, x)), np.isnan(ios_oracle.run(graph, x)))


@pytest.mark.parametrize('split,form', [(4, 'xcd'), (4, 'kernel')])
def test_split_k(split, form):
    rt.set_option('conv_split_k', split)
    rt.set_option('split_k_reduce', form)
    try:
        shape = (200, 8, 8)
        check_behind(network(shape, lambda b, v: ios.conv2d(b, [[v]], 33, (3, 3), (1, 1), (1, 1), act='relu', is_exit=True)), with_nans(shape, 2, 0.0003))
    finally:
        rt.set_option('split_k_reduce', 'xcd')


def residual(block, v):
    a = ios.conv2d(block, [[v]], 20, (3, 3), (1, 1), (1, 1), act='identity')
    b = ios.conv2d(block, [[a]], 20, (3, 3), (1, 1), (1, 1), act='identity')
    total = ios.addition(block, [[b, v]])
    ios.relu(block, [[total]], is_exit=True)


def pooled(block, v):
    p = ios.pool2d(block, [[v]], 'avg', (3, 3), (1, 1), (1, 1))
    ios.conv2d(block, [[p]], 12, (1, 1), act='relu', is_exit=True)


def summed(block, v):
    p = ios.pool2d(block, [[v]], 'avg', (3, 3), (1, 1), (1, 1))
    ios.relu(block, [[v, p]], is_exit=True)


BEHIND = {
    'relu': ((20, 9, 11), lambda b, v: ios.relu(b, [[v]], is_exit=True)),
    'relu of a sum': ((20, 9, 11), summed),
    'depth-wise': ((20, 9, 11), lambda b, v: ios.conv2d(b, [[v]], 20, (3, 3), (1, 1), (1, 1), groups=20, act='relu', is_exit=True)),
    'thin groups': ((20, 9, 11), lambda b, v: ios.conv2d(b, [[v]], 30, (3, 3), (1, 1), (1, 1), groups=10, act='relu', is_exit=True)),
    'first layer': ((3, 33, 35), lambda b, v: ios.conv2d(b, [[v]], 32, (3, 3), (2, 2), act='relu', is_exit=True)),
    'residual': ((20, 9, 11), residual),
    'pool behind its convolution': ((20, 9, 11), pooled),
}


@pytest.mark.parametrize('batch', [1, 37])
@pytest.mark.parametrize('case', sorted(BEHIND))
def test_behind(case, batch):
    rt.set_option('thin_conv_min_pixels', 0)
    shape, operators = BEHIND[case]
    check_behind(network(shape, operators), with_nans(shape, batch, 0.002 if batch > 1 else 0.004))


FRONT = {
    'depth-wise': ((20, 9, 11), lambda b, v: ios.relu_sep_conv(b, [[v]], 20, (3, 3), (1, 1), (1, 1), is_exit=True)),
    'depth-wise 5x5': ((20, 9, 11), lambda b, v: ios.relu_sep_conv(b, [[v]], 20, (5, 5), (1, 1), (2, 2), is_exit=True)),
    'depth-wise of a sum': ((20, 9, 11), lambda b, v: ios.relu_sep_conv(b, [[v, v]], 20, (3, 3), (1, 1), (1, 1), is_exit=True)),
    'first layer': ((3, 33, 35), lambda b, v: ios.relu_conv(b, [[v]], 32, (3, 3), (2, 2), is_exit=True)),
}


@pytest.mark.parametrize('batch', [1, 37])
@pytest.mark.parametrize('case', sorted(FRONT))
def test_in_front(case, batch):
    rt.set_option('thin_conv_min_pixels', 0)
    shape, operators = FRONT[case]
    check_in_front(network(shape, operators), with_nans(shape, batch))


def test_other_values_keep_their_bits():
    """Infinities, denormal numbers and zeros through a ReLU and through a copy."""
    tiny = np.array([1, 0x807fffff, 0x007fffff, 0x80000001], np.uint32).view(np.float32)
    row = np.concatenate([np.array([np.inf, -np.inf, 0.0, 3e38, -3e38, 1.5, -1.5], np.float32), tiny])
    shape = (11, 5, 7)
    x = np.broadcast_to(row[:, None, None], (3, *shape)).astype(np.float32)

    def both(block, v):
        r = ios.relu(block, [[v]])
        ios.identity(block, [[r], [v]], is_exit=True)

    got = run(network(shape, both), x)
    assert np.array_equal(got[:, :11], np.maximum(x, 0)) and np.array_equal(got[:, 11:].view(np.uint32), x.view(np.uint32))
