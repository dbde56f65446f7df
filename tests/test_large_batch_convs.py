"""The convolution kernels for large batches that stage both operands (x3p_*, wb_p_*, wh_p_*) or a window of the input
(x3_win_*, wb_win_*, wh_win_*) in LDS, at the edges of their tiles and windows, against the oracle."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph, Value
from test_gpu_parity import assert_close, ios_oracle, matrix_path_convs

pytestmark = pytest.mark.gpu

FAMILIES = [('fp32', ('x3p_', 'x3_win_'), None), ('bf16', ('wb_p_', 'wb_win_'), 'bf16_convs'), ('fp16', ('wh_p_', 'wh_win_'), 'fp16_convs')]
NAMES = [(name, precision, key) for precision, prefixes, key in FAMILIES for name in rt.conv_variant_names() if name.startswith(prefixes)]

# in_shape, out channels, kernel, padding, batch
CASES = [
    ((18, 9, 11), 33, (3, 3), (1, 1), 5),       # tiles over several images, channels that end inside a quad and a tile
    ((17, 13, 7), 64, (3, 3), (0, 0), 3),       # shrinking maps: tiles of one image each, the last one short
    ((40, 16, 17), 96, (1, 7), (0, 3), 2),      # one row, the taps beside the image masked
    ((35, 17, 9), 65, (7, 1), (3, 0), 2),
    ((16, 12, 12), 20, (5, 5), (2, 2), 4),      # 25 taps
    ((5, 3, 3), 200, (3, 3), (1, 1), 1),        # fewer pixels than any tile, one chunk of channels
    ((33, 6, 80), 31, (3, 3), (2, 0), 1),       # a map that grows in height: not for the window kernels
    ((20, 8, 200), 40, (3, 3), (1, 1), 1),      # rows too wide for the smaller windows
    ((24, 10, 10), 48, (2, 2), (0, 0), 2),      # an even number of taps
]


@pytest.fixture(autouse=True)
def default_options():
    rt.set_option('autotune', 0)
    yield
    for key, value in (('autotune', 0), ('executor', 'fused'), ('conv_variant', -1), ('conv_split_k', 0), ('precision', 'fp32'), ('split_k_reduce', 'xcd')):
        rt.set_option(key, value)


def build(case, reader):
    """The convolution reads a channel window of the input (from an odd channel on) and writes one of a concatenation."""
    in_shape, oc, kernel, pad, _ = case
    ios.reset_name()
    holder = ios.placeholder((in_shape[0] + 3, *in_shape[1:]))
    block = Block(holder.node, None, [], None)
    window = Value(holder.node, 1, in_shape[0] + 1)
    conv = ios.conv2d(block, [[window]], oc, kernel, (1, 1), pad, act='relu')
    if reader:
        other = ios.pool2d(block, [[conv]], 'max', (3, 3), (1, 1), (1, 1))
        ios.identity(block, [[other], [conv]], is_exit=True)
    else:
        ios.identity(block, [[conv]], is_exit=True)
    graph = Graph('large', holder.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    graph.sequential_schedule()
    return graph


@pytest.mark.parametrize('name,precision,key', NAMES, ids=[n[0] for n in NAMES])
def test_edges(name, precision, key):
    rt.set_option('precision', precision)
    rt.set_option('conv_variant', rt.device_info()['conv_variants'].index(name))
    for index, case in enumerate(CASES):
        graph = build(case, reader=index % 2 == 0)
        x = np.random.default_rng(index).standard_normal((case[4], *graph.enter_node.output_shape)).astype(np.float32)
        want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, case[4])} if key else {}))
        for split, reduce in ((1, 'xcd'), (2, ('xcd', 'inline', 'kernel')[index % 3])):
            rt.set_option('conv_split_k', split)
            rt.set_option('split_k_reduce', reduce)
            got = rt.graph_inference(graph, case[4], x)
            assert_close(got, want, f'{name} {case} split {split} {reduce}')


# channels, out channels, map, stride, padding, batch of 1 x 1 filters: one channel short of a quad, of an octet and of a stage's units; one
# channel beyond them; fewer channels than a stage; pixels beside the map
POINTS = [(31, 33, (9, 11), 1, 0, 3), (65, 64, (7, 5), 2, 0, 5), (23, 200, (6, 6), 1, 1, 2), (3, 20, (13, 17), 3, 0, 1), (96, 97, (3, 3), 2, 1, 4)]


@pytest.mark.parametrize('name,precision,key', [n for n in NAMES if '_win_' not in n[0]], ids=[n[0] for n in NAMES if '_win_' not in n[0]])
def test_filters_of_one_pixel(name, precision, key):
    """1 x 1 filters walk K by moving the ends of their buffers: what lies beside the channels they read is NaN and must not show."""
    rt.set_option('precision', precision)
    rt.set_option('conv_variant', rt.device_info()['conv_variants'].index(name))
    for channels, oc, size, stride, pad, batch in POINTS:
        ios.reset_name()
        holder = ios.placeholder((channels + 3, *size))
        block = Block(holder.node, None, [], None)
        ios.conv2d(block, [[Value(holder.node, 1, channels + 1)]], oc, (1, 1), (stride, stride), (pad, pad), act='identity', is_exit=True)
        graph = Graph('point', holder.node, [block])
        graph.init_weights(3, 'he_normal_bias')
        graph.sequential_schedule()
        x = np.random.default_rng(channels).standard_normal((batch, channels + 3, *size)).astype(np.float32)
        want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, batch)} if key else {}))
        x[:, 0] = x[:, channels + 1:] = np.nan
        for split, reduce in ((1, 'xcd'), (2, 'inline'), (3, 'kernel')):
            rt.set_option('conv_split_k', split)
            rt.set_option('split_k_reduce', reduce)
            assert_close(rt.graph_inference(graph, batch, x), want, f'{name} {channels} -> {oc} stride {stride} padding {pad} split {split} {reduce}')


@pytest.mark.parametrize('executor', ['fused', 'fused_graph'])
@pytest.mark.parametrize('precision,key', [('bf16', 'bf16_convs'), ('fp16', 'fp16_convs')])
def test_parallel_stage_launches_large_convolutions_by_themselves(precision, key, executor):
    """Measured configurations: two large convolutions of a parallel stage take kernels no fused launch holds; the small convolution
    and the pool beside them share one launch."""
    ios.reset_name()
    holder = ios.placeholder((64, 35, 35))
    block = Block(holder.node, None, [], None)
    first = ios.conv2d(block, [[holder]], 96, (3, 3), (1, 1), (1, 1))
    second = ios.conv2d(block, [[holder]], 96, (3, 3), (1, 1), (1, 1), act='identity')
    small = ios.conv2d(block, [[Value(holder.node, 3, 11)]], 7, (1, 1))
    pool = ios.pool2d(block, [[holder]], 'max', (3, 3), (1, 1), (1, 1))
    ios.identity(block, [[first], [second], [small], [pool]], is_exit=True)
    graph = Graph('stage', holder.node, [block])
    graph.init_weights(4, 'he_normal_bias')
    graph.greedy_schedule(8)
    x = np.random.default_rng(9).standard_normal((24, 64, 35, 35)).astype(np.float32)
    rt.set_option('precision', precision)
    rt.set_option('executor', executor)
    rt.set_option('autotune', 1)
    with rt.Session(graph, 24) as session:
        session.load_weights()
        session.set_input(x)
        kernels = [launch['kernel'] for launch in session.launches()]
        assert sum(name.startswith('conv_kernel<') for name in kernels) == 2 and sum(name.startswith('fused_kernel') for name in kernels) == 1, kernels
        for _ in range(3):
            session.run()
            got = session.output()
        convs = frozenset(op['node'] for op in session.describe() if op['kind'] == 'conv_mfma')
    assert_close(got, ios_oracle.run(graph, x, **{key: convs}), f'{precision} {executor}')


@pytest.mark.parametrize('variant', [None, 'x3p_m64n128_w1x4', 'wq_m64n32_w4_t32', 'm64n64k32_w2x2x1_t32'])
def test_an_input_of_a_gigabyte(variant):
    """85 images of 3 x 1024 x 1024: 1.07 GB of values, 1.43 GB with the pixels padded."""
    if variant is not None:
        rt.set_option('conv_variant', rt.conv_variant_names().index(variant))
    ios.reset_name()
    holder = ios.placeholder((3, 1024, 1024))
    block = Block(holder.node, None, [], None)
    ios.conv2d(block, [[holder]], 32, (5, 5), (4, 4), (2, 2), is_exit=True)
    graph = Graph('gigabyte', holder.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    graph.sequential_schedule()
    x = np.tile(np.random.default_rng(0).standard_normal((5, 3, 1024, 1024), dtype=np.float32), (17, 1, 1, 1))
    with rt.Session(graph, 85) as session:
        assert [op['kind'] for op in session.describe()] == ['conv_mfma']
        session.load_weights()
        session.set_input(x)
        session.run()
        got = session.output()
    want = ios_oracle.run(graph, x[:5])
    for image in (0, 1, 42, 63, 83, 84):   # 2^30 bytes of padded pixels end inside image 64
        assert_close(got[image], want[image % 5], f'image {image}')
