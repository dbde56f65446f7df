"""Batches that arrive in parts: images of many channels whose parts begin anywhere in a line of memory, and leading stages whose
convolutions share launches."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph
from test_gpu_parity import assert_close, ios_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('channels,side,batch', [(7, (61, 83), 33), (33, (37, 41), 19), (131, (17, 31), 17)])
def test_many_channels_at_odd_places(channels, side, batch):
    """A network that copies its input hands every value back, from parts of odd numbers of floats."""
    ios.reset_name()
    holder = ios.placeholder((channels, *side))
    block = Block(holder.node, None, [], None)
    largest = ios.pool2d(block, [[holder]], 'max', (1, 1))
    ios.identity(block, [[largest]], is_exit=True)
    graph = Graph('copy', holder.node, [block])
    graph.sequential_schedule()
    with rt.Session(graph, batch) as session:
        assert any('part_ends' in op for op in session.describe())
        for seed in range(3):
            x = np.random.default_rng(seed).standard_normal((batch, channels, *side)).astype(np.float32)
            session.set_input(x)
            session.run()
            assert np.array_equal(session.output(), x)


@pytest.mark.parametrize('batch', [16, 33])
@pytest.mark.parametrize('variant,precision', [('x3p_m64n64_w2x2', 'fp32'), ('wb_p_m64n128_w1x4', 'bf16')])
def test_shared_launches_on_parts(batch, variant, precision):
    """Two heads in one launch, part by part and on the whole batch: what the oracle has, in fp32, and bit for bit what they give apart.  (The
    heads are a second convolution: in bfloat16 it rounds sums that differ in their last bit from the oracle's to operands that differ by 2^-8.)"""
    ios.reset_name()
    v = ios.placeholder((3, 131, 127))
    block = Block(v.node)
    a = ios.conv2d(block, [[v]], 21, (3, 3), (2, 2))
    b, c = (ios.conv2d(block, [[a]], oc, (1, 1)) for oc in (8, 30))
    tail = ios.pool2d(block, [[b]], 'max', (3, 3), (1, 1), (1, 1))
    ios.identity(block, [[tail], [c]], is_exit=True)
    graph = Graph('t', v.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    graph.sequential_schedule()
    rt.set_option('autotune', 0)
    try:
        rt.set_option('precision', precision)
        rt.set_option('conv_variant', rt.conv_variant_names().index(variant))
        rt.set_option('conv_split_k', 1)
        outputs = {}
        for shared in (1, 0):
            rt.set_option('batch_convs', shared)
            with rt.Session(graph, batch) as session:
                session.load_weights()
                heads = [op for op in session.describe() if 'batch' in op]
                assert len(heads) == (2 if shared else 0) and all('part_ends' in op for op in heads)
                for seed in range(2):
                    x = np.random.default_rng(seed).standard_normal((batch, *graph.enter_node.output_shape)).astype(np.float32)
                    session.set_input(x)
                    session.run()
                    outputs.setdefault(seed, []).append(session.output())
                    session.run()   # (the input is there: the whole batch at once)
                    outputs[seed].append(session.output())
        for seed in range(2):
            if precision == 'fp32':
                x = np.random.default_rng(seed).standard_normal((batch, *graph.enter_node.output_shape)).astype(np.float32)
                assert_close(outputs[seed][0], ios_oracle.run(graph, x), f'{variant} {batch}')
            assert len(outputs[seed]) == 4 and all(np.array_equal(outputs[seed][0], other) for other in outputs[seed][1:])
    finally:
        for option, value in (('autotune', 1), ('conv_variant', -1), ('conv_split_k', 0), ('precision', 'fp32'), ('batch_convs', 1)):
            rt.set_option(option, value)
