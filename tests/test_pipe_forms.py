"""The kernels that stage both operands have one form for inputs with a folded ReLU or channels to mask and one for inputs with neither: the
rule between them at its edges, by itself and in shared launches, against the oracle, and what registers the forms take."""
import os
import re

import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph, Value
from test_gpu_parity import assert_close, ios_oracle, matrix_path_convs
from test_large_batch_convs import FAMILIES

PIPE = [(name, precision, key) for precision, prefixes, key in FAMILIES for name in rt.conv_variant_names() if name.startswith(prefixes[0])]
LOGS = os.path.join(os.path.dirname(os.path.abspath(rt.__file__)), '..', '..', 'csrc', 'build')

# terms, units of a stage, tiles of a wavefront, wavefronts, 1 x 1: the least wavefronts per SIMD that the registers of the masked form leave room for
MASKED_WAVES = {'Li1E.*Li4ELi1ELi1ELi1ELi2ELi2ELb0': 5, 'Li1E.*Li4ELi1ELi1ELi1ELi2ELi2ELb1': 7, 'Li1E.*Li4ELi1ELi2ELi1ELi1ELi4ELb1': 4,
                'Li1E.*Li4ELi1ELi2ELi1ELi2ELi2ELb0': 4, 'Li1E.*Li4ELi1ELi3ELi1ELi1ELi4ELb0': 3, 'Li2E.*Li2ELi1ELi1ELi1ELi2ELi2ELb0': 5,
                'Li2E.*Li2ELi1ELi1ELi1ELi2ELi2ELb1': 6, 'Li2E.*Li2ELi1ELi1ELi1ELi1ELi4ELb0': 5}


def test_registers_of_the_forms():
    """What the compiler reported when this library was built: no spills, and masked forms that do not pay for the others."""
    found = {}
    for log in ('conv_pipe.log', 'conv_pipe_plain.log'):
        path = os.path.join(LOGS, log)
        if not os.path.exists(path):
            pytest.skip('built elsewhere')
        for record in open(path).read().split('Function Name: ')[1:]:
            name = record.split()[0]
            figures = {key: int(re.search(pattern, record).group(1)) for key, pattern in
                       (('waves', r'Occupancy \[waves/SIMD\]: (\d+)'), ('spilled', r'ScratchSize \[bytes/lane\]: (\d+)'))}
            assert figures['spilled'] == 0, name
            found[name] = figures['waves']
    for pattern, least in MASKED_WAVES.items():
        waves = [w for name, w in found.items() if re.search('ConvPipeI' + pattern + 'ELb0EEE', name)]
        assert len(waves) >= 2 and min(waves) >= least, (pattern, waves)


@pytest.fixture
def pinned():
    rt.set_option('autotune', 0)
    yield
    for key, value in (('conv_variant', -1), ('conv_split_k', 0), ('precision', 'fp32')):
        rt.set_option(key, value)


@pytest.mark.gpu
@pytest.mark.parametrize('name,precision,key', PIPE, ids=[n[0] for n in PIPE])
def test_forms(name, precision, key, pinned):
    """Channels on both sides of whole stages (16, 32 or 64) and of whole quads, with and without a folded ReLU, alone and beside a
    convolution of the same view that folds none."""
    rt.set_option('precision', precision)
    rt.set_option('conv_variant', rt.conv_variant_names().index(name))
    rt.set_option('conv_split_k', 1)
    for channels, kernel in [(c, (1, 1)) for c in (63, 64, 80, 96, 128)] + [(c, (3, 3)) for c in (20, 22, 32)]:
        for form in ('plain', 'folded', 'beside'):
            ios.reset_name()
            holder = ios.placeholder((channels + 3, 9, 11))
            block = Block(holder.node, None, [], None)
            view, pad = Value(holder.node, 1, channels + 1), (kernel[0] // 2, kernel[1] // 2)
            parts = []
            if form != 'folded': parts.append(ios.conv2d(block, [[view]], 40, kernel, (1, 1), pad, act='identity'))
            if form != 'plain': parts.append(ios.relu_conv(block, [[view]], 33, kernel, (1, 1), pad))
            ios.identity(block, [[v] for v in parts], is_exit=True)
            graph = Graph('forms', holder.node, [block])
            graph.init_weights(3, 'he_normal_bias')
            graph.sequential_schedule()
            x = np.random.default_rng(channels).standard_normal((3, *graph.enter_node.output_shape)).astype(np.float32)
            want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, 3)} if key else {}))
            x[:, 0] = x[:, channels + 1:] = np.nan   # beside the channels that are read
            assert_close(rt.graph_inference(graph, 3, x), want, f'{name} {channels} {kernel} {form}')
