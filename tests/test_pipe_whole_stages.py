"""1 x 1 filters whose channels fill every stage of the kernels that stage both operands (the form without masks), against the oracle: few and
many stages, the last tile of pixels and of channels short, filters that are shared by the blocks of an XCD in either order of the tiles."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph, Value
from test_gpu_parity import assert_close, ios_oracle, matrix_path_convs
from test_large_batch_convs import NAMES, default_options  # noqa: F401

pytestmark = pytest.mark.gpu

# channels, out channels, map, stride, padding, batch: one stage, an even and an odd number of them; more filters than inputs and the other way
# round, with more tiles than XCDs; pixels beside the map
CASES = [(64, 33, (9, 11), 1, 0, 3), (128, 200, (7, 5), 2, 0, 5), (192, 40, (33, 31), 1, 0, 3), (576, 520, (4, 5), 1, 0, 2), (64, 97, (6, 6), 1, 1, 2)]


@pytest.mark.parametrize('name,precision,key', [n for n in NAMES if '_win_' not in n[0]], ids=[n[0] for n in NAMES if '_win_' not in n[0]])
def test_whole_stages(name, precision, key):
    """What lies beside the channels that are read is NaN and must not show."""
    rt.set_option('precision', precision)
    rt.set_option('conv_variant', rt.device_info()['conv_variants'].index(name))
    for channels, oc, size, stride, pad, batch in CASES:
        ios.reset_name()
        holder = ios.placeholder((channels + 3, *size))
        block = Block(holder.node, None, [], None)
        ios.conv2d(block, [[Value(holder.node, 1, channels + 1)]], oc, (1, 1), (stride, stride), (pad, pad), act='identity', is_exit=True)
        graph = Graph('stages', holder.node, [block])
        graph.init_weights(3, 'he_normal_bias')
        graph.sequential_schedule()
        x = np.random.default_rng(channels).standard_normal((batch, channels + 3, *size)).astype(np.float32)
        want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, batch)} if key else {}))
        x[:, 0] = x[:, channels + 1:] = np.nan
        for split in (1, 2):
            rt.set_option('conv_split_k', split)
            assert_close(rt.graph_inference(graph, batch, x), want, f'{name} {channels} -> {oc} stride {stride} padding {pad} split {split}')
