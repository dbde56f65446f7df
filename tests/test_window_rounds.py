"""The window convolution kernels on both sides of the longest window that the kernels of three rounds hold (384 input pixels where a block has
256 threads: 256 outputs, two further rows of a 3 x 3 filter or six of a 7 x 1 one), against the oracle."""
import numpy as np
import pytest

from ios.contrib import ios_runtime as rt
from test_gpu_parity import assert_close, ios_oracle, matrix_path_convs
from test_large_batch_convs import NAMES, build, default_options  # noqa: F401

pytestmark = pytest.mark.gpu

# in_shape, out channels, kernel, padding, batch: 255 + 2 * 63 + 3 = 384 pixels, 386; 255 + 6 * 21 + 1 = 382, 388; 8 further; channels that end inside a quad
CASES = [((20, 9, 63), 40, (3, 3), (1, 1), 2), ((20, 9, 64), 40, (3, 3), (1, 1), 2), ((36, 16, 21), 33, (7, 1), (3, 0), 3), ((36, 16, 22), 33, (7, 1), (3, 0), 3),
         ((18, 7, 120), 64, (3, 3), (1, 1), 1), ((33, 3, 90), 70, (1, 7), (0, 3), 2)]


@pytest.mark.parametrize('name,precision,key', [n for n in NAMES if '_win_' in n[0]], ids=[n[0] for n in NAMES if '_win_' in n[0]])
def test_windows_of_three_rounds_and_more(name, precision, key):
    rt.set_option('precision', precision)
    rt.set_option('conv_variant', rt.device_info()['conv_variants'].index(name))
    for index, case in enumerate(CASES):
        graph = build(case, reader=False)
        x = np.random.default_rng(index).standard_normal((case[4], *graph.enter_node.output_shape)).astype(np.float32)
        want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, case[4])} if key else {}))
        assert_close(rt.graph_inference(graph, case[4], x), want, f'{name} {case}')
