"""A session that was given no weights, as the latency entry points and the schedule search use it, computes on values of ordinary
size: kernels whose time depends on magnitudes are measured as a network runs them."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('net', ['inception_v3', 'resnet50', 'squeezenet_1_1', 'randwire_small', 'nasnet_mobile'])
def test_tensors_stay_in_the_plain_range(net):
    graph = getattr(ios.models, net)()
    graph.sequential_schedule()
    graph.infer_shape()
    rt.set_option('autotune', 0)
    try:
        with rt.Session(graph, 1) as session:
            session.set_input(np.random.default_rng(0).standard_normal((1, *graph.enter_node.output_shape), dtype=np.float32))
            session.run()
            largest = np.abs(session.output()).max()
    finally:
        rt.set_option('autotune', 1)
    assert 2.0 ** -7 <= largest <= 65504.0, largest
