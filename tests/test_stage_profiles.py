"""The times of single stages belong to the stages of the schedule, also where a pass launches convolutions of several stages together."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from test_conv_batches import heads
from test_library import _simulate


@pytest.fixture(autouse=True)
def default_options():
    yield
    for key, value in (('batch_convs', 1), ('batch_across_stages', 1), ('host_plan_batches', 0), ('arena_reuse', 1)):
        rt.set_option(key, value)


@pytest.mark.parametrize('level', [1, 2])
@pytest.mark.parametrize('name,schedule', [('inception_v3', 'sequential'), ('inception_v3', 'greedy'), ('nasnet_mobile', 'greedy')])
def test_operations_in_their_own_stages(name, schedule, level):
    """Without launches across stages nothing leaves its stage.  With them, what is read is still there in the stage of the schedule."""
    graph = getattr(ios.models, name)()
    if schedule == 'greedy':
        graph.greedy_schedule(8)
    else:
        graph.sequential_schedule()
    rt.set_option('arena_reuse', 0)
    plain = rt.plan_describe(graph, 2)
    rt.set_option('host_plan_batches', level)
    moved = [op for op in rt.plan_describe(graph, 2) if 'scheduled_stage' in op]
    assert len(moved) > 0 or schedule == 'greedy'
    rt.set_option('batch_across_stages', 0)
    within = rt.plan_describe(graph, 2)
    assert [op['stage'] for op in within] == [op['stage'] for op in plain] and not any('scheduled_stage' in op for op in within)
    rt.set_option('batch_across_stages', 1)
    rt.set_option('arena_reuse', 1)
    ops = rt.plan_describe(graph, 2)
    assert [op.get('scheduled_stage', op['stage']) for op in ops] == [op['stage'] for op in plain]
    # every operation where a pass with timed stages has it: shared launches of a stage, then its groups
    last = 1 + max(op.get('batch', 0) for op in ops)
    timed = [dict(op, stage=op.get('scheduled_stage', op['stage']) * (last + 1) + op.get('batch', last), group=0 if 'batch' in op else op['group']) for op in ops]
    order = [i for stage in sorted({o['stage'] for o in timed}) for i, o in enumerate(timed) if o['stage'] == stage]
    plain_order = [i for stage in sorted({o['stage'] for o in plain}) for i, o in enumerate(plain) if o['stage'] == stage]
    assert dict(zip(order, _simulate(timed))) == dict(zip(plain_order, _simulate(plain)))


@pytest.mark.gpu
@pytest.mark.parametrize('executor', ['fused', 'fused_graph', 'streams', 'graph'])
def test_times_of_stages(executor):
    """Four like convolutions of one view in a stage each: none of them may be timed as nothing."""
    rt.set_option('autotune', 0)
    try:
        rt.set_option('executor', executor)
        rt.set_option('conv_variant', rt.conv_variant_names().index('x3p_m64n64_w2x2'))
        rt.set_option('conv_split_k', 1)
        graph = heads((768, 17, 17), (192, 192, 192, 192), 1, 0, 'sequential')
        x = np.random.default_rng(1).standard_normal((64, *graph.enter_node.output_shape)).astype(np.float32)
        with rt.Session(graph, 64) as session:
            session.load_weights()
            convs = [op.get('scheduled_stage', op['stage']) for op in session.describe() if 'batch' in op]
            assert len(set(convs)) == 4 and len(set(op['stage'] for op in session.describe() if 'batch' in op)) == 1
            session.set_input(x)
            session.run()
            want = session.output()
            _, stages = session.measure(2, 4, 3, profile_stage=True)
            assert np.array_equal(session.output(), want)
            session.run()
            assert np.array_equal(session.output(), want)
        for times in (stages, rt.graph_latency(graph, 64, 2, 4, 3, profile_stage=True)[1]):
            mine = np.asarray(times).reshape(3, -1).mean(0)[convs]
            assert mine.min() > 0.4 * mine.max(), (executor, mine)
    finally:
        for key, value in (('executor', 'fused'), ('conv_variant', -1), ('conv_split_k', 0)):
            rt.set_option(key, value)
