"""1 x 1 convolutions of one view that share a launch: the plans on the host, and the kernels against single launches and the oracle."""
import os
import subprocess
import sys

import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph, Value
from test_gpu_parity import assert_close, ios_oracle, matrix_path_convs
from test_large_batch_convs import FAMILIES
from test_library import _simulate, _simulate_parts

POINT = [(name, precision, key) for precision, prefixes, key in FAMILIES for name in rt.conv_variant_names() if name.startswith(prefixes[0])]


@pytest.fixture(autouse=True)
def default_options():
    yield
    for key, value in (('batch_convs', 1), ('host_plan_batches', 0), ('arena_reuse', 1)):
        rt.set_option(key, value)


def heads(shape, channels, stride, pad, schedule, front=True):
    """Convolutions of an odd channel window: plain, behind a folded ReLU, in front of an average pool, into a concatenation."""
    ios.reset_name()
    holder = ios.placeholder((shape[0] + 3, *shape[1:]))
    block = Block(holder.node, None, [], None)
    source = ios.pool2d(block, [[holder]], 'max', (3, 3), (1, 1), (1, 1)) if front else holder
    window = [[Value(source.node, 1, shape[0] + 1)]]
    parts = [ios.conv2d(block, window, oc, (1, 1), (stride, stride), (pad, pad), act=act)
             for oc, act in zip(channels, ('relu', 'identity', 'tanh', 'relu', 'sigmoid', 'relu'))]
    # (no second convolution: it would round sums that differ in their last bit to operands that differ by 2^-11 or 2^-8, beyond the tolerance)
    tail = ios.pool2d(block, [[parts[0]]], 'max', (3, 3), (1, 1), (1, 1))
    joined = [[v] for v in parts[1:]] + [[tail]]
    ios.identity(block, joined, is_exit=True)
    graph = Graph('heads', holder.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    if schedule == 'greedy':
        graph.greedy_schedule(8)
    else:
        graph.sequential_schedule()
    return graph


def in_order(ops):
    """The operations as they run: a batch ahead of the groups of its stage."""
    return [dict(op, stage=2 * op['stage'] + ('batch' not in op), group=0 if 'batch' in op else op['group']) for op in ops]


@pytest.mark.parametrize('name,batch,schedule', [('inception_v3', 2, 'sequential'), ('inception_v3', 1, 'greedy'), ('resnet50', 2, 'sequential'),
                                                 ('nasnet_mobile', 1, 'greedy'), ('randwire_small', 1, 'greedy'), ('squeezenet_1_1', 2, 'sequential')])
def test_batches_read_what_single_launches_read(name, batch, schedule):
    graph = getattr(ios.models, name)()
    if schedule == 'greedy':
        graph.greedy_schedule(8)
    else:
        graph.sequential_schedule()
    rt.set_option('arena_reuse', 0)
    plain = rt.plan_describe(graph, batch)
    expected = _simulate(plain)
    rt.set_option('host_plan_batches', 1)
    for reuse in (0, 1):
        rt.set_option('arena_reuse', reuse)
        ops = rt.plan_describe(graph, batch)
        assert [op['node'] for op in ops] == [op['node'] for op in plain]
        batched = [op for op in ops if 'batch' in op]
        assert (len(batched) > 20) == (name in ('inception_v3', 'nasnet_mobile'))
        for op, old in zip(ops, plain):   # nothing else moves, and a batch only ahead
            assert op['stage'] == old['stage'] or ('batch' in op and op['stage'] < old['stage'])
        for op in batched:
            assert all(other['stage'] == op['stage'] and other['reads'] == op['reads'] for other in batched if other['batch'] == op['batch'])
        order = [i for stage in sorted({o['stage'] for o in in_order(ops)}) for i, o in enumerate(in_order(ops)) if o['stage'] == stage]
        plain_order = [i for stage in sorted({o['stage'] for o in plain}) for i, o in enumerate(plain) if o['stage'] == stage]
        assert dict(zip(order, _simulate(in_order(ops)))) == dict(zip(plain_order, expected))
    rt.set_option('batch_convs', 0)
    assert not any('batch' in op for op in rt.plan_describe(graph, batch))


def test_a_view_that_its_stage_completes_is_not_read_ahead():
    """The producer and its readers in one group of a stage: the batch would run before the producer."""
    graph = heads((13, 9, 7), (16, 24, 8), 1, 0, 'sequential')
    rt.set_option('host_plan_batches', 1)
    assert sum('batch' in op for op in rt.plan_describe(graph, 2)) == 3
    block = graph.blocks[0]
    names = [name for stage in block.stages for group in stage for name in group]
    block.stages = [[names]]
    assert not any('batch' in op for op in rt.plan_describe(graph, 2))
    block.stages = [[names[:2]], [names[2:]]]   # the first reader beside the producer, the others later
    assert [op['stage'] for op in rt.plan_describe(graph, 2) if 'batch' in op] == [1, 1]


@pytest.mark.parametrize('batch', [16, 33])
def test_batches_among_parts_of_a_batch(batch):
    """Leading stages that work on parts of the batch hold batches too."""
    ios.reset_name()
    v = ios.placeholder((3, 131, 127))
    block = Block(v.node)
    a = ios.conv2d(block, [[v]], 21, (3, 3), (2, 2))
    b, c = (ios.conv2d(block, [[a]], oc, (1, 1)) for oc in (8, 30))
    d = ios.conv2d(block, [[b]], 12, (3, 3), (1, 1), (1, 1))
    ios.identity(block, [[d], [c]], is_exit=True)
    graph = Graph('t', v.node, [block])
    graph.sequential_schedule()
    rt.set_option('host_plan_batches', 1)
    ops = rt.plan_describe(graph, batch)
    assert sum('batch' in op and 'part_ends' in op for op in ops) == 2
    rt.set_option('arena_reuse', 0)
    assert _simulate_parts(ops, batch) == _simulate_parts(rt.plan_describe(graph, batch), batch)


# channels in, map, channels of the members, stride, padding, batch: members that end inside a quad, a tile and before one; more members than a
# launch holds; fewer pixels than a tile; more filters than inputs (the tiles run along the filters); strides and pixels beside the map
BATCHES = [(33, (9, 11), (64, 65, 3, 130), 1, 0, 5), (96, (17, 17), (20, 128, 33, 64, 40, 7), 1, 0, 3), (70, (2, 3), (96, 200), 1, 0, 1),
           (200, (7, 7), (300, 90, 150), 1, 0, 1), (65, (13, 8), (48, 31), 2, 1, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize('name,precision,key', POINT, ids=[n[0] for n in POINT])
def test_batches_equal_single_launches(name, precision, key):
    rt.set_option('autotune', 0)
    try:
        rt.set_option('precision', precision)
        rt.set_option('conv_variant', rt.device_info()['conv_variants'].index(name))
        for ic, side, channels, stride, pad, batch in BATCHES:
            graph = heads((ic, *side), channels, stride, pad, 'sequential')
            x = np.random.default_rng(ic).standard_normal((batch, *graph.enter_node.output_shape)).astype(np.float32)
            want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, batch)} if key else {}))
            outputs = []
            for batched in (1, 0):
                rt.set_option('batch_convs', batched)
                with rt.Session(graph, batch) as session:
                    session.load_weights()
                    session.set_input(x)
                    session.run()
                    outputs.append(session.output())
                    assert sum('batch' in op for op in session.describe()) == (len(channels) if batched else 0)
            assert_close(outputs[0], want, f'{name} {channels}')
            assert np.array_equal(outputs[0], outputs[1])   # one body, one order of sums
    finally:
        for option, value in (('conv_variant', -1), ('precision', 'fp32')):
            rt.set_option(option, value)


@pytest.mark.gpu
@pytest.mark.parametrize('schedule', ['sequential', 'greedy'])
@pytest.mark.parametrize('executor', ['fused', 'fused_graph', 'streams', 'graph'])
def test_measured_batches_under_every_executor(executor, schedule):
    """Measured choices, replayed passes and the stateless call, whose weights arrive while it works."""
    rt.set_option('autotune', 1)
    try:
        rt.set_option('executor', executor)
        graph = heads((384, 17, 17), (192, 160, 160, 192), 1, 0, schedule)
        rng = np.random.default_rng(1)
        with rt.Session(graph, 12) as session:
            session.load_weights()
            # (one after the other they take twice as long as together; beside each other the measurement decides)
            batched = sum('batch' in op for op in session.describe())
            assert batched == 4 or (batched == 0 and schedule == 'greedy')
            assert sum(launch['kernel'].startswith('conv_batch_kernel') for launch in session.launches()) == batched // 4
            for _ in range(3):
                x = rng.standard_normal((12, *graph.enter_node.output_shape)).astype(np.float32)
                session.set_input(x)
                session.run()
                want = ios_oracle.run(graph, x)
                assert_close(session.output(), want, f'{executor} {schedule}')
            assert len(session.profile_launches(0, 1)) == len(session.launches())
            session.run()
            assert_close(session.output(), want, 'after a profile')
        assert_close(rt.graph_inference(graph, 12, x), want, 'stateless')
    finally:
        for option, value in (('autotune', 0), ('executor', 'fused')):
            rt.set_option(option, value)


SAVED = '''
import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph
ios.reset_name()
holder = ios.placeholder((96, 20, 20))
block = Block(holder.node, None, [], None)
ios.identity(block, [[ios.conv2d(block, [[holder]], oc, (1, 1))] for oc in (64, 64)], is_exit=True)
graph = Graph('saved', holder.node, [block])
graph.sequential_schedule()
with rt.Session(graph, 8) as session:
    print('batched', [op['variant'] for op in session.describe() if 'batch' in op])
'''


@pytest.mark.gpu
def test_saved_batches(tmp_path):
    """A choice from a file is taken over; one that the measurement could not have made is measured again."""
    path = tmp_path / 'choices'
    package = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'inter-operator-scheduler_amd')
    env = dict(os.environ, IOS_TUNE_CACHE=str(path), PYTHONPATH=package)

    def run():
        done = subprocess.run([sys.executable, '-c', SAVED], env=env, capture_output=True, text=True, timeout=100)
        assert done.returncode == 0, done.stderr[-2000:]
        return done.stdout

    assert 'batched' in run()
    lines = path.read_text().splitlines()
    batch = [line for line in lines if line.startswith('batch\t')]
    assert len(batch) == 1
    for name, taken in (('x3p_m32n128_w1x4_u2', True), ('wb_p_m64n64_w2x2', False), ('x3w_m64n64_w4', False), ('', False)):
        path.write_text('\n'.join([line for line in lines if line not in batch] + [batch[0].rsplit('\t', 1)[0] + '\t' + name]) + '\n')
        assert (f"batched ['{name}', '{name}']" in run()) == taken
        assert sum(line.startswith('batch\t') for line in path.read_text().splitlines()) == (1 if taken else 2)
