"""Convolutions of parallel branches that share a launch, with a pool beside them: the plans on the host, and the kernels against single
launches and the oracle."""
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
from test_library import _simulate

STAGED = [(name, precision, key) for precision, prefixes, key in FAMILIES for name in rt.conv_variant_names()
          if name.startswith(prefixes[0]) or name.startswith(prefixes[0].split('_')[0].rstrip('p') + '_win_')]


@pytest.fixture(autouse=True)
def default_options():
    yield
    for key, value in (('batch_convs', 1), ('host_plan_batches', 0), ('arena_reuse', 1)):
        rt.set_option(key, value)


def branches(shape, windows, channels, schedule):
    """Convolutions that read two views in turn, one of them a window of channels, and a pool, beside each other."""
    ios.reset_name()
    holder = ios.placeholder((shape[0] + 3, *shape[1:]))
    block = Block(holder.node, None, [], None)
    views = [Value(ios.pool2d(block, [[holder]], 'max', (3, 3), (1, 1), (1, 1)).node, 1, shape[0] + 1),
             ios.pool2d(block, [[holder]], 'avg', (3, 3), (1, 1), (1, 1))]
    parts = [ios.conv2d(block, [[views[i % 2]]], oc, (kh, kw), (1, 1), (kh // 2, kw // 2), act=act)
             for i, ((kh, kw), oc, act) in enumerate(zip(windows, channels, ('relu', 'identity', 'tanh', 'relu')))]
    parts.append(ios.pool2d(block, [[views[1]]], 'avg', (3, 3), (1, 1), (1, 1)))
    ios.identity(block, [[v] for v in parts], is_exit=True)
    graph = Graph('branches', holder.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    if schedule == 'greedy':
        graph.greedy_schedule(8)
    else:
        graph.sequential_schedule()
    return graph


@pytest.mark.parametrize('name,batch,schedule', [('inception_v3', 2, 'sequential'), ('inception_v3', 1, 'greedy'), ('resnet50', 2, 'greedy'),
                                                 ('nasnet_mobile', 1, 'greedy'), ('randwire_small', 1, 'greedy'), ('squeezenet_1_1', 2, 'greedy')])
def test_mixed_launches_read_what_single_launches_read(name, batch, schedule):
    graph = getattr(ios.models, name)()
    if schedule == 'greedy':
        graph.greedy_schedule(8)
    else:
        graph.sequential_schedule()
    rt.set_option('arena_reuse', 0)
    plain = rt.plan_describe(graph, batch)
    expected = _simulate(plain)
    rt.set_option('host_plan_batches', 2)
    for reuse in (0, 1):
        rt.set_option('arena_reuse', reuse)
        ops = rt.plan_describe(graph, batch)
        assert [op['node'] for op in ops] == [op['node'] for op in plain]
        for op, old in zip(ops, plain):   # nothing else moves, and a shared launch only ahead
            assert op['stage'] == old['stage'] or ('batch' in op and op['stage'] < old['stage'])
        # (launches of a stage follow each other: a later one may read what an earlier one wrote)
        last = 1 + max(op.get('batch', 0) for op in ops)
        ordered = [dict(op, stage=op['stage'] * (last + 1) + op.get('batch', last), group=0 if 'batch' in op else op['group']) for op in ops]
        order = [i for stage in sorted({o['stage'] for o in ordered}) for i, o in enumerate(ordered) if o['stage'] == stage]
        plain_order = [i for stage in sorted({o['stage'] for o in plain}) for i, o in enumerate(plain) if o['stage'] == stage]
        assert dict(zip(order, _simulate(ordered))) == dict(zip(plain_order, expected))


def test_a_pool_joins_the_convolutions_beside_it():
    rt.set_option('host_plan_batches', 2)
    ops = rt.plan_describe(branches((16, 9, 9), [(1, 7), (7, 1), (3, 3)], (8, 9, 10), 'greedy'), 2)
    assert sorted(op['kind'] for op in ops if 'batch' in op) == ['conv_mfma'] * 3 + ['pool']
    ops = rt.plan_describe(branches((16, 9, 9), [(1, 7), (7, 1), (3, 3)], (8, 9, 10), 'sequential'), 2)
    assert [op['kind'] for op in ops if 'batch' in op] == ['conv_mfma'] * 2   # (those of one view)


# channels in, map, windows, channels of the members, batch, maps that shrink: members of one number of taps and of several; tiles that end
# inside a quad, before and behind an edge; fewer pixels than a tile, so that blocks of a member have none
MIXED = [(33, (9, 11), [(1, 7), (7, 1)], (64, 65), 3, False), (64, (13, 13), [(1, 9), (3, 3), (9, 1)], (130, 20, 96), 2, False),
         (48, (12, 10), [(1, 7), (3, 3), (5, 5), (1, 3)], (33, 64, 7, 128), 4, False), (65, (14, 13), [(5, 3), (3, 5)], (40, 100), 3, True)]


def one_view(shape, windows, channels, valid):
    """Convolutions of an odd window of channels, one after the other."""
    ios.reset_name()
    holder = ios.placeholder((shape[0] + 3, *shape[1:]))
    block = Block(holder.node, None, [], None)
    view = Value(ios.pool2d(block, [[holder]], 'max', (3, 3), (1, 1), (1, 1)).node, 1, shape[0] + 1)
    parts = [ios.conv2d(block, [[view]], oc, (kh, kw), (1, 1), (0, 0) if valid else (kh // 2, kw // 2), act=act)
             for (kh, kw), oc, act in zip(windows, channels, ('relu', 'identity', 'tanh', 'relu'))]
    if valid:   # (to one size again)
        parts = [ios.pool2d(block, [[v]], 'max', (7 - kh, 7 - kw), (1, 1), (0, 0)) for v, (kh, kw) in zip(parts, windows)]
    ios.identity(block, [[v] for v in parts], is_exit=True)
    graph = Graph('view', holder.node, [block])
    graph.init_weights(3, 'he_normal_bias')
    graph.sequential_schedule()
    return graph


@pytest.mark.gpu
@pytest.mark.parametrize('name,precision,key', STAGED, ids=[n[0] for n in STAGED])
def test_mixed_launches_equal_single_launches(name, precision, key):
    rt.set_option('autotune', 0)
    try:
        rt.set_option('precision', precision)
        rt.set_option('conv_variant', rt.device_info()['conv_variants'].index(name))
        rt.set_option('conv_split_k', 1)   # (a convolution by itself would split its sums)
        for ic, side, windows, channels, batch, valid in MIXED:
            graph = one_view((ic, *side), windows, channels, valid)
            x = np.random.default_rng(ic).standard_normal((batch, *graph.enter_node.output_shape)).astype(np.float32)
            outputs = []
            for shared in (1, 0):
                rt.set_option('batch_convs', shared)
                with rt.Session(graph, batch) as session:
                    session.load_weights()
                    session.set_input(x)
                    session.run()
                    outputs.append(session.output())
                    assert sum('batch' in op for op in session.describe()) == (len(channels) if shared else 0)
            want = ios_oracle.run(graph, x, **({key: matrix_path_convs(graph, batch)} if key else {}))
            assert_close(outputs[0], want, f'{name} {windows}')
            assert np.array_equal(outputs[0], outputs[1])   # one body, one order of sums
    finally:
        for option, value in (('conv_variant', -1), ('conv_split_k', 0), ('precision', 'fp32')):
            rt.set_option(option, value)


SAVED = '''
import numpy as np
from ios.contrib import ios_runtime as rt
from test_conv_mixed import branches
from test_gpu_parity import assert_close, ios_oracle, matrix_path_convs
for case in CASES:
    graph = branches(*case, 'greedy')
    x = np.random.default_rng(1).standard_normal((2, *graph.enter_node.output_shape)).astype(np.float32)
    rt.set_option('precision', PRECISION)
    want = ios_oracle.run(graph, x, **({KEY: matrix_path_convs(graph, 2)} if KEY else {}))
    with rt.Session(graph, 2) as session:
        session.load_weights()
        session.set_input(x)
        session.run()
        assert_close(session.output(), want, str(case))
        print('shared', [op.get('variant') for op in session.describe() if 'batch' in op])
'''


@pytest.mark.gpu
@pytest.mark.parametrize('name,precision,key', [n for n in STAGED if n[0] in ('x3p_m64n64_w2x2', 'x3_win_m64n128_w2x4_d', 'wb_win_m64n128_w1x4', 'wh_p_m64n64_w2x2')])
def test_saved_choices_of_mixed_launches(name, precision, key, tmp_path):
    """Members that read different views, and a pool, on a configuration that the file names."""
    path = tmp_path / 'choices'
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, IOS_TUNE_CACHE=str(path), PYTHONPATH=os.path.join(os.path.dirname(here), 'inter-operator-scheduler_amd') + ':' + here)
    cases = [((70, 9, 11), [(1, 7), (7, 1)], (64, 65)), ((64, 13, 12), [(3, 3), (3, 3), (3, 3)], (33, 20, 96)), ((80, 12, 10), [(1, 7), (3, 3), (1, 3)], (33, 64, 7))]
    code = f'CASES, PRECISION, KEY = {cases!r}, {precision!r}, {key!r}\n' + SAVED

    def run():
        done = subprocess.run([sys.executable, '-c', code], env=env, capture_output=True, text=True, timeout=100)
        assert done.returncode == 0, done.stderr[-2000:]
        return done.stdout

    run()
    lines = path.read_text().splitlines()
    assert sum(line.startswith('batch\tmixed ') for line in lines) >= len(cases)   # (those refused are asked for by view again)
    path.write_text('\n'.join(line.rsplit('\t', 1)[0] + '\t' + name if line.startswith('batch\tmixed ') else line for line in lines) + '\n')
    shared = run()
    for _, windows, _ in cases:   # (a pool goes along)
        assert f'shared {[name] * len(windows) + [None]}' in shared, shared


@pytest.mark.gpu
@pytest.mark.parametrize('executor', ['fused', 'fused_graph', 'streams', 'graph'])
def test_measured_mixed_launches_under_every_executor(executor):
    rt.set_option('autotune', 1)
    try:
        rt.set_option('executor', executor)
        graph = branches((192, 17, 17), [(1, 7), (7, 1)], (192, 192), 'greedy')
        rng = np.random.default_rng(1)
        with rt.Session(graph, 16) as session:
            session.load_weights()
            mixed = sum(launch['kernel'].startswith('conv_mixed_kernel') for launch in session.launches())
            assert mixed == 0 or executor.startswith('fused')   # (branches on streams run beside each other as they are)
            for _ in range(3):
                x = rng.standard_normal((16, *graph.enter_node.output_shape)).astype(np.float32)
                session.set_input(x)
                session.run()
                want = ios_oracle.run(graph, x)
                assert_close(session.output(), want, executor)
            assert len(session.profile_launches(0, 1)) == len(session.launches())
            session.run()
            assert_close(session.output(), want, 'after a profile')
        assert_close(rt.graph_inference(graph, 16, x), want, 'stateless')
    finally:
        for option, value in (('autotune', 0), ('executor', 'fused')):
            rt.set_option(option, value)
