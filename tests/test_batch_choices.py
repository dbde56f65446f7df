"""What the measurement compares that decides on shared launches: convolutions as they run otherwise, those of one stage beside each other and
those of different stages one after the other, on the kernels and launches that the executor then takes."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

PROGRAM = '''
import numpy as np
import ios
from ios.contrib import ios_runtime as rt
from test_conv_batches import heads
from test_gpu_parity import assert_close, ios_oracle
graph = heads(*SHAPE, 1, 0, 'sequential')
block = graph.blocks[0]
names = [name for stage in block.stages for group in stage for name in group]
block.stages = [[[n] for n in names[first:first + WIDTH]] if 1 <= first < 5 else [[names[first]]] for first in [0, *range(1, 5, WIDTH), *range(5, len(names))]]
rt.set_option('executor', EXECUTOR)
x = np.random.default_rng(1).standard_normal((BATCH, *graph.enter_node.output_shape)).astype(np.float32)
with rt.Session(graph, BATCH) as session:
    session.load_weights()
    session.set_input(x)
    for _ in range(3):
        session.run()
        assert_close(session.output(), ios_oracle.run(graph, x), EXECUTOR)
    print('shared', sum('batch' in op for op in session.describe()))
'''


def run(path, executor, width, shape=((384, 17, 17), (192, 160, 160, 192)), batch=12):
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, IOS_TUNE_CACHE=str(path), PYTHONPATH=os.path.join(os.path.dirname(here), 'inter-operator-scheduler_amd') + ':' + here)
    done = subprocess.run([sys.executable, '-c', f'EXECUTOR, WIDTH, SHAPE, BATCH = {executor!r}, {width}, {shape!r}, {batch}\n' + PROGRAM], env=env, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr[-2000:]
    return done.stdout


@pytest.mark.parametrize('executor', ['fused', 'streams', 'graph'])
@pytest.mark.parametrize('width,stages', [(1, None), (2, ['0', '0', '1', '1']), (4, ['0'] * 4)])
def test_stages_are_told_apart(tmp_path, executor, width, stages):
    """A choice for convolutions beside each other is none for the same ones in stages of their own."""
    path = tmp_path / 'choices'
    run(path, executor, width)
    line, = [line for line in path.read_text().splitlines() if line.startswith('batch\t') and 'mixed' not in line]
    members = line.split('\t')[1].split(' | ')[1:]
    assert [m.split('@')[1] if '@' in m else None for m in members] == (stages or [None] * 4)


def test_wide_registers_beside_1024_threads(tmp_path):
    """No fused launch holds both, so that such a level is launched one by one: that is measured, and takes longer than a shared launch."""
    path = tmp_path / 'choices'
    run(path, 'fused', 4)
    lines = [line.split() for line in path.read_text().splitlines() if not line.startswith('batch\t')]
    heads = [line for line in lines if line[1] == '384' and line[5] == '1']
    assert len(heads) == 2   # (two shapes, each twice)
    for line, name in zip(heads, ('wq_m16n16_w16_t16', 'x3w_m64n32_w4')):
        line[13:] = [name, '1'] * 4
    path.write_text('\n'.join(' '.join(line) for line in lines) + '\n')
    assert 'shared 4' in run(path, 'fused', 4)
    assert 'none' not in [line.split('\t')[2] for line in path.read_text().splitlines() if line.startswith('batch\t') and 'mixed' not in line]


@pytest.mark.parametrize('executor', ['streams', 'graph'])
def test_sums_in_slices_beside_each_other(tmp_path, executor):
    """Slices of K that meet in the L2 of one XCD: which one it is depends on the stream, and on a captured fork nobody knows."""
    path = tmp_path / 'choices'
    shape, batch = ((640, 8, 8), (96, 64, 128, 80)), 2
    run(path, executor, 4, shape, batch)
    lines = [line.split() for line in path.read_text().splitlines() if not line.startswith('batch\t')]
    heads = [line for line in lines if line[1] == '640']
    assert len(heads) == 4
    for line in heads:
        line[13:] = ['wq_m32n32_w4_t16', '4'] * 4
    path.write_text('\n'.join(' '.join(line) for line in lines) + '\n')
    run(path, executor, 4, shape, batch)
    assert sum(line.startswith('batch\t') and 'mixed' not in line for line in path.read_text().splitlines()) == 1   # (measured again)
