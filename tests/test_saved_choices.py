"""Kernel configurations from a file: one that names two-term operands for a small K, as a file may that was written when the name
stood for three terms, is measured again, as is one that the tuner does not measure for the shape, or that cannot be read; others are
taken over."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

PROGRAM = '''
import sys
import numpy as np
import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block
ios.reset_name()
holder = ios.placeholder((int(sys.argv[1]), 9, 11))
block = Block(holder.node, None, [], None)
ios.conv2d(block, [[holder]], 40, (1, 1), is_exit=True)
graph = ios.Graph('point', holder.node, [block])
graph.init_weights(3, 'he_normal')
graph.sequential_schedule()
with rt.Session(graph, 2) as session:
    session.load_weights()
    print('variant', [op['variant'] for op in session.describe() if op['kind'] == 'conv_mfma'][0])
'''


@pytest.mark.parametrize('channels,taken', [(63, False), (64, True)])
def test_two_terms_for_a_small_k(tmp_path, channels, taken):
    path = tmp_path / 'choices'
    path.write_text(f'2 {channels} 9 11 40 1 1 1 1 0 0 1 cost/1024/xcd' + ' x3w_m64n64_w4 1' * 4 + '\n')
    package = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'inter-operator-scheduler_amd')
    env = dict(os.environ, IOS_TUNE_CACHE=str(path), PYTHONPATH=package)
    done = subprocess.run([sys.executable, '-c', PROGRAM, str(channels)], env=env, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr[-2000:]
    assert ('variant x3w_m64n64_w4' in done.stdout) == taken, done.stdout
    assert len(path.read_text().splitlines()) == (1 if taken else 2)   # (a shape that was measured is appended)


# three terms where the tuner measures two; one it leaves out; one that cannot compute a filter of one tap; numbers that no shape has
@pytest.mark.parametrize('shape,name', [('', 'x3_m64n128_w2x2'), ('', 'm64n64k32_w2x2x1_t32'), ('', 'x3_win_m64n128_w1x4_d'), ('2 0 9 11 40 1 1 0 0 0 0 0', 'x3w_m64n64_w4')])
def test_choices_of_other_builds(tmp_path, shape, name):
    path = tmp_path / 'choices'
    path.write_text((shape or '2 64 9 11 40 1 1 1 1 0 0 1') + ' cost/1024/xcd' + f' {name} 1' * 4 + '\n')
    package = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'inter-operator-scheduler_amd')
    env = dict(os.environ, IOS_TUNE_CACHE=str(path), PYTHONPATH=package)
    done = subprocess.run([sys.executable, '-c', PROGRAM, '64'], env=env, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr[-2000:]
    assert 'variant ' in done.stdout and f'variant {name}\n' not in done.stdout, done.stdout
    assert len(path.read_text().splitlines()) == 2
