"""Convolutions of parallel branches and the pool beside them in one launch, under every executor that holds such launches: passes one after the
other, replayed, timed launch by launch and stateless."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

PROGRAM = '''
import numpy as np
from ios.contrib import ios_runtime as rt
from test_conv_mixed import branches
from test_gpu_parity import assert_close, ios_oracle
graph = branches((70, 9, 11), [(1, 7), (7, 1)], (64, 65), 'greedy')
rng = np.random.default_rng(1)
for executor in ('fused', 'fused_graph'):
    rt.set_option('executor', executor)
    with rt.Session(graph, 3) as session:
        session.load_weights()
        print(executor, 'shared', sorted(op['kind'] for op in session.describe() if 'batch' in op))
        mixed = [launch['kernel'] for launch in session.launches() if launch['kernel'].startswith('conv_mixed_kernel')]
        print(executor, 'launches', len(mixed))
        for _ in range(4):
            x = rng.standard_normal((3, *graph.enter_node.output_shape)).astype(np.float32)
            want = ios_oracle.run(graph, x)
            session.set_input(x)
            for _ in range(2):
                session.run()
                assert_close(session.output(), want, executor)
        assert len(session.profile_launches(0, 1)) == len(session.launches())
        session.measure(1, 2, 1, profile_stage=True)
        assert_close(session.output(), want, executor + ', stages timed')
        session.run()
        assert_close(session.output(), want, executor + ', again')
    for _ in range(3):
        x = rng.standard_normal((3, *graph.enter_node.output_shape)).astype(np.float32)
        assert_close(rt.graph_inference(graph, 3, x), ios_oracle.run(graph, x), executor + ', stateless')
'''


@pytest.mark.parametrize('name', ['x3p_m64n64_w2x2', 'x3_win_m64n128_w2x4_d'])
def test_every_way_to_run_a_mixed_launch(name, tmp_path):
    path = tmp_path / 'choices'
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, IOS_TUNE_CACHE=str(path), PYTHONPATH=os.path.join(os.path.dirname(here), 'inter-operator-scheduler_amd') + ':' + here)

    def run():
        done = subprocess.run([sys.executable, '-c', PROGRAM], env=env, capture_output=True, text=True, timeout=100)
        assert done.returncode == 0, done.stderr[-2000:]
        return done.stdout

    run()
    lines = path.read_text().splitlines()
    path.write_text('\n'.join(line.rsplit('\t', 1)[0] + '\t' + name if line.startswith('batch\tmixed ') else line for line in lines) + '\n')
    shared = run()
    for executor in ('fused', 'fused_graph'):
        assert f"{executor} shared ['conv_mfma', 'conv_mfma', 'pool']" in shared and f'{executor} launches 1' in shared, shared
