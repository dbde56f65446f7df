"""The threads that share out copies of host memory: compiled by themselves, no GPU involved."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'inter-operator-scheduler_amd', 'csrc')


@pytest.mark.skipif(shutil.which('g++') is None, reason='no host compiler')
def test_a_failing_copy_leaves_the_threads_in_order(tmp_path):
    program = str(tmp_path / 'check')
    subprocess.run(['g++', '-std=c++17', '-O1', '-g', '-pthread', '-I', CSRC, os.path.join(ROOT, 'tests', 'host_copier_check.cpp'),
                    os.path.join(CSRC, 'host_copier.cpp'), '-o', program], check=True)
    result = subprocess.run([program], capture_output=True, text=True, timeout=120)
    assert result.returncode == 0, result.stdout + result.stderr
