"""The line that bench.py prints holds what was measured to seven digits."""
import json

import bench


def test_numbers_keep_seven_digits():
    result = {'value': 2815.651781346316, 'n': 20, 'ok': True, 'none': None, 'name': 'x 1', 'nested': [{'ms': 0.3551575541496277, 'flops': 1.234567891e11}, (1.0, -2.5e-7)]}
    line = bench.result_line(result)
    assert '\n' not in line
    back = json.loads(line)
    assert back['value'] == 2815.652 and back['nested'][0] == {'ms': 0.3551576, 'flops': 123456800000.0} and back['nested'][1] == [1.0, -2.5e-7]
    assert back['n'] == 20 and back['ok'] is True and back['none'] is None and back['name'] == 'x 1'
