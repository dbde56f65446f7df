"""Images that reach the device in the host's layout: rows of planes that begin anywhere in a line of memory, at the edges of the
tiles in which they are turned.  A network that copies its input hands every value back."""
import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Block, Graph

pytestmark = pytest.mark.gpu

# channels, map, batch: one to four channels and more (tiles of 32 channels x 240 pixels): pixels that end before, at and
# behind a tile and a line; bands of a single large image; many small ones; a batch that arrives in parts
CASES = [(1, (1, 1), 1), (3, (5, 7), 4), (3, (32, 32), 2), (4, (25, 41), 3), (2, (31, 33), 5), (3, (299, 299), 2), (3, (701, 523), 1), (1, (900, 901), 1),
         (5, (1, 1), 3), (33, (15, 16), 2), (32, (16, 15), 1), (64, (13, 37), 3), (131, (37, 53), 3), (31, (241, 3), 2), (300, (61, 47), 1), (7, (3, 3), 70), (3, (131, 127), 17)]


@pytest.mark.parametrize('channels,side,batch', CASES)
def test_every_value_arrives_at_its_place(channels, side, batch):
    ios.reset_name()
    holder = ios.placeholder((channels, *side))
    block = Block(holder.node, None, [], None)
    largest = ios.pool2d(block, [[holder]], 'max', (1, 1))
    ios.identity(block, [[largest]], is_exit=True)
    graph = Graph('copy', holder.node, [block])
    graph.sequential_schedule()
    with rt.Session(graph, batch) as session:
        for seed in range(3):
            x = np.random.default_rng(seed).standard_normal((batch, channels, *side)).astype(np.float32)
            session.set_input(x)
            session.run()
            assert np.array_equal(session.output(), x)
