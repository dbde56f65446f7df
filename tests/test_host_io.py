"""Transfers between a caller's arrays and the device at the sizes where the paths of csrc/host_io.hip change over."""
import gc
import time

import numpy as np
import pytest

import ios
from ios.contrib import ios_runtime as rt
from ios.ir import Graph

pytestmark = pytest.mark.gpu


def relu_graph(channels, height, width):
    """y = max(x, 0): what comes back is what went there."""
    ios.reset_name()
    v = ios.placeholder((channels, height, width))
    block = ios.Block(v.node)
    ios.relu(block, [[v]], is_exit=True)
    graph = Graph('t', v.node, [block])
    graph.sequential_schedule()
    return graph


# floats: one value; the ends of one-kernel results (16 KB, 64 KB) and of results fetched by one thread; uploads in one, in several
# and in shared-out steps; the largest result a pass delivers and the largest upload a kernel pulls (4 MB); beyond both
@pytest.mark.parametrize('floats', [1, 4095, 4096, 4097, 16383, 16385, 49152, 49153, 65537, 98305, 393215, 393217, 1 << 20, (1 << 20) + 1, 3000001])
def test_input_and_result_of_every_size(floats):
    session = rt.Session(relu_graph(1, 1, floats) if floats < 65536 else relu_graph(floats // 65536 + 1, 256, 256), 1)
    rng = np.random.default_rng(floats)
    for _ in range(3):   # delivered, delivered again, and after a result that nobody fetched
        x = rng.standard_normal(session.input_shape, dtype=np.float32)
        session.set_input(x)
        session.run()
        assert np.array_equal(session.output(), np.maximum(x, 0))
    session.run()
    session.set_input(-x)
    session.run()
    assert np.array_equal(session.output(), np.maximum(-x, 0))


@pytest.mark.parametrize('batch', [16, 17, 23, 64])
@pytest.mark.parametrize('executor', ['fused', 'fused_graph', 'streams', 'graph'])
def test_batches_arrive_in_parts(batch, executor):
    """Leading stages on the parts of a batch, against the same images one by one."""
    rt.set_option('executor', executor)
    rt.set_option('autotune', 0)
    try:
        ios.reset_name()
        v = ios.placeholder((3, 161, 159))
        block = ios.Block(v.node)
        w = ios.conv2d(block, [[v]], 19, (3, 3), (2, 2))
        w = ios.pool2d(block, [[w]], 'max', (3, 3), (2, 2))
        w = ios.conv2d(block, [[w]], 33, (3, 3), (1, 1), (1, 1))
        ios.pool2d(block, [[w]], 'global_avg', is_exit=True)
        graph = Graph('t', v.node, [block])
        graph.init_weights(seed=1, scheme='he_normal_bias')
        graph.sequential_schedule()
        session, single = rt.Session(graph, batch), rt.Session(graph, 1)
        session.load_weights()
        single.load_weights()
        rng = np.random.default_rng(batch)
        for _ in range(2):
            x = rng.standard_normal(session.input_shape, dtype=np.float32)
            session.set_input(x)
            session.run()
            got = session.output()
            session.run()   # the same input again, now resident
            assert np.array_equal(got, session.output())
            for i in (0, batch // 2 - 1, batch // 2, batch // 2 + 1, batch - 1):
                single.set_input(x[i:i + 1])
                single.run()
                assert np.allclose(got[i:i + 1], single.output(), rtol=1e-4, atol=1e-5)
    finally:
        rt.set_option('executor', 'fused')
        rt.set_option('autotune', 1)


@pytest.mark.parametrize('no_alloc', [False, True])
def test_inference_calls_take_turns(no_alloc):
    """Networks, batches, weights and inputs change from call to call; every call computes with its own."""
    graphs = []
    for width in (20, 33, 48, 64, 70, 96):   # more documents than plans are kept
        ios.reset_name()
        v = ios.placeholder((5, 14, 15))
        block = ios.Block(v.node)
        a = ios.conv2d(block, [[v]], width, (3, 3), (1, 1), (1, 1))
        b = ios.conv2d(block, [[v]], 24, (1, 1))
        ios.conv2d(block, [[a], [b]], 17, (1, 1), is_exit=True)
        graph = Graph('t', v.node, [block])
        graph.greedy_schedule(4)
        graphs.append(graph)
    for step in range(14):
        graph, batch = graphs[(step * step) % 6], 1 + step % 3
        graph.init_weights(seed=step, scheme='he_normal_bias')
        x = np.random.default_rng(step).standard_normal((batch, 5, 14, 15)).astype(np.float32)
        got = rt.graph_inference(graph, batch, x, no_alloc=no_alloc)
        session = rt.Session(graph, batch)
        session.load_weights()
        session.set_input(x)
        session.run()
        assert np.allclose(got, session.output(), rtol=1e-4, atol=1e-5)
        session.close()


# beyond what a pass delivers, in one and in several parts, ends of parts inside images, planes and quads of channels
@pytest.mark.parametrize('batch,shape', [(5, (37, 101, 103)), (2, (1, 1024, 1031)), (2100, (501, 1, 1)), (3, (350, 32, 32)), (70001, (15, 1, 1))])
def test_large_results_of_several_images(batch, shape):
    """A tensor that shares its pixels with another one's channels, and a result that does not fit the pass's delivery."""
    ios.reset_name()
    v = ios.placeholder(shape)
    block = ios.Block(v.node)
    a = ios.relu(block, [[v]])
    b = ios.pool2d(block, [[v]], 'max', (1, 1), (1, 1), (0, 0))
    ios.identity(block, [[a], [b]], is_exit=True)
    graph = Graph('t', v.node, [block])
    graph.sequential_schedule()
    x = np.random.default_rng(batch).standard_normal((batch, *shape), dtype=np.float32)
    with rt.Session(graph, batch) as session:
        session.set_input(x)
        session.run()
        want = np.concatenate([np.maximum(x, 0), x], axis=1)
        assert np.array_equal(session.output(), want)
        assert np.array_equal(session.tensor(a.node), want[:, :shape[0]])
        assert np.array_equal(session.tensor(b.node), want[:, shape[0]:])


# three parts; five parts, which take 32 MB and more
@pytest.mark.parametrize('batch,side', [(17, 161), (64, 225), (61, 231)])
@pytest.mark.parametrize('executor', ['fused', 'fused_graph'])
def test_tensors_of_a_batch_that_arrived_in_parts(batch, side, executor):
    """The result and every tensor that can be asked for, among them those that a pass on parts holds for one part at a time."""
    rt.set_option('executor', executor)
    rt.set_option('autotune', 0)
    try:
        ios.reset_name()
        v = ios.placeholder((3, side, side - 2))
        block = ios.Block(v.node)
        a = ios.conv2d(block, [[v]], 19, (3, 3), (2, 2))
        b = ios.pool2d(block, [[a]], 'max', (3, 3), (1, 1), (1, 1))
        c = ios.conv2d(block, [[a], [b]], 26, (3, 3), (2, 2))
        d = ios.conv2d(block, [[c]], 33, (3, 3), (1, 1), (1, 1))
        ios.pool2d(block, [[d], [c]], 'global_avg', is_exit=True)
        graph = Graph('t', v.node, [block])
        graph.init_weights(seed=1, scheme='he_normal_bias')
        graph.sequential_schedule()
        parts = [op['part_ends'] for op in rt.plan_describe(graph, batch) if 'part_ends' in op]
        assert parts and len(parts[0]) == (5 if batch * 3 * side * (side - 2) >= 8 << 20 else 3)
        with rt.Session(graph, batch) as session, rt.Session(graph, 1) as single:
            session.load_weights()
            single.load_weights()
            x = np.random.default_rng(batch).standard_normal(session.input_shape, dtype=np.float32)
            for step in range(2):
                x = x[::-1].copy()
                session.set_input(x)
                session.run()
                got = session.output()
                held = []
                for value in (a, b, c, d):
                    try:
                        tensor = session.tensor(value.node)
                    except RuntimeError as e:
                        assert 'shares its memory' in str(e)
                        continue
                    held.append(value)
                    for i in (0, batch // 3, batch - 1):
                        single.set_input(x[i:i + 1])
                        single.run()
                        try:
                            assert np.allclose(tensor[i:i + 1], single.tensor(value.node), rtol=1e-4, atol=1e-5)
                        except RuntimeError as e:
                            assert 'shares its memory' in str(e)
                        assert np.allclose(got[i:i + 1], single.output(), rtol=1e-4, atol=1e-5)
                assert held and np.array_equal(got, session.output())
                session.run()   # the same input again, now resident
                assert np.array_equal(got, session.output())
            # a timed pass and a profile work on the whole batch, also where the input has only just been set
            for profile in (lambda: session.measure(0, 1, 1, profile_stage=True), session.profile_ops, session.profile_launches):
                session.set_input(x)
                profile()
                tensors = [session.tensor(value.node) for value in held]
                session.run()
                assert held and all(np.array_equal(t, session.tensor(value.node)) for t, value in zip(tensors, held))
                assert np.array_equal(got, session.output())
            # an input that no pass has worked on: tensors of the last pass are there or are refused, the result is the last pass's
            session.set_input(-x)
            session.run()
            negative = session.output()
            session.set_input(x)
            for value in (a, b, c, d):
                try:
                    session.tensor(value.node)
                except RuntimeError as e:
                    assert 'shares its memory' in str(e) or 'changed since' in str(e)
            assert np.array_equal(negative, session.output())
            session.run()
            assert np.array_equal(got, session.output())
    finally:
        rt.set_option('executor', 'fused')
        rt.set_option('autotune', 1)


def test_an_input_beyond_the_staging_buffer():
    """335 MB go through the 256 MB buffer in two groups of images."""
    session = rt.Session(relu_graph(1, 4096, 4096), 5)
    x = np.random.default_rng(5).standard_normal(session.input_shape, dtype=np.float32)
    for _ in range(2):
        x = -x
        session.set_input(x)
        session.run()
        assert np.array_equal(session.output(), np.maximum(x, 0))
    session.close()


@pytest.mark.parametrize('floats', [4096, 65537, 640000])
def test_sessions_take_turns(floats):
    """A result that a pass has delivered stays there until another pass delivers one, whatever passes run in between."""
    channels = floats // 65536 + 1
    first, second, large = (rt.Session(relu_graph(c, h, w), 1) for c, h, w in
                            ((1, 1, floats) if floats < 65536 else (channels, 256, 256), (channels, 256, 255), (17, 256, 257)))
    rng = np.random.default_rng(floats)
    x, y, z = (rng.standard_normal(s.input_shape, dtype=np.float32) for s in (first, second, large))
    for session, data in ((first, x), (second, y), (large, z)):
        session.set_input(data)
        session.run()
        assert np.array_equal(session.output(), np.maximum(data, 0))
    for step in range(4):
        first.set_input(x + step)
        first.run()
        if step % 2:
            large.run()     # too large to be delivered
            second.enqueue()
            second.synchronize()
        if step == 3:
            second.run()    # delivers: the first one's result is copied from its own tensor
        assert np.array_equal(first.output(), np.maximum(x + step, 0))
        assert np.array_equal(first.output(), np.maximum(x + step, 0))
        assert np.array_equal(second.output(), np.maximum(y, 0))
        assert np.array_equal(large.output(), np.maximum(z, 0))


def test_a_delivered_result_is_fetched_at_once_after_passes_that_deliver_nothing():
    """2.5 MB, 40 chunks: the wait for chunks of another pass would take half a millisecond for each."""
    first, large = rt.Session(relu_graph(10, 256, 256), 1), rt.Session(relu_graph(17, 256, 257), 1)
    x = np.random.default_rng(0).standard_normal(first.input_shape, dtype=np.float32)
    first.set_input(x)
    times = []
    for _ in range(12):
        first.run()
        large.run()
        start = time.perf_counter()
        y = first.output()
        times.append(time.perf_counter() - start)
        assert np.array_equal(y, np.maximum(x, 0))
    assert min(times) < 2e-3, times


def test_host_threads():
    """Copies shared out over other numbers of threads, the caller alone among them."""
    try:
        for threads in (1, 2, 5, 0):
            rt.set_option('host_threads', threads)
            assert threads == 0 or rt.device_info()['host_threads'] == threads
            test_input_and_result_of_every_size(3000001)
            test_input_and_result_of_every_size(98305)
        with pytest.raises(RuntimeError, match='host_threads'):
            rt.set_option('host_threads', -1)
    finally:
        rt.set_option('host_threads', 0)


def test_staging_memory_goes_with_the_last_session():
    """67 MB of input: its staging buffer stays while there is a session, and shrinks to 16 MB at most behind the last one."""
    gc.collect()
    rt.set_option('release_staging', 1)
    assert rt.device_info()['staged_bytes'] <= 32 << 20
    small, large = rt.Session(relu_graph(1, 1, 100), 1), rt.Session(relu_graph(1, 4096, 4096), 1)
    x = np.random.default_rng(0).standard_normal(large.input_shape, dtype=np.float32)
    for _ in range(2):
        large.set_input(x)
        large.run()
        assert np.array_equal(large.output(), np.maximum(x, 0))
    assert rt.device_info()['staged_bytes'] >= 64 << 20
    large.close()
    assert rt.device_info()['staged_bytes'] >= 64 << 20
    small.close()
    assert rt.device_info()['staged_bytes'] <= 32 << 20
    with rt.Session(relu_graph(1, 4096, 4096), 1) as again:
        again.set_input(-x)
        again.run()
        assert np.array_equal(again.output(), np.maximum(-x, 0))
    # inference calls alone keep it, also where an option makes them plan anew
    graph = relu_graph(1, 4096, 4096)
    for _ in range(2):
        assert np.array_equal(rt.graph_inference(graph, 1, x), np.maximum(x, 0))
        assert rt.device_info()['staged_bytes'] >= 64 << 20
        rt.set_option('executor', 'fused')
        assert rt.device_info()['staged_bytes'] >= 64 << 20
    rt.set_option('release_staging', 1)
    assert rt.device_info()['staged_bytes'] <= 32 << 20
    assert np.array_equal(rt.graph_inference(graph, 1, -x), np.maximum(-x, 0))
    rt.set_option('release_staging', 1)
