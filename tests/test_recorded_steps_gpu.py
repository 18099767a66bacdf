"""Nodes of a recorded step that read one input share a launch: the bits of a call by itself, and only where nothing depends on the order."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth

pytestmark = pytest.mark.gpu


class Node:
    """A node over constant weights with its tensors on the GPU. `bias`: None, a broadcast [n], or a view of Y's shape."""

    def __init__(self, ep, k, n, bs, dt, seed, zero_points=True, bias=None, **attrs):
        self.ep, self.k, self.n, self.dt = ep, k, n, dt
        b, s, zp = synth.make_weights(n, k, bs, seed, zero_points=zero_points, scale_lo=0.002, scale_hi=0.01, scale_dtype=dt)
        self.tensors = [ep.upload(x) if x is not None else None for x in (b, s, zp)]
        view = lambda buf, code, shape: E.TensorView(buf.ptr, code, shape) if buf is not None else E.TensorView.absent(code)  # noqa: E731
        kb = -(-k // bs)
        self.rest = [view(self.tensors[0], E.U8, (n, kb, bs // 2)), view(self.tensors[1], dt, (n, kb)), view(self.tensors[2], E.U8, (n, (kb + 1) // 2)),
                     E.TensorView.absent(E.I32)]
        self.bias = bias
        if isinstance(bias, str):
            values = synth.to_dtype(np.random.default_rng(seed).standard_normal(n).astype(np.float32), dt)
            self.tensors.append(ep.upload(values))
            self.bias = E.TensorView(self.tensors[-1].ptr, dt, (n,))
        self.kernel = ep.get_kernel({"K": k, "N": n, "bits": 4, "block_size": bs, **attrs})
        self.kernel.set_constant_inputs([False, True, True, True])

    def __call__(self, x, y, m):
        inputs = [E.TensorView(x, self.dt, (m, self.k))] + self.rest + ([self.bias] if self.bias is not None else [])
        self.kernel.execute(inputs, [E.TensorView(y, self.dt, (m, self.n))])


def rows(ep, m, k, dt, seed):
    return ep.upload(synth.make_activation(m, k, seed, dt))


def recorded(ep, calls):
    """Runs the calls eagerly, then records them; -> the graph."""
    for node, x, y, m in calls:
        node(x, y, m)
    ep.sync()
    ep.capture_begin()
    for node, x, y, m in calls:
        node(x, y, m)
    return ep.capture_end()


def check(ep, calls, launches, outputs=None):
    """The graph has `launches` nodes and every replay leaves the bits of the eager calls in (address, bytes) of `outputs`."""
    outputs = outputs or [(y, m * node.n * 2) for node, _, y, m in calls]
    graph = recorded(ep, calls)

    def read():
        got = []
        for at, size in outputs:
            got.append(np.empty(size, np.uint8))
            ep.copy_to_host(got[-1], at)
        return got

    def clear():
        for at, size in outputs:
            ep.copy_from_host(at, np.full(size, 0x55, np.uint8))

    clear()
    for node, x, y, m in calls:
        node(x, y, m)
    want = read()
    assert graph.num_nodes == launches
    for _ in range(3):
        clear()
        graph.replay()
        ep.sync()
        for w, g in zip(want, read()):
            assert np.array_equal(w, g)
    graph.release()


@pytest.mark.parametrize("m", [1, 2, 4, 5, 16])
@pytest.mark.parametrize("dt,bs,k", [(E.F16, 32, 896), (E.BF16, 64, 4864), (E.BF16, 128, 1000), (E.F16, 128, 18944)])
def test_three_nodes_are_one_launch(ep, dt, bs, k, m):
    """Widths that end inside a column group, a bias of each kind."""
    x = rows(ep, m, k, dt, m)
    residual = rows(ep, m, 33, dt, m + 1)
    nodes = [Node(ep, k, 896, bs, dt, 1, bias="row"), Node(ep, k, 33, bs, dt, 2, bias=E.TensorView(residual.ptr, dt, (m, 33)), folded_bias=1), Node(ep, k, 130, bs, dt, 3, zero_points=False)]
    y = [ep.allocate(m * node.n * 2) for node in nodes]
    check(ep, [(node, x.ptr, out.ptr, m) for node, out in zip(nodes, y)], 1)


def test_four_nodes_fill_a_launch(ep):
    m, k, dt = 1, 896, E.F16
    x = rows(ep, m, k, dt, 0)
    nodes = [Node(ep, k, n, 32, dt, n) for n in (16, 48, 17, 128, 64)]
    y = [ep.allocate(m * node.n * 2) for node in nodes]
    check(ep, [(node, x.ptr, out.ptr, m) for node, out in zip(nodes, y)], 2)


@pytest.mark.parametrize("case", ["reads_result", "residual_is_result", "same_result", "results_overlap", "writes_input", "result_is_residual", "other_input", "other_rows", "other_k",
                                  "first_writes_input", "copy_between"])
def test_nodes_that_depend_on_each_other_stay_in_order(ep, case):
    m, k, n, bs, dt = 2, 896, 896, 32, E.F16
    pool = ep.upload(synth.make_activation(8 * m, k, 3, dt))
    at = lambda i: pool.ptr + i * m * k * 2                                        # noqa: E731
    first, second = Node(ep, k, n, bs, dt, 1), Node(ep, k, n, bs, dt, 2)
    calls = [(first, at(0), at(2), m), (second, at(0), at(3), m)]
    if case == "reads_result":
        calls[1] = (second, at(2), at(3), m)
    elif case == "residual_is_result":
        second.bias = E.TensorView(at(2), dt, (m, n))
    elif case == "same_result":
        calls[1] = (second, at(0), at(2), m)
    elif case == "results_overlap":
        calls[1] = (second, at(0), at(2) + m * n * 2 - 16, m)
    elif case == "writes_input":
        calls[1] = (second, at(0), at(0) + m * k * 2 - 16, m)
    elif case == "result_is_residual":
        first.bias = E.TensorView(at(3), dt, (m, n))
    elif case == "other_input":
        calls[1] = (second, at(1), at(3), m)
    elif case == "other_rows":
        calls[1] = (second, at(0), at(3), 1)
    elif case == "other_k":
        calls[1] = (Node(ep, 512, n, bs, dt, 2), at(0), at(3), m)
    elif case == "first_writes_input":
        calls[0] = (first, at(1), at(0), m)
    if case == "copy_between":
        for node, x, y, rows_ in calls:
            node(x, y, rows_)
        ep.sync()
        ep.capture_begin()
        first(at(0), at(2), m)
        ep.copy(E.DeviceBuffer(at(4), m * k * 2), E.DeviceBuffer(at(5), m * k * 2), m * k * 2)
        second(at(0), at(3), m)
        graph = ep.capture_end()
        assert graph.num_nodes == 3
        graph.release()
        return
    start = np.empty(8 * m * k * 2, np.uint8)
    ep.copy_to_host(start, pool)
    for node, x, y, rows_ in calls:                                                # (repacks the weights)
        node(x, y, rows_)
    ep.copy_from_host(pool, start)
    for node, x, y, rows_ in calls:
        node(x, y, rows_)
    want, got = np.empty_like(start), np.empty_like(start)
    ep.copy_to_host(want, pool)
    ep.capture_begin()
    for node, x, y, rows_ in calls:
        node(x, y, rows_)
    graph = ep.capture_end()
    assert graph.num_nodes == 2
    for _ in range(0 if case == "writes_input" else 3):                            # (a call that writes what it reads has no one result)
        ep.copy_from_host(pool, start)
        graph.replay()
        ep.copy_to_host(got, pool)
        assert np.array_equal(want, got)
    graph.release()


def test_a_step_of_layers(ep):
    """q, k, v / o / gate, up / down, twice, each reading what the node before it wrote: four launches a layer."""
    m, h, kv, inter, bs, dt = 1, 896, 128, 4864, 32, E.F16
    buffers = {"x": rows(ep, m, h, dt, 5)}
    calls, x = [], buffers["x"].ptr
    for layer in range(2):
        sizes = {"q": (h, h), "k": (h, kv), "v": (h, kv), "o": (h, h), "gate": (h, inter), "up": (h, inter), "down": (inter, h)}
        out = {name: ep.allocate(m * n * 2) for name, (_, n) in sizes.items()}
        buffers[layer] = out
        reads = {"q": x, "k": x, "v": x, "o": out["q"].ptr, "gate": out["o"].ptr, "up": out["o"].ptr, "down": out["gate"].ptr}
        for i, (name, (k, n)) in enumerate(sizes.items()):
            calls.append((Node(ep, k, n, bs, dt, 10 * layer + i), reads[name], out[name].ptr, m))
        x = out["down"].ptr
    check(ep, calls, 8)


@pytest.mark.parametrize("m,dt,bs", [(1, E.F16, 32), (3, E.BF16, 128), (9, E.BF16, 64)])
def test_a_chain_that_reads_weights_ahead(ep, m, dt, bs):
    """Each launch reads weights of the next: grids that do not end on a multiple of eight workgroups, next ones of fewer than eight, streams longer than a block's share, and pairs
    of nodes behind a launch."""
    widths = [896, 304, 72, 1000, 16, 4096, 896]
    buffers = [rows(ep, m, widths[0], dt, 5)] + [ep.allocate(m * n * 2) for n in widths[1:]]
    calls = [(Node(ep, k, n, bs, dt, i), buffers[i].ptr, buffers[i + 1].ptr, m) for i, (k, n) in enumerate(zip(widths, widths[1:]))]
    side = ep.allocate(m * 304 * 2)
    calls.insert(6, (Node(ep, 4096, 304, bs, dt, 9), buffers[5].ptr, side.ptr, m))
    check(ep, calls, 6)


@pytest.mark.parametrize("m,dt,bs", [(1, E.F16, 32), (3, E.BF16, 128), (16, E.BF16, 64)])
def test_a_narrow_node_may_come_first(ep, m, dt, bs):
    """k, v, q: the rows of the first nodes end long before the grid does."""
    k = 896
    x = rows(ep, m, k, dt, 7)
    nodes = [Node(ep, k, n, bs, dt, n, bias=bias) for n, bias in ((16, "row"), (130, None), (1000, "row"))]
    y = [ep.allocate(m * node.n * 2) for node in nodes]
    calls = [(node, x.ptr, out.ptr, m) for node, out in zip(nodes, y)]
    check(ep, calls, 1)
    before = ep.kernel_launch_count()
    graph = recorded(ep, calls)
    assert ep.kernel_launch_count() - before == 2 * len(calls)                     # (run once and recorded once; a recorded call counts whether or not it shares a launch)
    graph.release()
