"""Which infers replay a graph and which run operator by operator although they repeat (gpu): launch-bound models keep the graph whatever
large tensors they hold but do not read, and so do models of many operators; a few operators whose kernels outlast their launches go without."""
import numpy as np
import pytest

import openvino_contrib_amd.plugin_capi as P
from openvino_contrib_amd import device_case as H
from test_gpu_plugin_layer import BF16, F32, rope_tables, storage

pytestmark = pytest.mark.gpu

KINDS = ["embedding", "rotary tables", "views", "adds that the caches hold", "long products", "many long products"]


def _model(hip, kind, rng):
    """-> (model text, [(input, device buffer or host array, type, shape)], reference or None)"""
    g = P.GraphText(kind.replace(" ", "_"))
    if kind == "rotary tables":  # 25 MB each, named by every operator
        x_st, x = storage(rng.standard_normal((4, 128)), BF16)
        cos, sin = (hip.DeviceBuffer(50000 * 128 * 4) for _ in range(2))
        cos.fill(0), sin.fill(0)
        inputs = [(hip.DeviceBuffer.from_numpy(x_st), BF16, [4, 128]), (cos, F32, [50000, 128]), (sin, F32, [50000, 128]),
                  (hip.DeviceBuffer.from_numpy(np.arange(4, dtype=np.int32)), P.I32, [4])]
        y = g.parameter("x", BF16, [4, 128])
        c, s, p = g.parameter("cos", F32, [50000, 128]), g.parameter("sin", F32, [50000, 128]), g.parameter("positions", P.I32, [4])
        for i in range(12):
            y = g.add("RoPE", "rope%d" % i, [y, c, s, p], head_cnt=1, head_size=128, rotary_ndims=128, gather_position_arg_id=3)
        g.result("out", y)
        return g, inputs, np.zeros((4, 128), np.float32)
    if kind.endswith("long products"):
        x_st, _ = storage(rng.standard_normal((8, 4096)), BF16)
        w = hip.DeviceBuffer(4096 * 4096 * 2)
        w.fill(0)
        y, weight = g.parameter("x", BF16, [8, 4096]), g.parameter("w", BF16, [4096, 4096])
        for i in range(40 if kind.startswith("many") else 7):
            y = g.add("MatMul", "mm%d" % i, [y, weight], transpose_a=False, transpose_b=True)
        g.result("out", y)
        return g, [(hip.DeviceBuffer.from_numpy(x_st), BF16, [8, 4096]), (w, BF16, [4096, 4096])], np.zeros((8, 4096), np.float32)
    if kind == "adds that the caches hold":  # 12 MB to an operator, but the host takes longer to launch it
        n, count = 1 << 20, 32
        y, one = g.parameter("x", F32, [n]), g.parameter("one", F32, [n])
        for i in range(count):
            y = g.add("Add", "add%d" % i, [y, one])
        g.result("out", y)
        ones = np.ones(n, np.float32)
        return g, [(hip.DeviceBuffer.from_numpy(ones), F32, [n]), (hip.DeviceBuffer.from_numpy(ones), F32, [n])], ones * (count + 1)
    # 100 MB of table, of which a step reads four rows
    table = hip.DeviceBuffer(100000 * 256 * 4)
    table.fill(0)
    ids = np.array([3, 99999, 0, 7], np.int32)
    one = np.ones((4, 256), np.float32)
    y = g.parameter("table", F32, [100000, 256])
    if kind == "views":
        for i in range(4):
            shape = [256, 100000] if i % 2 == 0 else [100000, 256]
            y = g.add("Reshape", "view%d" % i, [y, g.constant("shape%d" % i, np.array(shape, np.int64), "i64")], special_zero=False)
    y = g.add("Gather", "rows", [y, g.parameter("ids", P.I32, [4]), g.constant("axis", np.array(0, np.int64), "i64")], batch_dims=0)
    b = g.parameter("one", F32, [4, 256])
    for i in range(8):
        y = g.add("Add", "add%d" % i, [y, b])
    g.result("out", y)
    return g, [(table, F32, [100000, 256]), (hip.DeviceBuffer.from_numpy(ids), P.I32, [4]), (hip.DeviceBuffer.from_numpy(one), F32, [4, 256])], 8 * one


@pytest.mark.parametrize("kind", KINDS)
def test_what_replays_a_graph(hip, kind):
    g, inputs, ref = _model(hip, kind, np.random.default_rng(3))
    compiled = P.Plugin().compile_model(g.model())
    request = compiled.create_infer_request()
    for i, (buffer, dtype, shape) in enumerate(inputs):
        request.set_device_input(i, buffer.ptr, dtype, shape)
    for _ in range(4):
        request.infer()
        out, dtype = request.output(0)
        np.testing.assert_array_equal(H.storage_to_f32(out, dtype), ref)
    graphs, launches = (int(compiled.get_property(name)) for name in ("HIP_NUMBER_OF_GRAPHS", "HIP_GRAPH_LAUNCHES"))
    assert (graphs, launches) == ((0, 0) if kind == "long products" else (1, 3))
    for buffer, _, _ in inputs:
        buffer.free()
