"""Projections of few rows with what follows them (hipops_projection) against the oracle's operators one after the other, and the
plugin's groups against the same model run operator by operator.
Bounds: one rounding of the result and 1e-6 sqrt(k) for the fp32 sum of k products (three times that behind the SwiGLU, whose slope
stays below 1.1 and whose factors reach 2.5 here); the norm divides by a root mean square that carries the sum's error once more, and is
taken of the rounded sum, of which the last bit may fall either way: one more rounding."""
import numpy as np
import pytest

import openvino_contrib_amd.plugin_capi as P
from openvino_contrib_amd import device_case as H
from test_gpu_layer_ops import BF16, F16, F32, ROUND, download, ops, rope_tables, scaled_error, upload  # noqa: F401
from test_gpu_plugin_layer import storage

pytestmark = pytest.mark.gpu


def _weights(hip, rng, n, k, dtype):
    return [upload(hip, rng.standard_normal((x, k)) / np.sqrt(k), dtype) for x in n]


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("m,n,k,head,rotated", [(1, (64, 64, 64), 64, 64, 3), (4, (4096, 1024, 1024), 4096, 128, 3), (16, (256, 64, 64), 704, 64, 1),
                                                (17, (512, 128), 320, 128, 2), (64, (1024, 256, 256), 1024, 128, 3), (33, (192,), 192, 24, 1),
                                                (5, (104, 8), 128, 8, 0)])
def test_products_with_rotary_embedding(hip, ops, oracle, m, n, k, head, rotated, dtype):  # noqa: F811
    rng = np.random.default_rng(m + k)
    dx, x = upload(hip, rng.standard_normal((m, k)), dtype)
    w = _weights(hip, rng, n, k, dtype)
    cos, sin = rope_tables(rng, 2 * m + 3, head, False, head)
    positions = rng.permutation(2 * m + 3)[:m].astype(np.int32)
    dcos, dsin, dpos = (hip.DeviceBuffer.from_numpy(t) for t in (cos.astype(np.float32), sin.astype(np.float32), positions))
    workspace = hip.DeviceBuffer(32 << 20)
    for with_positions in (True, False):
        outs = [hip.DeviceBuffer(m * i * 2) for i in n]
        for o in outs:
            o.fill(0xFF)
        ops.projection(ops.PROJECTION_ROPE, dtype, m, k, n, dx, [b for b, _ in w], outs, workspace, rotated=rotated, head_size=head, table_dtype=F32,
                       table_row_stride=head, cos=dcos, sin=dsin, positions=dpos if with_positions else None)
        for i, size in enumerate(n):
            ref = oracle.matmul(x, w[i][1], False, True)
            if (rotated >> i) & 1:
                ref = oracle.rope(ref.reshape(m, size // head, head), cos, sin, positions if with_positions else None).reshape(m, size)
            assert scaled_error(download(hip, outs[i], dtype, (m, size)), ref) <= ROUND[dtype] + 2e-6 * np.sqrt(k)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (4, 4096, 4096), (15, 1000, 448), (64, 4096, 1024), (33, 16384, 128), (49, 264, 5376)])
def test_product_residual_and_norm(hip, ops, oracle, m, n, k, dtype):  # noqa: F811
    rng = np.random.default_rng(m + n + k)
    dx, x = upload(hip, rng.standard_normal((m, k)), dtype)
    (dw, w), = _weights(hip, rng, (n,), k, dtype)
    dr, r = upload(hip, rng.standard_normal((m, n)), dtype)
    dg, g = upload(hip, 1 + 0.1 * rng.standard_normal(n), dtype)
    workspace = hip.DeviceBuffer(32 << 20)
    ref = oracle.matmul(x, w, False, True) + r
    for norm in (True, False):
        out, normalised = hip.DeviceBuffer(m * n * 2), hip.DeviceBuffer(m * n * 2)
        out.fill(0xFF), normalised.fill(0xFF)
        ops.projection(ops.PROJECTION_ADD, dtype, m, k, (n,), dx, [dw], [out], workspace, residual=dr, gamma=dg if norm else None, gamma_dtype=dtype,
                       normalised=normalised if norm else None, eps=1e-5)
        assert scaled_error(download(hip, out, dtype, (m, n)), ref) <= ROUND[dtype] + 1e-6 * np.sqrt(k)
        if norm:
            assert scaled_error(download(hip, normalised, dtype, (m, n)), oracle.rms_norm(ref, g, 1e-5)) <= 3 * ROUND[dtype] + 2e-6 * np.sqrt(k)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("rows,n", [(65, 8), (300, 4096), (1000, 1000), (3, 16384), (70, 4104)])
def test_residual_and_norm_behind_a_product(hip, ops, oracle, rows, n, dtype):  # noqa: F811
    """The sum is the Add's bit for bit; the norm as a single RMS: fp32 and one rounding."""
    rng = np.random.default_rng(rows + n)
    (dp, p), (dr, r) = (upload(hip, rng.standard_normal((rows, n)), dtype) for _ in range(2))
    dg, g = upload(hip, 1 + 0.1 * rng.standard_normal(n), F32)
    out, normalised, alone = (hip.DeviceBuffer(rows * n * 2) for _ in range(3))
    out.fill(0xFF), normalised.fill(0xFF)
    ops.residual_norm(dp, dr, dg, out, normalised, rows, n, 1e-5, dtype, F32)
    ops.binary(0, dp, dr, alone, [rows, n], [rows, n], [rows, n], dtype)
    got = download(hip, out, dtype, (rows, n))
    np.testing.assert_array_equal(got, download(hip, alone, dtype, (rows, n)))
    assert scaled_error(download(hip, normalised, dtype, (rows, n)), oracle.rms_norm(got, g, 1e-5)) <= ROUND[dtype] + 1e-6
    with pytest.raises(ops.HipOpsError) as e:
        ops.residual_norm(dp, dr, dg, out, normalised, rows, n + 4, 1e-5, dtype, F32)
    assert e.value.status == hip.UNSUPPORTED


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("m,width,k,activation,gate_first", [(1, 4, 64, 0, True), (4, 14336, 4096, 0, True), (16, 100, 320, 1, False), (33, 1376, 512, 2, True),
                                                             (64, 11008, 256, 0, False), (20, 44, 704, 0, True), (61, 14340, 128, 0, True),
                                                             (25, 16420, 64, 0, False)])
def test_product_and_glu(hip, ops, oracle, m, width, k, activation, gate_first, dtype):  # noqa: F811
    rng = np.random.default_rng(m + width + k)
    dx, x = upload(hip, rng.standard_normal((m, k)), dtype)
    (dw, w), = _weights(hip, rng, (2 * width,), k, dtype)
    out = hip.DeviceBuffer(m * width * 2)
    out.fill(0xFF)
    ops.projection(ops.PROJECTION_GLU, dtype, m, k, (2 * width,), dx, [dw], [out], activation=activation, gate_first=gate_first)
    ref = oracle.glu(oracle.matmul(x, w, False, True), activation, gate_first)
    assert scaled_error(download(hip, out, dtype, (m, width)), ref) <= ROUND[dtype] + 3e-6 * np.sqrt(k)


def test_what_the_kernels_do_not_take_is_refused(hip, ops):  # noqa: F811
    buf, ws = hip.DeviceBuffer(1 << 20), hip.DeviceBuffer(1 << 20)
    for kwargs, status in ((dict(rows=65), hip.UNSUPPORTED), (dict(k=96), hip.UNSUPPORTED), (dict(n=(12,)), hip.UNSUPPORTED), (dict(dtype=F32), hip.UNSUPPORTED),
                           (dict(workspace=None), hip.UNSUPPORTED), (dict(residual=None), hip.INVALID_ARGUMENT), (dict(kind=7), hip.INVALID_ARGUMENT),
                           (dict(gamma=buf, normalised=None), hip.INVALID_ARGUMENT), (dict(kind=ops.PROJECTION_GLU), hip.UNSUPPORTED)):
        call = dict(dict(kind=ops.PROJECTION_ADD, dtype=BF16, rows=8, k=64, n=(64,), x=buf, weights=[buf], outs=[buf], workspace=ws, residual=buf), **kwargs)
        with pytest.raises(ops.HipOpsError) as e:
            ops.projection(**call)
        assert e.value.status == status, kwargs


@pytest.mark.parametrize("m,n,k,taken", [(8, 7160, 1536, True), (8, 7160, 1600, False), (8, 7168, 2048, True), (1, 7168, 2112, False), (9, 8, 2048, True), (32, 11000, 2112, False),
                                         (33, 4088, 1600, False), (33, 4096, 2048, True), (64, 11008, 2112, True), (64, 512, 8192, False), (4, 28672, 4096, True)])
def test_glu_behind_a_long_k_goes_operator_by_operator(hip, ops, m, n, k, taken):  # noqa: F811
    """Either side of the lines: weights of few rows on a long k are a product in parts and an operator."""
    x, w, out = hip.DeviceBuffer(m * k * 2), hip.DeviceBuffer(n * k * 2), hip.DeviceBuffer(m * n)
    x.fill(0), w.fill(0), out.fill(0xFF)
    call = lambda: ops.projection(ops.PROJECTION_GLU, BF16, m, k, (n,), x, [w], [out])
    if not taken:
        with pytest.raises(ops.HipOpsError) as e:
            call()
        assert e.value.status == hip.UNSUPPORTED
    else:
        call()
    assert (download(hip, out, BF16, (m, n // 2)) == 0).all() == taken


def _model(tokens, hidden, ffn, heads, kv_heads, size, extra_reader):
    """norm -> q, k, v -> RoPE of q and k -> (their parts put together, as far as they are wide) -> o -> Add -> norm -> gate|up -> GLU -> down -> Add."""
    rng = np.random.default_rng(tokens + hidden)
    g = P.GraphText("projections")
    const = lambda name, shape, std: g.constant(name, storage(rng.standard_normal(shape) * std, BF16)[0], "bf16")
    weight = lambda name, rows, cols: const(name, (rows, cols), cols ** -0.5)
    mm = lambda name, x, w: g.add("MatMul", name, [x, w], transpose_a=False, transpose_b=True)
    rms = lambda name, x: g.add("RMS", name, [x, const(name + "_gamma", (hidden,), 1.0)], epsilon=1e-5, output_type="dynamic")
    x = g.parameter("x", BF16, [-1, hidden])
    cos, sin, pos = g.parameter("cos", F32, [-1, size]), g.parameter("sin", F32, [-1, size]), g.parameter("positions", P.I32, [-1])
    n1 = rms("norm1", x)
    q, k, v = (mm(n, n1, weight("w" + n, h * size, hidden)) for n, h in (("q", heads), ("k", kv_heads), ("v", kv_heads)))
    rope = dict(head_size=size, rotary_ndims=size, gather_position_arg_id=3)
    qr = g.add("RoPE", "rope_q", [q, cos, sin, pos], head_cnt=heads, **rope)
    kr = g.add("RoPE", "rope_k", [k, cos, sin, pos], head_cnt=kv_heads, **rope)
    kv = g.add("Multiply", "kv", [kr, v])
    if extra_reader:
        g.result("q_before", q)  # (read outside: what is between must be written)
    o = g.add("Add", "residual1", [mm("o", qr, weight("wo", hidden, heads * size)), x])
    act = g.add("GLU", "glu", [mm("gate_up", rms("norm2", o), weight("wgu", 2 * ffn, hidden))], axis=-1, split_lengths=ffn, glu_type=0, split_to_glu_idx=0,
                output_type="dynamic")
    g.result("out", g.add("Add", "residual2", [o, mm("down", act, weight("wd", hidden, ffn))]))
    g.result("kv_out", kv)
    return g.model()


@pytest.mark.parametrize("extra_reader", [False, True])
@pytest.mark.parametrize("hidden,ffn,heads,kv_heads,size", [(256, 704, 4, 2, 64), (384, 320, 3, 3, 128)])
def test_groups_of_the_plugin(hip, extra_reader, hidden, ffn, heads, kv_heads, size):
    """One compiled model over batches that a group takes, declines and takes again (the third and fourth infer of a size replay a graph),
    against the operators one by one (a model compiled for profiling).  Both round to bf16 at most eleven times on the way to an output;
    the norms keep every intermediate at one or below, so that three roundings' worth is ample."""
    plugin, timed = P.Plugin(), P.Plugin()
    timed.set_property("PERF_COUNT", "YES")
    text = _model(0, hidden, ffn, heads, kv_heads, size, extra_reader)
    requests = [p.compile_model(text).create_infer_request() for p in (plugin, timed)]
    rng = np.random.default_rng(1)
    for tokens in (1, 6, 7, 64, 65, 33, 64):
        x = storage(rng.standard_normal((tokens, hidden)), BF16)[0]
        cos, sin = rope_tables(rng, tokens + 9, size, False, size)
        pos = rng.permutation(tokens + 9)[:tokens].astype(np.int32)
        results = []
        for request in requests:
            for _ in range(4):
                for i, value in enumerate(((x, BF16), (cos.astype(np.float32), F32), (sin.astype(np.float32), F32), (pos, P.I32))):
                    request.set_input(i, *value)
                request.infer()
            results.append([H.storage_to_f32(request.output(i)[0], BF16) for i in range(3 if extra_reader else 2)])
        for got, ref in zip(*results):
            assert np.isfinite(ref).all() and scaled_error(got, ref) <= 6 * ROUND[BF16], tokens


def test_norms_over_a_part_of_their_inputs_are_refused(hip, ops):  # noqa: F811
    m, n, k = 16, 512, 64
    size = m * n * 2
    memory, ws = hip.DeviceBuffer(8 * size), hip.DeviceBuffer(1 << 20)
    memory.fill(0)

    class At:
        nbytes = size

        def __init__(self, offset):
            self.ptr = type(memory.ptr)(memory.ptr.value + offset)

    x, w, product, residual, gamma = At(0), At(size), At(2 * size), At(3 * size), At(5 * size)
    free, other = At(6 * size), At(7 * size)
    for out, normalised, taken in ((free, other, True), (free, residual, True), (residual, other, True), (free, At(3 * size + 1024), False),
                                   (free, At(4 * size), True), (free, At(2 * size + 16), False), (At(5 * size - 1024), other, False), (gamma, other, False),
                                   (At(5 * size + 1024), other, True)):
        calls = (lambda: ops.residual_norm(product, residual, gamma, out, normalised, m, n, 1e-5, BF16, BF16),
                 lambda: ops.projection(ops.PROJECTION_ADD, BF16, m, k, (n,), x, [w], [out], ws, residual=residual, gamma=gamma, gamma_dtype=BF16,
                                        normalised=normalised, eps=1e-5))
        for call in calls:
            if taken:
                call()
                continue
            with pytest.raises(ops.HipOpsError) as e:
                call()
            assert e.value.status == hip.UNSUPPORTED
    hip.DeviceBuffer(16).download(np.uint8, (1,))  # (waits for what was launched)


def _bind(request, inputs, outputs):
    for i, (buffer, dtype, shape, offset) in enumerate(inputs):
        request.set_device_input(i, buffer.ptr.value + offset, dtype, shape)
    for i, (buffer, dtype, shape, offset) in enumerate(outputs):
        request.set_device_output(i, buffer.ptr.value + offset, dtype, shape)


@pytest.mark.parametrize("tokens", [8, 64, 66, 6000])
@pytest.mark.parametrize("where", ["sum over the residual", "norm over the residual", "norm half the rows behind the residual", "sum over gamma"])
def test_norm_group_with_results_over_its_inputs(hip, where, tokens):
    """The caller's device tensors may overlap as far as the operators one by one allow: against the same model run that way."""
    n, k, row = 1024, 256, 2048
    rng = np.random.default_rng(tokens)
    g = P.GraphText("over")
    x, r, gamma = g.parameter("x", BF16, [-1, k]), g.parameter("residual", BF16, [-1, n]), g.parameter("gamma", BF16, [n])
    y = g.add("MatMul", "mm", [x, g.constant("w", storage(rng.standard_normal((n, k)) / 16, BF16)[0], "bf16")], transpose_a=False, transpose_b=True)
    total = g.add("Add", "sum", [y, r])
    g.result("norm", g.add("RMS", "rms", [total, gamma], epsilon=1e-5, output_type="dynamic"))
    g.result("total", total)
    text = g.text()
    xs, rs, gs = (storage(rng.standard_normal(shape), BF16)[0] for shape in ((tokens, k), (tokens, n), (n,)))
    results = []
    for profiled in (False, True):
        plugin = P.Plugin()
        if profiled:
            plugin.set_property("PERF_COUNT", "YES")
        request = plugin.compile_model(P.Model.from_text(text)).create_infer_request()
        # one allocation: [x][residual][half as many rows more][gamma, rows of space behind it][free, free]
        at = [0, tokens * k * 2]
        at += [at[1] + tokens * 3 // 2 * row]
        at += [at[2] + tokens * row, at[2] + 2 * tokens * row]
        memory = hip.DeviceBuffer(at[4] + tokens * row)
        image = np.zeros(memory.nbytes, np.uint8)
        for offset, a in zip(at, (xs, rs, gs)):
            image[offset:offset + a.nbytes] = a.reshape(-1).view(np.uint8)
        outs = {"sum over the residual": (at[4], at[1]), "norm over the residual": (at[1], at[3]), "norm half the rows behind the residual": (at[1] + tokens // 2 * row, at[3]),
                "sum over gamma": (at[4], at[2])}[where]
        _bind(request, [(memory, BF16, [tokens, k], at[0]), (memory, BF16, [tokens, n], at[1]), (memory, BF16, [n], at[2])],
              [(memory, BF16, [tokens, n], o) for o in outs])
        for _ in range(3):
            memory.upload(image)
            request.infer()
            after = memory.download(np.uint8, (memory.nbytes,))
            results.append([H.storage_to_f32(after[o:o + tokens * row].view(np.uint16), BF16) for o in outs])
        memory.free()
    for got in results[:3]:
        for a, b in zip(got, results[3]):
            assert np.isfinite(b).all() and scaled_error(a, b) <= 3 * ROUND[BF16]


@pytest.mark.parametrize("tokens", [4, 33, 64])
@pytest.mark.parametrize("shift", [0, -512, 512])
def test_glu_group_with_its_result_over_its_input(hip, tokens, shift):
    """Through the plugin: the result's device tensor is (in part) the input's, which the product of every column reads."""
    k = 256
    rng = np.random.default_rng(tokens)
    g = P.GraphText("over")
    x = g.parameter("x", BF16, [-1, k])
    y = g.add("MatMul", "mm", [x, g.constant("w", storage(rng.standard_normal((2 * k, k)) / 16, BF16)[0], "bf16")], transpose_a=False, transpose_b=True)
    g.result("out", g.add("GLU", "glu", [y], axis=-1, split_lengths=k, glu_type=0, split_to_glu_idx=0, output_type="dynamic"))
    request = P.Plugin().compile_model(g.model()).create_infer_request()
    xs = storage(rng.standard_normal((tokens, k)), BF16)[0]
    size = tokens * k * 2
    memory, apart = hip.DeviceBuffer(size + 1024), hip.DeviceBuffer(size)
    results = []
    for out in ((apart, BF16, [tokens, k], 0), (memory, BF16, [tokens, k], 512 + shift)):
        _bind(request, [(memory, BF16, [tokens, k], 512)], [out])
        for _ in range(3):
            image = np.zeros(size + 1024, np.uint8)
            image[512:512 + size] = xs.reshape(-1).view(np.uint8)
            memory.upload(image)
            request.infer()
            whole = out[0].download(np.uint8, (out[0].nbytes,))
            results.append(H.storage_to_f32(whole[out[3]:out[3] + size].view(np.uint16), BF16))
    for got in results[1:3]:
        np.testing.assert_array_equal(got, results[0])
    for got in results[3:]:
        assert scaled_error(got, results[0]) <= 3 * ROUND[BF16]
