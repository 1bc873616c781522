"""GPU parity (through the C ABI) of the packed product on the matrix cores, nine rows of activations and more: the
oracle's dense reconstruction multiplied in float64."""

import numpy as np
import pytest
import torch

from oracle import scaling

import helpers

pytestmark = pytest.mark.gpu

F32 = np.float32
INT4 = scaling.int_values(4)
SEVEN = np.array([-1, -0.5, -0.25, 0, 0.25, 0.5, 1], dtype=F32)
# name -> (values, bits, integer)
CODECS = {"int4": (INT4, 4, True), "nf4": (scaling.NF4_VALUES, 4, False), "seven": (SEVEN, 3, False),
          "int3": (scaling.int_values(3), 3, True), "int2": (scaling.int_values(2), 2, True),
          "int8": (scaling.int_values(8), 8, True)}
# An output is rounded once to x's type (2^-12 / 2^-9 of it).
RANGE_TOLERANCE = {torch.float16: 1e-3, torch.bfloat16: 8e-3}


def run(layer, x, bias=None, scale_dtype=torch.float16):
    from mlkit_amd import native

    def device(array, dtype):
        return None if array is None else torch.from_numpy(np.ascontiguousarray(array)).to(device="cuda", dtype=dtype)

    rows, width = layer["shape"]
    packed, scales = device(layer["packed"], torch.uint8), device(layer["scales"], scale_dtype)
    zeros, values = device(layer["zero"], scale_dtype), device(layer["values"], torch.float32)
    y = torch.full((x.shape[0], rows), float("nan"), dtype=x.dtype, device="cuda")
    uniform = int(np.allclose(np.diff(layer["values"]), layer["values"][1] - layer["values"][0]))
    minimum, step = float(layer["values"][0]), float(layer["values"][1] - layer["values"][0])
    status = native.library().mk_packed_matmul(
        x.data_ptr(), native.dtype_code(x), packed.data_ptr(), scales.data_ptr(), native.dtype_code(scales), values.data_ptr(),
        values.numel(), native.pointer(zeros), native.pointer(bias), 0 if bias is None else native.dtype_code(bias), y.data_ptr(),
        x.shape[0], rows, width, layer["group"], layer["bits"], uniform, minimum, step, native.current_stream(x.device))
    native.check(status)
    torch.cuda.synchronize()
    return y


def check(y, layer, x, bias=None):
    expected = x.double().cpu().numpy() @ layer["dense"].astype(np.float64).T
    if bias is not None:
        expected = expected + bias.double().cpu().numpy()
    error = np.abs(y.double().cpu().numpy() - expected).max() / np.abs(expected).max()
    assert error <= RANGE_TOLERANCE[y.dtype], error


@pytest.mark.parametrize("name,rows,width,group,samples,asym", [
    # one tile of each kind, every format, rows / columns / samples that do not fill it
    ("int4", 1, 32, 64, 9, False),
    ("int4", 77, 416, 128, 17, True),
    ("int4", 130, 1056, 256, 33, False),        # a scale for two steps of 128 columns, a ragged last group
    ("int4", 100, 160, 160, 128, True),         # one scale a row
    ("int4", 66, 4096 + 96, 64, 40, False),     # two groups a step, the last step half empty
    ("nf4", 31, 224, 64, 16, False),
    ("nf4", 40, 384, 128, 65, True),            # a table with offsets
    ("seven", 50, 672, 64, 20, False),          # 48 bits a lane, from 2-byte boundaries
    ("int3", 35, 2080, 128, 48, True),          # three dwords a lane
    ("int2", 48, 352, 64, 10, False),
    ("int2", 33, 288, 128, 96, True),
    ("int8", 47, 544, 128, 31, True),
    ("int8", 20, 192, 64, 12, False),
    # the tiles the launch chooses among: 2 x 1, 2 x 2, 4 x 1, 4 x 2, two workgroups of 2 x 4 on a compute unit
    ("int4", 4096 + 5, 64, 64, 17, False),
    ("int4", 4000, 256, 128, 64, False),
    ("nf4", 14336, 64, 64, 16, False),
    ("int4", 14336, 128, 128, 32, True),
    ("int8", 8200, 128, 128, 100, False),
    ("int4", 20000, 32, 32, 16, False),         # more tiles than compute units at 4 x 1 and at 4 x 2
    ("int3", 20000, 64, 64, 30, False),
    # eight wavefronts of many steps
    ("int4", 96, 18944, 128, 24, True),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_product_matches_the_dense_reconstruction(name, rows, width, group, samples, asym, dtype):
    values, bits, integer = CODECS[name]
    layer = helpers.quantised_layer(helpers.normal_weight(rows, width, seed=rows + width), values, bits=bits, group=group,
                                    integer=integer, asym=asym)
    x = helpers.activations(samples, width, seed=samples, dtype=dtype).cuda()
    bias = torch.randn(rows, generator=torch.Generator().manual_seed(3)).to(device="cuda", dtype=dtype) if rows % 2 else None
    check(run(layer, x, bias), layer, x, bias)


def test_bf16_scales_and_activations_with_a_common_offset():
    """The operands carry an offset that sums of x cancel: activations far from zero mean keep the tolerance."""
    layer = helpers.quantised_layer(helpers.normal_weight(64, 1024, seed=5), INT4, bits=4, group=128, integer=True, fmt="bf16")
    for dtype in (torch.float16, torch.bfloat16):
        x = (helpers.activations(20, 1024, seed=1, dtype=torch.float32) + 3).to(dtype).cuda()
        check(run(layer, x, scale_dtype=torch.bfloat16), layer, x)


WIDE = np.array([-1, -0.3, -0.11, -0.03, -0.011, -0.003, -0.0011, 0, 0.0007, 0.0023, 0.007, 0.023, 0.07, 0.23, 0.7, 1], dtype=F32)
FITTED3 = np.array([-1, -0.61, -0.33, -0.1, 0.1, 0.33, 0.61, 0.97], dtype=F32)


@pytest.mark.parametrize("values,bits,group,asym", [
    (scaling.NF4_VALUES, 4, 64, False), (scaling.NF4_VALUES, 4, 128, True), (WIDE, 4, 128, False),
    (scaling.NF4_VALUES * F32(2.0e-6), 4, 64, False), (scaling.NF4_VALUES * F32(3.0e6), 4, 2048, False),   # past fp16's range
    (FITTED3, 3, 64, False), (FITTED3, 3, 128, True), (np.array([-1, -0.31, 0.31, 1], dtype=F32), 2, 64, False),
])
@pytest.mark.parametrize("samples", [9, 40])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_activations_with_a_mean_on_values_their_type_does_not_hold(values, bits, group, asym, samples, dtype):
    """Weights of one code share the error of its value, which activations of one sign add up: with both parts of a value
    (2^-17 of it and better) nothing but the rounding of an output remains, half a unit of at most 2^-8 / 2^-11 of it; an
    eighth of that is left for the sums."""
    layer = helpers.quantised_layer(helpers.normal_weight(64, 4096, seed=bits), values, bits=bits, group=group, integer=False, asym=asym)
    x = torch.relu(helpers.activations(samples, 4096, seed=samples, dtype=torch.float32)).to(dtype).cuda()
    y = run(layer, x).double().cpu().numpy()
    expected = x.double().cpu().numpy() @ layer["dense"].astype(np.float64).T
    half_unit = 2.0**-9 if dtype == torch.bfloat16 else 2.0**-12
    assert np.linalg.norm(y - expected) <= 1.125 * half_unit * np.linalg.norm(expected)


@pytest.mark.parametrize("name,held", [("nf4", False), ("seven", True), ("int3", True), ("int2", True)])
def test_a_wrong_statement_about_a_table_costs_time_and_not_digits(name, held):
    """`values_held` chooses the kernel with one operand a value; over a table that needs two, it works its outputs out
    by their definition."""
    import mlkit_amd as mk

    values, bits, _ = CODECS[name]
    linear = torch.nn.Linear(640, 70, bias=False, device="cuda", dtype=torch.bfloat16)
    layer = mk.PackedLinear(linear, mk.scaled(mk.grid.values(values.tolist(), bits=bits), group=64)(linear.weight.detach()))
    assert layer.values_held is held
    x = torch.relu(torch.randn((33, 640), device="cuda")).bfloat16()
    dense = torch.empty((70, 640), device="cuda")
    layer.storage_dtype = torch.float32
    dense.copy_(layer.weight)
    expected = (x.double() @ dense.double().T)
    for stated in (True, False):
        layer.values_held = stated
        layer._launch = None
        with torch.no_grad():
            y = layer._product(x, 33)
        assert (y.double() - expected).norm() <= 1.125 * 2.0**-9 * expected.norm()


def test_refuses_what_it_does_not_take():
    layer = helpers.quantised_layer(helpers.normal_weight(16, 96, seed=5), INT4, bits=4, group=32, integer=True)
    x = helpers.activations(16, 96, seed=1).cuda()
    with pytest.raises(ValueError, match="scale groups"):
        run(layer, x)
    with pytest.raises(ValueError, match="fp16 or bf16 activations"):
        run(layer, x.float())


@pytest.mark.parametrize("samples", [9, 128, 129, 300])
def test_packed_linear_on_both_sides_of_the_row_limit(samples):
    import mlkit_amd as mk

    torch.manual_seed(samples)
    linear = torch.nn.Linear(512, 320, device="cuda", dtype=torch.bfloat16)
    packed = mk.PackedLinear(linear, mk.int(4, 128, asym=True)(linear.weight.detach()))
    x = torch.randn(3, samples // 3, 512, device="cuda", dtype=torch.bfloat16)[:, :, :] if samples % 3 == 0 else \
        torch.randn(1, samples, 512, device="cuda", dtype=torch.bfloat16)
    expected = torch.nn.functional.linear(x.float(), packed.weight.float(), packed.bias.float())
    with torch.no_grad():
        y = packed(x)
    assert y.shape == expected.shape
    # the decoded weight is rounded to bf16 (2^-9 relative), the output once more
    assert ((y.float() - expected).norm() / expected.norm()).item() < 6e-3
    x.requires_grad_(True)
    packed(x).float().sum().backward()     # more than eight rows stay differentiable in the input
    assert torch.isfinite(x.grad).all()


@pytest.mark.parametrize("name,asym", [("int4", True), ("int4", False), ("nf4", False), ("seven", False), ("int2", True), ("int8", True)])
def test_infinite_activations_reach_the_outputs_as_in_a_dense_product(name, asym):
    values, bits, integer = CODECS[name]
    rng = np.random.default_rng(5)
    layer = helpers.quantised_layer(helpers.normal_weight(37, 224, seed=2), values, bits=bits, group=64, integer=integer, asym=asym)
    x = torch.from_numpy(rng.standard_normal((19, 224), dtype=F32)).to("cuda", torch.bfloat16)
    x[3, 7], x[4, 100], x[5, 9] = float("inf"), float("-inf"), float("nan")
    y = run(layer, x).double().cpu().numpy()
    with np.errstate(invalid="ignore"):
        expected = (x.double().cpu().numpy()[:, None, :] * layer["dense"].astype(np.float64)[None]).sum(-1)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(expected))
    np.testing.assert_array_equal(np.isinf(y) * np.sign(y), np.isinf(expected) * np.sign(expected))


@pytest.mark.parametrize("name,group,asym", [("int4", 128, True), ("nf4", 64, False), ("int3", 1184, True), ("int2", 64, False), ("int8", 128, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_outputs_by_their_definition_on_rows_of_several_pieces(name, group, asym, dtype):
    """Rows that are neither a whole number of 512 columns nor of tiles: infinities of one sign and of both in different
    pieces, a NaN in the last one, and finite activations whose products with operand and offset overflow although the
    outputs do not."""
    values, bits, integer = CODECS[name]
    layer = helpers.quantised_layer(helpers.normal_weight(37, 1184, seed=3), values, bits=bits, group=group, integer=integer, asym=asym)
    x = helpers.activations(21, 1184, seed=2, dtype=torch.float32)
    if dtype == torch.bfloat16:
        x[1] *= 1e36   # 128 columns times operands of 128 pass 2^128
    x = x.to(dtype)
    x[3, 1183], x[4, 0], x[4, 600], x[5, 511], x[6, 1183], x[20, 512] = (float(v) for v in ("inf", "inf", "-inf", "-inf", "nan", "inf"))
    y = run(layer, x.cuda()).double().cpu().numpy()
    with np.errstate(invalid="ignore"):
        expected = (x.double().numpy()[:, None, :] * layer["dense"].astype(np.float64)[None]).sum(-1)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(expected))
    np.testing.assert_array_equal(np.isinf(y) * np.sign(y), np.isinf(expected) * np.sign(expected))
    for sample in (0, 1, 2, 7, 19):
        error = np.abs(y[sample] - expected[sample]).max() / np.abs(expected[sample]).max()
        assert error <= RANGE_TOLERANCE[dtype], (sample, error)


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_an_activation_that_is_not_finite_does_not_make_a_call_a_slow_one(value):
    """One such row (a padded token behind a masked softmax) among 32: a few more microseconds, no other order of magnitude."""
    import mlkit_amd as mk

    linear = torch.nn.Linear(14336, 4096, bias=False, device="cuda", dtype=torch.bfloat16)
    layer = mk.PackedLinear(linear, mk.int(4, 128, asym=True)(linear.weight.detach()))
    finite = torch.randn((32, 14336), device="cuda", dtype=torch.bfloat16)
    other = finite.clone()
    other[3, 100] = value

    def microseconds(x):
        best = float("inf")
        with torch.no_grad():
            layer(x)
            for _ in range(10):
                start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                start.record()
                layer(x)
                stop.record()
                stop.synchronize()
                best = min(best, 1e3 * start.elapsed_time(stop))
        return best

    assert microseconds(other) <= 10 * microseconds(finite)


def test_calls_that_are_recorded_batched_differentiated_or_cast_take_the_dense_product():
    import torch.autograd.forward_ad as forward_ad

    import mlkit_amd as mk

    linear = torch.nn.Linear(256, 48, device="cuda", dtype=torch.float16)
    layer = mk.PackedLinear(linear, mk.int(4, 128)(linear.weight.detach()))
    x = torch.randn((17, 256), device="cuda", dtype=torch.float16)

    def dense(inputs):
        return torch.nn.functional.linear(inputs, layer.weight.to(inputs.dtype), layer.bias)

    stacked = torch.stack([x, 2 * x])
    assert torch.equal(torch.func.vmap(layer)(stacked), torch.func.vmap(dense)(stacked))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert layer(x).dtype == torch.bfloat16
    traced = torch.jit.trace(layer, (x,), check_trace=False)
    torch.testing.assert_close(traced(3 * x), dense(3 * x))
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(layer(forward_ad.make_dual(x, torch.ones_like(x))))
        torch.testing.assert_close(out.tangent, torch.nn.functional.linear(torch.ones_like(x), layer.weight))
    wanted = x.clone().requires_grad_()
    layer(wanted).sum().backward()
    assert wanted.grad is not None
    with pytest.raises(RuntimeError):
        layer(x.bfloat16())   # a bias of another type: refused, as the dense product refuses it


@pytest.mark.parametrize("cache_dense", [False, True])
def test_a_call_does_not_depend_on_the_calls_before_it(cache_dense):
    """A cached dense weight is asked for once and for all: from the first call of more than eight rows on it is there and
    used; without it, a longer call or a look at the weight changes nothing."""
    import mlkit_amd as mk

    linear = torch.nn.Linear(512, 320, device="cuda", dtype=torch.bfloat16)
    quantized = mk.int(4, 128, asym=True)(linear.weight.detach())
    layer = mk.PackedLinear(linear, quantized, cache_dense=cache_dense)
    x, longer = torch.randn((32, 512), device="cuda").bfloat16(), torch.randn((300, 512), device="cuda").bfloat16()
    with torch.no_grad():
        first = layer(x)
        assert (layer._dense_weight is not None) is cache_dense
        if cache_dense:
            assert torch.equal(first, torch.nn.functional.linear(x, layer.weight, layer.bias))
        layer(longer)
        layer.weight
        assert torch.equal(layer(x), first)


def test_a_layer_pickled_before_the_product_existed():
    import mlkit_amd as mk

    linear = torch.nn.Linear(512, 320, device="cuda", dtype=torch.bfloat16)
    layer = mk.PackedLinear(linear, mk.nf4(64)(linear.weight.detach()))
    state = layer.__getstate__()
    del state["maximum_product_rows"], state["values_held"]
    older = mk.PackedLinear.__new__(mk.PackedLinear)
    older.__setstate__(state)
    for rows in (3, 20):
        x = torch.randn((rows, 512), device="cuda").bfloat16()
        with torch.no_grad():
            assert torch.allclose(older(x).float(), layer(x).float(), rtol=2e-2, atol=2e-2)


def test_a_function_mode_sees_the_dense_product():
    """A mode that watches torch calls (a counter of operations, say) is shown `linear`, as before there was a product on
    the codes; a default device watches nothing and changes nothing."""
    from torch.overrides import TorchFunctionMode

    import mlkit_amd as mk

    class Watch(TorchFunctionMode):
        def __torch_function__(self, function, types, args=(), kwargs=None):
            seen.append(function)
            return function(*args, **(kwargs or {}))

    linear = torch.nn.Linear(512, 320, device="cuda", dtype=torch.bfloat16)
    layer = mk.PackedLinear(linear, mk.int(4, 128)(linear.weight.detach()))
    x = torch.randn((32, 512), device="cuda").bfloat16()
    seen = []
    with torch.no_grad():
        on_codes = layer(x)
        with Watch():
            watched = layer(x)
        assert torch.nn.functional.linear in seen or torch._C._nn.linear in seen
        assert torch.equal(watched, torch.nn.functional.linear(x, layer.weight, layer.bias))
        with torch.device("cuda"):
            assert torch.equal(layer(x), on_codes)


@pytest.mark.parametrize("rows,width,quantizer,limit", [
    (320, 512, "int4", 256), (320, 512, "nf4", 192), (320, 512, "int8", 192), (12800, 512, "int4", 128),   # up to 2^24 weights
    (4100, 4128, "int4", 128), (4100, 4128, "nf4", 64), (17000, 1024, "int4", 64), (2048, 8224, "seven", 128),
])
def test_which_calls_reach_the_product(rows, width, quantizer, limit):
    """Exactly the calls of 9 rows to the layer's limit are multiplied on their codes, and agree with the dense product."""
    import mlkit_amd as mk

    quantizers = {"int4": mk.int(4, 128), "nf4": mk.nf4(64), "int8": mk.int(8, 128), "seven": mk.scaled(mk.grid.values(SEVEN.tolist(), bits=3), group=64)}
    linear = torch.nn.Linear(width, rows, device="cuda", dtype=torch.float16)
    layer = mk.PackedLinear(linear, quantizers[quantizer](linear.weight.detach()))
    made = []
    product = layer._product
    layer._product = lambda inputs, samples: made.append(samples) or product(inputs, samples)
    for samples in (8, 9, limit, limit + 1):
        x = torch.randn((samples, width), device="cuda").half()
        with torch.no_grad():
            y = layer(x)
        expected = torch.nn.functional.linear(x.float(), layer.weight.float(), layer.bias.float())
        assert ((y.float() - expected).norm() / expected.norm()).item() < 2e-3
    assert made == [9, limit]


def test_bytes_on_a_fractional_grid_take_the_dense_product():
    """255 steps of a rounded length do not end on the last value: the error is one for all weights, so such layers stay
    with the decoded weight, whose own rounding hides part of it."""
    import mlkit_amd as mk

    linear = torch.nn.Linear(512, 64, bias=False, device="cuda", dtype=torch.float16)
    x = torch.relu(torch.randn((16, 512), device="cuda")).half()
    for values, taken in ((torch.linspace(-0.7, 1.1, 256), False), (torch.arange(-128.0, 128.0), True)):
        layer = mk.PackedLinear(linear, mk.scaled(mk.grid.values(values.tolist(), bits=8), group=None)(linear.weight.detach()))
        assert layer.uniform_grid and (layer.maximum_product_rows > 0) is taken
        if not taken:
            with torch.no_grad():
                assert torch.equal(layer(x), torch.nn.functional.linear(x, layer.weight))


def test_calls_the_library_refuses_take_the_dense_product():
    """Activations that start off 16 bytes, and scales that were cast to fp32 after the layer was built."""
    import mlkit_amd as mk

    linear = torch.nn.Linear(512, 320, device="cuda", dtype=torch.float16)
    layer = mk.PackedLinear(linear, mk.int(4, 128)(linear.weight.detach()))
    x = torch.randn(20 * 512 + 1, device="cuda").half()[1:].view(20, 512)
    with torch.no_grad():
        assert layer._product(x, 20) is None
        assert torch.equal(layer(x), torch.nn.functional.linear(x, layer.weight, layer.bias))
        aligned = x.clone()
        expected = layer(aligned).float()
        layer.float()
        assert layer.scales.dtype == torch.float32
        torch.testing.assert_close(layer(aligned.float()), expected, rtol=2e-3, atol=2e-3)
        layer.bias = layer.bias.half()
        assert layer._product(aligned, 20) is None
        torch.testing.assert_close(layer(aligned).float(), expected, rtol=2e-3, atol=4e-3)
