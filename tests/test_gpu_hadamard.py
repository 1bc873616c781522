"""GPU parity (through the C ABI) of the Walsh-Hadamard kernels against the oracle:
bit for bit against the stage-by-stage fp32 restatement, to 1e-4 against the Sylvester
matrix product in float64 (the reference's own bound, tests/quantization/test_operations.py:99-100)."""

import numpy as np
import pytest
import torch

from oracle import transforms

pytestmark = pytest.mark.gpu

F32 = np.float32


def dev(array):
    return torch.from_numpy(np.ascontiguousarray(array)).cuda()


def host(tensor):
    torch.cuda.synchronize()
    return tensor.float().cpu().numpy()


@pytest.mark.parametrize("width", [1, 2, 4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 8192, 16384, 32768])
@pytest.mark.parametrize("normalize", [True, False])
def test_transform_is_bit_exact(width, normalize):
    from mlkit_amd.kernels import hadamard

    rng = np.random.default_rng(width)
    rows = 5 if width >= 4096 else 37
    value = rng.standard_normal((rows, width)).astype(F32)
    out = host(hadamard.transform(dev(value), normalize=normalize))
    np.testing.assert_array_equal(out, transforms.fwht(value, normalize))
    if width <= 2048:
        exact = value.astype(np.float64) @ transforms.sylvester(width)
        if normalize:
            exact = exact / np.sqrt(width)
        np.testing.assert_allclose(out, exact, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("width", [256, 512, 1024, 2048, 4096])
def test_register_transform_of_many_rows_is_bit_exact(width):
    """4096 fp32 rows and more take `fwht_rows_kernel` (a row in the registers of one wavefront, no
    LDS): the stagewise oracle on sampled rows, and the workgroup kernel (fewer rows per call) on
    all of them, bit for bit; with signs in front and behind whose period spans three rows."""
    from mlkit_amd.kernels import hadamard

    rows = 4098   # not a multiple of the four rows a workgroup takes
    generator = torch.Generator(device="cuda").manual_seed(width)
    value = torch.randn((rows, width), device="cuda", generator=generator)
    out = hadamard.transform(value)
    picked = [0, 1, 2, 3, 1000, 4095, 4096, 4097]
    np.testing.assert_array_equal(host(out[picked]), transforms.fwht(host(value[picked])))
    pieces = torch.cat([hadamard.transform(value[:2049].contiguous()), hadamard.transform(value[2049:].contiguous())])
    assert torch.equal(out, pieces)
    assert torch.equal(hadamard.transform(value, normalize=False)[:7], hadamard.transform(value[:7].contiguous(), normalize=False))
    signs = dev(transforms.deterministic_signs(3 * width, seed=2))
    blocks = value[: 4098 - 4098 % 3].view(-1, 3, width)
    signed = hadamard.transform(blocks, signs_before=signs, signs_after=signs)
    expected = torch.cat([hadamard.transform(blocks[:600].contiguous(), signs_before=signs, signs_after=signs),
                          hadamard.transform(blocks[600:].contiguous(), signs_before=signs, signs_after=signs)])
    assert torch.equal(signed, expected)
    in_place = value.clone()
    hadamard.transform(in_place, out=in_place)
    assert torch.equal(in_place, out)


def test_leading_dimensions_and_involution():
    from mlkit_amd.kernels import hadamard

    rng = np.random.default_rng(1)
    value = rng.standard_normal((3, 7, 256)).astype(F32)
    once = hadamard.transform(dev(value))
    np.testing.assert_array_equal(host(once), transforms.fwht(value))
    np.testing.assert_allclose(host(hadamard.transform(once)), value, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(np.linalg.norm(host(once)), np.linalg.norm(value), rtol=1e-5)


def test_rejects_other_widths():
    from mlkit_amd.kernels import hadamard

    with pytest.raises(ValueError, match="power-of-two"):
        hadamard.transform(torch.zeros((4, 12), device="cuda"))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_half_precision_rows_compute_in_fp32(dtype):
    from mlkit_amd.kernels import hadamard

    generator = torch.Generator().manual_seed(2)
    value = torch.randn((8, 4096), generator=generator).to(dtype)
    out = hadamard.transform(value.cuda())
    assert out.dtype == dtype
    expected = torch.from_numpy(transforms.fwht(value.float().numpy())).to(dtype)
    torch.cuda.synchronize()
    assert torch.equal(out.cpu(), expected)


def test_fused_signs_match_separate_multiplication():
    from mlkit_amd.kernels import hadamard

    rng = np.random.default_rng(3)
    value = rng.standard_normal((9, 1024)).astype(F32)
    signs = transforms.deterministic_signs(1024, seed=77)
    forward = hadamard.transform(dev(value), signs_before=dev(signs))
    np.testing.assert_array_equal(host(forward), transforms.fwht((value * signs).astype(F32)))
    inverse = hadamard.transform(forward, signs_after=dev(signs))
    np.testing.assert_allclose(host(inverse), value, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("width", [12, 20, 28, 96, 896, 4864, 7, 14336])
def test_blocked_transform_matches_oracle(width):
    from mlkit_amd.kernels import hadamard

    order, power, basis = transforms.transform_factor(width)
    rng = np.random.default_rng(width)
    rows = 6
    value = rng.standard_normal((rows, width)).astype(F32)
    signs = transforms.deterministic_signs(width, seed=5)
    blocks = hadamard.transform(dev(value).view(rows, order, power), signs_before=dev(signs))
    np.testing.assert_array_equal(host(blocks).reshape(rows, width),
                                  transforms.fwht((value * signs).astype(F32).reshape(rows, order, power)).reshape(rows, width))
    mixed = hadamard.mix_blocks(blocks, dev(basis), transpose=False).view(rows, width)
    expected = transforms.randomized(value, signs)
    np.testing.assert_allclose(host(mixed), expected, rtol=1e-5, atol=1e-5)
    # inverse: H blocks, transposed basis, signs afterwards
    back = hadamard.transform(mixed.view(rows, order, power))
    back = hadamard.mix_blocks(back, dev(basis), transpose=True, signs_after=dev(signs)).view(rows, width)
    np.testing.assert_allclose(host(back), value, rtol=1e-5, atol=2e-5)
    np.testing.assert_allclose(host(back), transforms.randomized(expected, signs, inverse=True), rtol=1e-5, atol=2e-5)


@pytest.mark.parametrize("width", [896, 4864, 11008, 14336])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_one_launch_blocked_transform_equals_the_two_calls(width, dtype):
    """`mk_rotate_blocks` against `mk_fwht` + `mk_basis_mix` (+ the cast), bit for bit, forward
    with the signs in front and inverse with the signs behind; 5 rows and 1 row."""
    from mlkit_amd.kernels import hadamard

    order, power, basis = transforms.transform_factor(width)
    assert hadamard.fits_one_launch(order, power)
    generator = torch.Generator(device="cuda").manual_seed(width)
    signs = dev(transforms.deterministic_signs(width, seed=9))
    for rows in (5, 1):
        value = torch.randn((rows, order, power), device="cuda", generator=generator).to(dtype)
        for inverse in (False, True):
            before, after = (None, signs) if inverse else (signs, None)
            staged = torch.empty(value.shape, device="cuda", dtype=torch.float32)
            hadamard.transform(value, signs_before=before, out=staged)
            expected = hadamard.mix_blocks(staged, dev(basis), transpose=inverse, signs_after=after).to(dtype)
            result = hadamard.rotate_blocks(value, dev(basis), transpose=inverse, signs_before=before, signs_after=after)
            assert result.dtype == dtype
            assert torch.equal(result, expected)


@pytest.mark.parametrize("width", [14336, 7168, 5120, 6144])
def test_one_pass_rotation_of_many_rows_equals_the_two_calls(width):
    """More than 256 outer rows of fp32 take `rotate_matrix_kernel` (transform between registers
    and lanes, one LDS exchange, basis product on the matrix cores): bit for bit what `mk_fwht` +
    `mk_basis_mix` give, forward with the signs in front and inverse with the signs behind; and
    `mk.rht` on a weight-sized tensor goes that way."""
    from mlkit_amd.kernels import hadamard

    order, power, basis = transforms.transform_factor(width)
    rows = 301
    generator = torch.Generator(device="cuda").manual_seed(width)
    value = torch.randn((rows, order, power), device="cuda", generator=generator)
    assert hadamard.streams_in_one_pass(value, order, power)
    signs = dev(transforms.deterministic_signs(width, seed=9))
    for inverse in (False, True):
        before, after = (None, signs) if inverse else (signs, None)
        staged = hadamard.transform(value, signs_before=before)
        expected = hadamard.mix_blocks(staged, dev(basis), transpose=inverse, signs_after=after)
        result = hadamard.rotate_blocks(value, dev(basis), transpose=inverse, signs_before=before, signs_after=after)
        assert torch.equal(result, expected)
        assert torch.equal(hadamard.rotate_blocks(value, dev(basis), transpose=inverse), 
                           hadamard.mix_blocks(hadamard.transform(value), dev(basis), transpose=inverse))
    import mlkit_amd as mk

    flat = value.view(rows, width)
    rotated = mk.rht(flat, seed=3)
    torch.testing.assert_close(rotated.norm(dim=1), flat.norm(dim=1), rtol=1e-5, atol=0)
    torch.testing.assert_close(mk.rht(rotated, seed=3, inverse=True), flat, rtol=1e-5, atol=2e-5)
    np.testing.assert_allclose(host(mk.structured_transform(flat[:4].contiguous())),
                               host(mk.structured_transform(flat))[:4], rtol=1e-5, atol=1e-5)  # few rows: the LDS kernel


def test_one_launch_blocked_transform_declines_what_does_not_fit():
    from mlkit_amd.kernels import hadamard

    assert not hadamard.fits_one_launch(7, 16)       # blocks narrower than an MFMA tile
    assert not hadamard.fits_one_launch(97, 64)      # basis beyond three MFMA row tiles
    assert not hadamard.fits_one_launch(3, 32768)    # more than 160 KB of LDS
    value = torch.zeros((2, 7, 16), device="cuda")
    with pytest.raises(Exception, match="do not fit one workgroup"):
        hadamard.rotate_blocks(value, torch.eye(7, device="cuda"), transpose=False)


def test_weight_sized_rotation_keeps_norms():
    """4096 x 14336 fp32 along K as 7 x 2048 blocks (the literal blocked FWHT) and along
    4096: row norms are preserved and the transform is its own inverse."""
    from mlkit_amd.kernels import hadamard

    generator = torch.Generator(device="cuda").manual_seed(4)
    weight = torch.randn((4096, 14336), device="cuda", generator=generator) * 0.02
    blocks = hadamard.transform(weight.view(4096, 7, 2048))
    torch.testing.assert_close(blocks.view(4096, -1).norm(dim=1), weight.norm(dim=1), rtol=1e-5, atol=0)
    torch.testing.assert_close(hadamard.transform(blocks).view_as(weight), weight, rtol=1e-5, atol=1e-6)
    sample = weight[:3].cpu().numpy().reshape(3, 7, 2048)
    np.testing.assert_array_equal(host(blocks[:3]), transforms.fwht(sample))


@pytest.mark.parametrize("width", [32, 64, 512, 896, 4096, 4864, 11008, 14336, 32768])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_row_rotation_kernel_matches_oracle(width, dtype):
    """mk_rotate_rows (mix, then one Walsh-Hadamard transform per output block; the online
    rotation of activations) against the oracle's transform-then-mix: the same linear map in
    another summation order, so fp32 results agree to rounding (the reference's own bound for
    the basis product, rtol 1e-5 of the row norm scale), and rows are independent."""
    from mlkit_amd.quantization.transforms import OnlineRotation, random_signs

    rotation = OnlineRotation(seed=width + 1)
    signs = host(random_signs(width, width + 1, "cuda"))
    for rows in (1, 8, 33):
        generator = torch.Generator().manual_seed(width + rows)
        value = torch.randn((rows, width), generator=generator).to(dtype)
        rotated = rotation(value.cuda())
        assert rotated.dtype == dtype and rotated.shape == value.shape
        expected = transforms.randomized(value.float().numpy(), signs)
        if dtype == torch.float32:
            np.testing.assert_allclose(host(rotated), expected, rtol=1e-5, atol=2e-5)
            np.testing.assert_allclose(np.linalg.norm(host(rotated), axis=1), np.linalg.norm(value.numpy(), axis=1), rtol=1e-5)
        else:
            rounded = torch.from_numpy(expected).to(dtype).float().numpy()
            step = 2.0 ** (-10 if dtype == torch.float16 else -7)
            assert np.abs(host(rotated.float()) - rounded).max() <= step * np.abs(expected).max()
            assert (host(rotated.float()) == rounded).mean() > 0.99          # one rounding: only near-ties move
    first = rotation(value[:1].cuda())
    assert torch.equal(first, rotated[:1])


def test_known_answers_of_the_bases_on_the_device():
    """The device path applies the known Paley sign patterns and scipy's DCT-II to the outer axis
    (tests/golden/transform_known_answers.json, worked out with Python integers): a unit vector e_f comes out
    as column f of the basis, and with a power-of-two factor as that column times the Sylvester block."""
    import json
    import pathlib

    import scipy.fft

    from mlkit_amd.quantization import codecs, transforms as device_transforms

    known = json.loads((pathlib.Path(__file__).resolve().parent / "golden" / "transform_known_answers.json").read_text())
    for order in (12, 20, 28, 44):
        pattern = np.array(known["paley"][str(order)], dtype=np.float64) / np.sqrt(order)
        out = host(device_transforms.structured_transform(torch.eye(order, device="cuda")))
        np.testing.assert_allclose(out, pattern.T, atol=1e-6)
        back = host(device_transforms.structured_transform(torch.eye(order, device="cuda"), inverse=True))
        np.testing.assert_allclose(back, pattern, atol=1e-6)
    pattern = np.array(known["paley"]["28"], dtype=np.float64) / np.sqrt(28)
    for power in (2, 32, 512):                                        # 56, 896, 14336 = 28 x power
        width = 28 * power
        rows = torch.zeros(3, width, device="cuda")
        picks = [(0, 0), (1, power + 1), (2, 14 * power + power - 1)]  # e_(f, p) at rows 0, 1, 2
        for row, index in picks:
            rows[row, index] = 1.0
        out = host(device_transforms.structured_transform(rows)).reshape(3, 28, power)
        sylvester = transforms.sylvester(power) / np.sqrt(power)
        for row, index in picks:
            f, p = divmod(index, power)
            np.testing.assert_allclose(out[row], np.outer(pattern[:, f], sylvester[:, p]), atol=1e-6)
    for width, order in ((7, 7), (43, 43), (86, 43), (11008, 43)):
        power = width // order
        dct = scipy.fft.dct(np.eye(order), type=2, norm="ortho", axis=0)
        rows = torch.zeros(order, width, device="cuda")
        rows[torch.arange(order), torch.arange(order) * power] = 1.0   # e_(f, 0)
        out = host(device_transforms.structured_transform(rows)).reshape(order, order, power)
        np.testing.assert_allclose(out[:, :, 0], dct.T / np.sqrt(power), atol=1e-6)
    for case in known["signs"]:
        assert codecs.deterministic_signs(16, case["seed"], "cuda").tolist() == case["first"]


@pytest.mark.parametrize("rows", [256, 640, 1024, 1216, 2048, 4096, 8192])
@pytest.mark.parametrize("columns", [1, 7, 16, 129, 260])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_columns_are_transformed_as_the_rows_of_the_turned_matrix(rows, columns, dtype):
    """`rotate_columns` (one kernel for 1024, 2048 and 4096 rows, a turned matrix otherwise), there and back, against the row
    transform of the same fp32 numbers: log2(rows) additions in another order, each rounding 2^-24 of the norm."""
    from mlkit_amd.quantization import transforms as device_transforms
    from mlkit_amd.quantization.codecs import deterministic_signs

    generator = torch.Generator(device="cuda").manual_seed(rows + columns)
    matrix = torch.randn((rows, columns), device="cuda", generator=generator).to(dtype)
    signs = deterministic_signs(rows, 5, matrix.device)
    for inverse in (False, True):
        out = device_transforms.rotate_columns(matrix, signs=signs, inverse=inverse)
        expected = device_transforms.rotate(matrix.float().T.contiguous(), signs=signs, inverse=inverse).T
        assert out.dtype == torch.float32 and out.shape == matrix.shape
        assert (out - expected).norm() <= 16 * 2.0**-24 * expected.norm()
    back = device_transforms.rotate_columns(device_transforms.rotate_columns(matrix, signs=signs), signs=signs, inverse=True)
    assert (back - matrix.float()).norm() <= 64 * 2.0**-24 * matrix.float().norm()
    view = torch.randn((columns, rows), device="cuda", generator=generator).T   # another order of strides
    np.testing.assert_allclose(host(device_transforms.rotate_columns(view, signs=signs)),
                               host(device_transforms.rotate_columns(view.contiguous(), signs=signs)), rtol=0, atol=0)


@pytest.mark.parametrize("rows", [640, 1024, 2048, 4096])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_columns_and_rows_run_their_stages_in_one_order(rows, dtype):
    """The transform of columns rounds exactly as that of the turned matrix: ascending strides, signs and scale alike."""
    from mlkit_amd.quantization import transforms as device_transforms
    from mlkit_amd.quantization.codecs import deterministic_signs

    matrix = torch.randn((rows, 131), device="cuda").to(dtype)
    signs = deterministic_signs(rows, 9, matrix.device)
    for inverse in (False, True):
        expected = device_transforms.rotate(matrix.float().T.contiguous(), signs=signs, inverse=inverse).T
        assert torch.equal(device_transforms.rotate_columns(matrix, signs=signs, inverse=inverse), expected)


@pytest.mark.parametrize("width,rows", [(6080, 1), (6080, 19), (6080, 300), (8320, 5), (8320, 900)])
def test_large_bases_sum_in_parts(width, rows):
    """Bases of more than 256 rows: 64 products at a time, then their sums.  Both roundings walk at random, so the error is about
    2^-24 sqrt(64 / 3 + parts / 3) over the terms' spread, and the transform's stages add a little: 2.2e-7 covers both widths,
    where one chain gives 3.5e-7 and 5.5e-7.  A weight that is quantized behind it keeps the product of tensor operations."""
    from mlkit_amd.quantization import transforms as device_transforms

    generator = torch.Generator(device="cuda").manual_seed(width + rows)
    value = torch.randn((rows, width), device="cuda", generator=generator)
    order, power, basis = device_transforms.transform_factor(width)
    assert order > 256
    points = torch.ones((1, 1), device="cuda", dtype=torch.float64)
    while points.shape[0] < power:
        points = torch.cat([torch.cat([points, points], 1), torch.cat([points, -points], 1)])
    exact = torch.matmul(basis.cuda().double(), value.double().reshape(rows, order, power) @ points / power**0.5).reshape(rows, width)
    assert (device_transforms.rotate(value) - exact).norm() <= 2.2e-7 * exact.norm()
    signs = device_transforms.random_signs(width, 3, "cuda")
    kept = device_transforms._structured_on_host(value * signs, order, power, basis, False)
    assert torch.equal(device_transforms.randomized_weight(value, seed=3), kept)


@pytest.mark.parametrize("rows,columns", [(4096, 2047), (4096, 2048), (4096, 2061), (2048, 2049), (4096, 262147)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_columns_at_the_edges_of_their_workgroups(rows, columns, dtype):
    """Both sides of the rule for 8 or 16 columns a workgroup, and a matrix whose bytes take offsets of more than 32 bits: signs
    that are any numbers, scattered columns and the last ones, bit for bit the transform of rows."""
    from mlkit_amd.quantization import transforms as device_transforms

    generator = torch.Generator(device="cuda").manual_seed(columns)
    signs = torch.randn((rows,), device="cuda", generator=generator)
    looked_at = torch.cat([torch.arange(0, columns, 211), torch.arange(columns - 40, columns)]).cuda()
    matrix = torch.randn((rows, columns), device="cuda", generator=generator, dtype=dtype)
    rows_of = matrix[:, looked_at].float().T.contiguous()
    for inverse in (False, True):
        out = device_transforms.rotate_columns(matrix, signs=signs, inverse=inverse)[:, looked_at]
        assert torch.equal(out, device_transforms.rotate(rows_of, signs=signs, inverse=inverse).T)


@pytest.mark.parametrize("rows", [2, 3])
def test_columns_of_a_very_wide_matrix(rows):
    """More columns than a launch has workgroups in its second dimension (65535 tiles of 64)."""
    from mlkit_amd.quantization import transforms as device_transforms

    matrix = torch.randn((rows, 64 * 65536 + 1), device="cuda").half()
    signs = torch.tensor([1.0, -1.0, 1.0][:rows], device="cuda")
    expected = device_transforms.rotate(matrix.float().T.contiguous(), signs=signs).T
    assert torch.equal(device_transforms.rotate_columns(matrix, signs=signs), expected)


# 1472 and 6080: bases of 368 and 380 rows; 33000: past the row kernels, in tensor operations
@pytest.mark.parametrize("rows", [64, 1024, 1472, 4099, 6080, 33000])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
def test_a_rotated_basis_is_entered_in_fp32(rows, dtype):
    """Whatever type a weight has, the inner quantizer sees the rotation of its fp32 numbers, and a reconstruction that
    comes back in 16 bits leaves the basis as the turned matrix would."""
    import mlkit_amd as mk
    from mlkit_amd.quantization import transforms as device_transforms
    from mlkit_amd.quantization.codecs import deterministic_signs
    from mlkit_amd.quantization.core import layer_seed

    weight = torch.randn((rows, 24), device="cuda").to(dtype)
    entered = []

    def inner(value, ctx):
        entered.append(value)
        return mk.Q(value.half(), bits=1)

    ctx = mk.Ctx("layer", device="cuda")
    left = mk.incoherent(inner, right=None)(weight, ctx).w
    signs = deterministic_signs(rows, layer_seed("layer", ctx._seed) % 2**32, weight.device)
    expected = device_transforms.rotate(weight.float().T.contiguous(), signs=signs).T
    assert entered[0].dtype == torch.float32 and torch.equal(entered[0], expected)
    back = device_transforms.rotate(expected.half().T.contiguous(), inverse=True, signs=signs).T
    assert left.dtype == back.dtype and torch.equal(left, back)


@pytest.mark.parametrize("rows,order,power", [
    (1, 33, 4), (3, 43, 64), (70, 64, 128), (5, 65, 512), (130, 97, 8), (33, 129, 4), (1, 380, 16), (700, 204, 32), (9, 1040, 8),
    (2100, 60, 16)])
@pytest.mark.parametrize("transpose", [False, True])
def test_mixing_with_large_bases(rows, order, power, transpose):
    """More than 32 blocks: small and large tiles, blocks shorter and longer than a tile, edges in all three directions.  Every
    sum within its rounding bound of 64 bits ((order + 1) half ulps of the magnitudes added)."""
    from mlkit_amd.kernels import hadamard

    generator = torch.Generator(device="cuda").manual_seed(rows + order)
    value = torch.randn((rows, order, power), device="cuda", generator=generator)
    basis = torch.randn((order, order), device="cuda", generator=generator)
    signs = (torch.rand(order * power + 1, device="cuda", generator=generator) < 0.5).float()[1:] * 2 - 1   # off 16 bytes
    mix = (basis.T if transpose else basis).double()
    expected = torch.matmul(mix, value.double())
    bound = (order + 1) * 2.0**-24 * torch.matmul(mix.abs(), value.double().abs())
    for given in (None, signs, signs.clone()):
        out = hadamard.mix_blocks(value, basis, transpose=transpose, signs_after=given)
        exact = expected if given is None else expected * given.double().reshape(order, power)
        assert ((out.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("width", [736, 1472, 4992, 6080])   # bases of 368, 368, 312 and 380 rows, blocks of 2, 4, 16 and 16
@pytest.mark.parametrize("rows", [1, 19, 300])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_rotations_with_bases_of_more_than_256_rows(width, rows, dtype):
    """There and back against 64 bits, with fp32 signs and without any.  fp32 results: rounding of width additions at most; 16
    bits: of the result."""
    from mlkit_amd.quantization import transforms as device_transforms
    from mlkit_amd.quantization.codecs import deterministic_signs

    order, power, basis = device_transforms.transform_factor(width)
    value = torch.randn((rows, width), device="cuda").to(dtype)
    signs = deterministic_signs(width, 3, value.device)
    hadamard = device_transforms.hadamard(torch.eye(power, dtype=torch.float64)).cuda()
    whole = torch.kron(basis.double().cuda(), hadamard)
    step = {torch.float32: width * 2.0**-24, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}
    for inverse in (False, True):
        for given in (signs, None):
            out = device_transforms.rotate(value, inverse=inverse, signs=given)
            flips = 1 if given is None else given
            expected = (value.double() @ whole) * flips if inverse else (value.double() * flips) @ whole.T
            assert out.dtype == (dtype if given is None else torch.float32)   # as the same operations on tensors have it
            # (blocks of two values go through tensor operations, which round 16-bit ones on the way: width 736)
            allowed = step[dtype] if power < 4 else step[out.dtype]
            assert (out.double() - expected).norm() <= allowed * expected.norm()


@pytest.mark.parametrize("width", [64, 896, 6080])   # no basis, and bases of 28 and 380 rows
@pytest.mark.parametrize("inverse", [False, True])
def test_trained_signs_receive_their_gradient(width, inverse):
    """Rows, columns and separate blocks of a value that needs no gradient itself.  A gradient is a sum over five rows of
    products of a probe and a rotated value, each within the width's rounding of 64 bits."""
    from mlkit_amd.quantization import transforms as device_transforms
    from mlkit_amd.quantization.codecs import deterministic_signs

    value, probe = torch.randn((2, 5, width), device="cuda")
    signs = deterministic_signs(width, 3, value.device).requires_grad_()
    exact = signs.detach().double().requires_grad_()

    def turned(matrix, **options):
        return device_transforms.rotate_columns(matrix.T, **options).T

    def in_blocks(matrix, **options):
        return device_transforms.rotate(matrix, block=32, **options)

    for rotated in (device_transforms.rotate, turned, in_blocks):
        expected, = torch.autograd.grad((rotated(value.double(), inverse=inverse, signs=exact) * probe.double()).sum(), exact)
        given, = torch.autograd.grad((rotated(value, inverse=inverse, signs=signs) * probe).sum(), signs)
        assert (given.double() - expected).norm() <= width * 2.0**-24 * expected.norm()


@pytest.mark.parametrize("width", [1472, 6080])   # bases of 368 and 380 rows
@pytest.mark.parametrize("inverse", [False, True])
def test_large_bases_take_the_signs_that_tensor_operations_take(width, inverse):
    """Signs of 64 bits (which come after an FP32 transform on the way back), one for all columns and one for each value; too few
    are refused."""
    from mlkit_amd.quantization import transforms as device_transforms
    from mlkit_amd.quantization.codecs import deterministic_signs

    value = torch.randn((3, width), device="cuda")
    signs = deterministic_signs(width, 3, value.device)

    def exact(matrix, given):
        return device_transforms.rotate(matrix.double(), inverse=inverse, signs=given)

    def close(out, expected, step):
        return (out.double() - expected).norm() <= width * step * expected.norm()

    wide = device_transforms.rotate(value, inverse=inverse, signs=signs.double())
    assert wide.dtype == torch.float64 and close(wide, exact(value, signs.double()), 2.0**-24 if inverse else 2.0**-53)
    columns = device_transforms.rotate_columns_in_type(value.half().T, inverse=inverse, signs=signs.double())
    assert columns.dtype == torch.float64
    for given in (torch.tensor(-1.0, device="cuda"), signs * torch.tensor([[1.0], [-1.0], [1.0]], device="cuda")):
        assert close(device_transforms.rotate(value, inverse=inverse, signs=given), exact(value, given), 2.0**-24)
    with pytest.raises(RuntimeError):
        device_transforms.rotate(value, inverse=inverse, signs=signs[:16].contiguous())


@torch.inference_mode()   # (where an earlier capture of the process may have left the random generator's state)
def test_a_captured_rotation_keeps_its_large_basis():
    """Replays after the cache was emptied and the memory it gave back was written over, against the eager result."""
    from mlkit_amd.quantization import transforms as device_transforms

    width = 6080
    value = torch.randn((3, width), device="cuda")
    expected = device_transforms.rht(value, seed=5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = device_transforms.rht(value, seed=5)
    device_transforms.large_bases.clear()
    torch.cuda.synchronize()
    for _ in range(3):
        written = [torch.full((380 * 380,), float("nan"), device="cuda") for _ in range(8)]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, expected) and len(written) == 8
        assert torch.equal(device_transforms.rht(value, seed=5), expected)


@pytest.mark.parametrize("order", [33, 64, 65, 72, 73, 96, 97])
@pytest.mark.parametrize("rows,power", [(1, 1), (9, 2), (33000, 1), (70, 4), (3, 64)])
@pytest.mark.parametrize("transpose", [False, True])
def test_mixing_short_blocks_and_unaligned_tensors(order, rows, power, transpose):
    """What the kernel for large bases does not take: register tiles or a thread per column, every
    sum within its rounding bound of 64 bits, and the bits of the kernel for large bases."""
    from mlkit_amd.kernels import hadamard

    generator = torch.Generator(device="cuda").manual_seed(rows + order)
    storage = torch.randn(rows * order * power + 1, device="cuda", generator=generator)
    basis = torch.randn((order, order), device="cuda", generator=generator)
    signs = (torch.rand(order * power + 1, device="cuda", generator=generator) < 0.5).float()[1:] * 2 - 1
    value = storage[1:].view(rows, order, power) if power >= 4 else storage[:-1].view(rows, order, power)
    mix = (basis.T if transpose else basis).double()
    bound = (order + 1) * 2.0**-24 * torch.matmul(mix.abs(), value.double().abs())
    expected = torch.matmul(mix, value.double())
    out = hadamard.mix_blocks(value, basis, transpose=transpose)
    assert ((out.double() - expected).abs() <= bound).all()
    assert torch.equal(hadamard.mix_blocks(value, basis, transpose=transpose, signs_after=signs), out * signs.view(order, power))
    if power >= 4:   # the kernel for large bases sums in the same order
        assert torch.equal(out, hadamard.mix_blocks(value.clone(), basis, transpose=transpose))


def test_mixing_refuses_signs_of_another_length():
    from mlkit_amd.kernels import hadamard

    value, basis = torch.randn((2, 40, 8), device="cuda"), torch.randn((40, 40), device="cuda")
    for signs in (torch.ones(8, device="cuda"), torch.ones(40 * 8, device="cuda").half(), torch.ones(2 * 40 * 8, device="cuda")[::2]):
        with pytest.raises(ValueError, match="sign vectors"):
            hadamard.mix_blocks(value, basis, transpose=False, signs_after=signs)


@pytest.mark.parametrize("rows,columns", [(1, 1), (3, 70), (64, 64), (65, 4), (100, 132), (260, 68)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_turning_a_matrix(rows, columns, dtype):
    from mlkit_amd.kernels import hadamard

    matrix = torch.randn((rows, columns), device="cuda").to(dtype)
    assert torch.equal(hadamard.turned(matrix), matrix.float().T.contiguous())
    if rows > 1:   # a base that is not 16-byte aligned
        assert torch.equal(hadamard.turned(matrix.reshape(-1)[columns:].view(rows - 1, columns)), matrix[1:].float().T.contiguous())


@pytest.mark.parametrize("seed", [0, 1, 2**32 - 17, 2**40 + 3])
def test_signs_of_a_seed_are_the_same_on_every_device(seed):
    from mlkit_amd.quantization.codecs import deterministic_signs

    assert torch.equal(deterministic_signs(1003, seed, "cuda").cpu(), deterministic_signs(1003, seed, "cpu"))
