"""GPU parity (through the C ABI) of the error-feedback kernels against the C oracle:
reconstructions, codes, solved continuations and the trailing update bit for bit."""

import numpy as np
import pytest
import torch

from oracle import feedback as oracle_feedback, scaling

import helpers

pytestmark = pytest.mark.gpu

F32 = np.float32
INT4 = scaling.int_values(4)
SEVEN = np.array([-1, -0.5, -0.25, 0, 0.25, 0.5, 1], dtype=F32)


def dev(array):
    return None if array is None else torch.from_numpy(np.ascontiguousarray(array)).cuda()


def host(tensor):
    torch.cuda.synchronize()
    return tensor.cpu().numpy()


def problem(rows, width, seed, samples=None):
    """Weights and the unit upper coefficient matrix of a correlated synthetic Hessian."""
    rng = np.random.default_rng(seed)
    weight = helpers.normal_weight(rows, width, seed=seed)
    samples = samples or 2 * width
    inputs = rng.standard_normal((samples, width)).astype(F32)
    inputs[:, ::7] *= 4
    inputs += 0.5 * np.roll(inputs, 1, axis=1)
    hessian = (inputs.T @ inputs / samples).astype(F32)
    coeff, status = oracle_feedback.coefficients(hessian, 0.01)
    assert status == 0
    return weight, coeff, hessian


@pytest.mark.parametrize("rows,width,tile_start,tile_width,group,values,integer,asym", [
    (71, 96, 0, 96, 32, INT4, True, False),          # the reference's own tile test shape
    (64, 256, 128, 128, 128, INT4, True, False),
    (64, 256, 0, 128, 64, INT4, True, True),
    (35, 512, 128, 200, 128, INT4, True, False),     # four-slot kernel
    (19, 640, 64, 300, 50, INT4, True, True),        # sixteen-slot kernel, ragged groups
    (64, 256, 128, 128, 64, scaling.NF4_VALUES, False, False),
    (33, 128, 0, 100, 128, SEVEN, False, True),
    # tables of 17 to 256 values: the sixteen lanes of a row search the table together
    (64, 256, 128, 128, 64, np.sinh(np.linspace(-3, 3, 256)).astype(F32), False, False),
    (37, 256, 0, 128, 32, np.sinh(np.linspace(-3, 3, 256)).astype(F32), False, True),
    (50, 384, 128, 100, 128, (np.linspace(-1, 1, 40) ** 3).astype(F32), False, False),   # ragged tile, 40 values
    (16, 128, 0, 128, 128, np.linspace(-1, 1, 17).astype(F32), False, True),              # 17 values: ties to the lower entry
])
def test_round_tile_matches_oracle(rows, width, tile_start, tile_width, group, values, integer, asym):
    from mlkit_amd.kernels import error_feedback

    weight, coeff, _ = problem(rows, width, seed=rows + tile_width)
    rng = np.random.default_rng(1)
    feedback = (rng.standard_normal((rows, width)) * 0.004).astype(F32)
    region_start = tile_start - (group if tile_start >= group and tile_start % group == 0 else 0)
    region = weight[:, region_start:tile_start + tile_width]
    scales, zeros = oracle_feedback.fit_scales(region, values, group, asym)
    expected_out = np.zeros_like(weight)
    expected_codes = np.zeros(weight.shape, dtype=np.uint8)
    oracle_feedback.round_tile(weight, feedback, coeff, scales, zeros, values, expected_out, expected_codes,
                               region_start=region_start, tile_start=tile_start, tile_width=tile_width,
                               group=group, integer=integer)
    output = torch.zeros((rows, width), device="cuda")
    encoded = torch.zeros((rows, width), device="cuda", dtype=torch.uint8)
    bits = 4 if integer else int(np.ceil(np.log2(len(values))))
    error_feedback.round_tile(dev(weight), dev(feedback), dev(coeff), dev(scales), dev(zeros), output, encoded,
                              region_start=region_start, tile_start=tile_start, tile_width=tile_width,
                              group=group, bits=bits, values=dev(values), integer_grid=integer)
    np.testing.assert_array_equal(host(encoded), expected_codes)
    np.testing.assert_array_equal(host(output), expected_out)


@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("tile_width", [128, 96])
def test_round_tile_on_quotients_next_to_half_integers(asym, tile_width):
    """Every target of the tile divides by its scale to k + 1/2 exactly, or to the fp32 numbers right next to
    it on either side: the cases in which the correctly rounded quotient, and not a product with the scale's
    reciprocal, decides the code (a sweep that multiplied by reciprocals would miss a few per cent of these
    codes, as the last assertion shows).  No feedback and no coefficients, so that every column is such a
    case; codes and reconstructions equal the oracle's (true division, round half to even)."""
    from mlkit_amd.kernels import error_feedback

    rows, width, group = 192, 256, 64
    rng = np.random.default_rng(31 + tile_width)
    scales = (rng.random((rows, width // group)) * 0.05 + 0.002).astype(np.float16).astype(F32)
    scales[::3] = (2.0 ** rng.integers(-9, -3, (len(scales[::3]), width // group))).astype(F32)     # exact ties
    zeros = (rng.standard_normal((rows, width // group)) * 0.01).astype(np.float16).astype(F32) if asym else None
    halves = rng.integers(-9, 9, (rows, width)).astype(F32) + F32(0.5)
    wide = np.repeat(scales, group, axis=1)
    weight = (halves * wide).astype(F32)
    if asym:
        weight = (weight + np.repeat(zeros, group, axis=1)).astype(F32)
    nudge = rng.integers(-2, 3, (rows, width))
    weight = np.where(nudge < 0, np.nextafter(weight, F32(-np.inf)), np.where(nudge > 0, np.nextafter(weight, F32(np.inf)), weight)).astype(F32)
    weight[5, 7] = np.nan                                             # a value that is not a number takes the division, too
    feedback = np.zeros_like(weight)
    coeff = np.eye(width, dtype=F32)
    expected_out = np.zeros_like(weight)
    expected_codes = np.zeros(weight.shape, dtype=np.uint8)
    oracle_feedback.round_tile(weight, feedback, coeff, scales, zeros, INT4, expected_out, expected_codes,
                               region_start=0, tile_start=64, tile_width=tile_width, group=group, integer=True)
    output = torch.zeros((rows, width), device="cuda")
    encoded = torch.zeros((rows, width), device="cuda", dtype=torch.uint8)
    error_feedback.round_tile(dev(weight), dev(feedback), dev(coeff), dev(scales), None if zeros is None else dev(zeros), output,
                              encoded, region_start=0, tile_start=64, tile_width=tile_width, group=group, bits=4,
                              values=dev(INT4), integer_grid=True)
    keep = np.ones(weight.shape, dtype=bool)
    keep[5, 7] = False
    np.testing.assert_array_equal(host(encoded)[keep], expected_codes[keep])
    np.testing.assert_array_equal(host(output)[keep], expected_out[keep])
    # the crafted cases really sit at the boundaries: a product with the reciprocal alone would miss some codes
    inside = slice(64, 64 + tile_width)
    centered = weight[:, inside] - (np.repeat(zeros, group, axis=1)[:, inside] if asym else 0)
    by_reciprocal = np.clip(np.rint((centered.astype(F32) * (F32(1) / wide[:, inside])).astype(F32)), -8, 7) + 8
    assert (by_reciprocal[keep[:, inside]] != expected_codes[:, inside][keep[:, inside]]).sum() > 0


@pytest.mark.parametrize("rows,width,start,stop", [(64, 384, 128, 256), (37, 512, 192, 492), (16, 1024, 0, 1024)])
def test_pending_continuation_matches_oracle(rows, width, start, stop):
    from mlkit_amd.kernels import error_feedback

    weight, coeff, _ = problem(rows, width, seed=width + start)
    rng = np.random.default_rng(2)
    feedback = (rng.standard_normal((rows, width)) * 0.01).astype(F32)
    expected = oracle_feedback.pending(feedback, coeff, start, stop)
    solved = error_feedback.pending_continuation(dev(feedback), dev(coeff), start, stop)
    np.testing.assert_array_equal(host(solved), expected)
    targets = error_feedback.pending_continuation(dev(feedback), dev(coeff), start, stop, original=dev(weight))
    np.testing.assert_array_equal(host(targets), (weight[:, start:stop] + expected).astype(F32))
    # the textbook definition: x U = feedback[:, region]
    block = coeff[start:stop, start:stop].astype(np.float64)
    np.testing.assert_allclose(expected @ block, feedback[:, start:stop], rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("rows,width,start,stop", [(128, 512, 0, 128), (200, 700, 128, 256), (71, 333, 64, 101),
                                                   (64, 256, 0, 255)])
def test_block_update_matches_fma_chain(rows, width, start, stop):
    from mlkit_amd.kernels import error_feedback

    weight, coeff, _ = problem(rows, width, seed=width + stop)
    rng = np.random.default_rng(3)
    output = (weight + rng.standard_normal(weight.shape).astype(F32) * 0.003).astype(F32)
    feedback = (rng.standard_normal(weight.shape) * 0.01).astype(F32)
    expected = feedback.copy()
    oracle_feedback.block_update(expected, weight, output, coeff, start, stop, mode=0)
    updated = dev(feedback)
    error_feedback.block_update(updated, dev(weight), dev(output), dev(coeff), start, stop)
    np.testing.assert_array_equal(host(updated), expected)
    exact = feedback[:, stop:].astype(np.float64) + (weight - output)[:, start:stop].astype(np.float64) @ coeff[start:stop, stop:].astype(np.float64)
    np.testing.assert_allclose(host(updated)[:, stop:], exact, rtol=1e-4, atol=1e-6)
    np.testing.assert_array_equal(host(updated)[:, :stop], feedback[:, :stop])


@pytest.mark.parametrize("rows,width,first,chain,chains,begin,end", [
    (130, 1024, 0, 128, 4, 512, 1024),     # a deferred super-block reaching the far columns
    (64, 700, 64, 96, 3, 352, 700),        # ragged widths, unaligned end
    (64, 640, 128, 128, 1, 256, 384),      # the narrow update inside a super-block
    (33, 333, 10, 50, 2, 111, 333),        # nothing aligned: scalar loads
])
def test_chained_block_update_equals_tile_after_tile(rows, width, first, chain, chains, begin, end):
    from mlkit_amd.kernels import error_feedback

    weight, coeff, _ = problem(rows, width, seed=width + chains)
    rng = np.random.default_rng(4)
    output = (weight + rng.standard_normal(weight.shape).astype(F32) * 0.003).astype(F32)
    feedback = (rng.standard_normal(weight.shape) * 0.01).astype(F32)
    expected = feedback.copy()
    for index in range(chains):   # the oracle applies one tile at a time to every later column
        start = first + index * chain
        scratch = expected.copy()
        oracle_feedback.block_update(scratch, weight, output, coeff, start, start + chain, mode=0)
        expected[:, begin:end] = scratch[:, begin:end]
    updated = dev(feedback)
    error_feedback.block_update_range(updated, dev(weight), dev(output), dev(coeff), first, chain, chains, begin, end)
    np.testing.assert_array_equal(host(updated), expected)


@pytest.mark.parametrize("rows,width,first,chain,chains,begin,end", [
    (2048, 5120, 0, 128, 4, 512, 5120),     # 576 tiles: a whole round of 512 on large tiles, 64 as quarter tiles
    (1024, 9216, 128, 128, 2, 384, 9216),   # 552 tiles, two chains
    (2048, 5120, 0, 256, 2, 512, 5120),     # chains of 256 columns: large tiles throughout
    (256, 1024, 0, 128, 4, 512, 1024),      # fewer tiles than slots
    (256, 640, 128, 128, 1, 256, 512),      # one chain over a few tiles: quarter tiles only
])
def test_update_from_kept_deviations_equals_the_recomputing_update(rows, width, first, chain, chains, begin, end):
    """mk_feedback_block_update_staged (deviations handed over column-major; whole rounds on
    128 x 128 tiles, a short last round as 64 x 64 tiles) against mk_feedback_block_update_range,
    which the test above pins to the oracle: the same sums, bit for bit."""
    from mlkit_amd import native
    from mlkit_amd.kernels import error_feedback

    generator = torch.Generator(device="cuda").manual_seed(rows + width)
    weight = torch.randn((rows, width), device="cuda", generator=generator) * 0.02
    output = weight + torch.randn((rows, width), device="cuda", generator=generator) * 0.003
    coeff = torch.randn((width, width), device="cuda", generator=generator).triu(1) * 0.05
    feedback = torch.randn((rows, width), device="cuda", generator=generator) * 0.01
    expected = feedback.clone()
    error_feedback.block_update_range(expected, weight, output, coeff, first, chain, chains, begin, end)
    deviations = (weight - output).T.contiguous()
    updated = feedback.clone()
    native.check(native.library().mk_feedback_block_update_staged(
        updated.data_ptr(), deviations.data_ptr(), coeff.data_ptr(), rows, width, first, chain, chains, begin, end,
        native.current_stream(updated.device)))
    assert torch.equal(updated, expected)
    assert torch.equal(updated[:, :begin], feedback[:, :begin])


@pytest.mark.parametrize("rows,width", [(1, 260), (3, 389), (63, 516), (130, 641), (129, 1157), (260, 1284), (517, 2049), (1029, 3076),
                                        (128, 640), (256, 1284), (1024, 3072)])
def test_sweep_with_kept_deviations_equals_the_one_without(rows, width):
    """Rows and columns that fill no whole tile, on 16-byte boundaries and off them, and whole ones: the kernels that read the
    kept deviations (64 x 64 and 128 x 128 tiles) against the one that works them out again, bit for bit."""
    from mlkit_amd import native

    generator = torch.Generator(device="cuda").manual_seed(rows * width)
    weight = torch.randn((rows, width), device="cuda", generator=generator) * 0.02
    coeff = (torch.randn((width, width), device="cuda", generator=generator) * 0.05).triu(1) + torch.eye(width, device="cuda")
    values = torch.arange(-8.0, 8.0, device="cuda")
    groups, results = -(-width // 128), []
    for kept in (False, True):
        feedback, output = torch.zeros_like(weight), torch.empty_like(weight)
        encoded = torch.empty((rows, width), dtype=torch.uint8, device="cuda")
        scales, workspace = torch.empty((rows, groups), device="cuda"), torch.empty((rows, 128), device="cuda")
        deviations = torch.full((width, rows), float("nan"), device="cuda") if kept else None
        native.check(native.library().mk_feedback_sweep(
            weight.data_ptr(), feedback.data_ptr(), output.data_ptr(), encoded.data_ptr(), coeff.data_ptr(), scales.data_ptr(), None,
            workspace.data_ptr(), native.pointer(deviations), values.data_ptr(), 16, rows, width, 128, 128, 128, 1, -8.0, 7.0, 0,
            0.125, -8.0, native.SCALE_FORMAT_CODES["fp16"], 4, native.current_stream(weight.device)))
        results.append((encoded, output, scales, feedback))
    for one, other in zip(*results):
        assert torch.equal(one, other)


@pytest.mark.parametrize("width,step", [(1024, 1), (1100, 1), (1536, 8), (2304, 1)])
def test_blocked_factorisation_matches_the_float64_coefficients(width, step):
    """`feedback_coefficients` on the device factors matrices of 1024 columns and more block by
    block (`mk_cholesky_block` plus matrix products).  Against the float64 definition at the
    reference's tolerance (tests/quantization/test_algorithms.py:142-166, rtol 1e-3 on the
    upper triangle), and against the library factorisation of the same matrix."""
    import mlkit_amd as mk

    rng = np.random.default_rng(width)
    inputs = rng.standard_normal((2 * width, width)).astype(np.float32)
    inputs[:, ::13] *= 6
    inputs[:, 5] = 0   # a dead channel
    hessian = (inputs.T @ inputs / inputs.shape[0]).astype(np.float32)
    result, status = mk.feedback_coefficients(dev(hessian).clone(), step)
    assert status == 0
    expected, expected_status = oracle_feedback.coefficients(hessian) if step == 1 else (None, 0)
    assert expected_status == 0
    if step == 1:
        upper = np.triu(np.ones((width, width), dtype=bool), 1)
        np.testing.assert_allclose(host(result)[upper], expected[upper], rtol=1e-3, atol=2e-6)
    library, library_status = mk.feedback_coefficients(torch.from_numpy(hessian).clone(), step)   # CPU: LAPACK
    assert library_status == 0
    blocks = np.kron(np.eye(width // step, dtype=bool), np.ones((step, step), dtype=bool))
    outside = np.triu(np.ones((width, width), dtype=bool), 1) & ~blocks
    np.testing.assert_allclose(host(result)[outside], library.numpy()[outside], rtol=1e-3, atol=2e-6)


@pytest.mark.parametrize("width", [1664, 2304])
def test_look_ahead_factorisation_equals_the_one_stream_order(width, monkeypatch):
    """From `LOOK_AHEAD_WIDTH` columns on, the far part of every trailing update runs on a second
    stream; events keep the order in which updates reach an entry, so the coefficients (the
    entries above the diagonal; below it both leave leftovers) are the same bit for bit.
    Twice, because a race would not show every time."""
    import mlkit_amd as mk
    from mlkit_amd.quantization import feedback

    rng = np.random.default_rng(width + 1)
    inputs = rng.standard_normal((2 * width, width)).astype(np.float32)
    inputs[:, ::7] *= 4
    hessian = dev((inputs.T @ inputs / inputs.shape[0]).astype(np.float32))
    monkeypatch.setattr(feedback, "FACTOR_GRAPHS", False)       # launch by launch, with the constants set here
    monkeypatch.setattr(feedback, "FACTORIZATION_PANEL", 256)   # several panels at these widths
    monkeypatch.setattr(feedback, "LOOK_AHEAD_WIDTH", 1 << 30)
    expected, status = mk.feedback_coefficients(hessian.clone(), 1)
    assert status == 0
    monkeypatch.setattr(feedback, "LOOK_AHEAD_WIDTH", 1024)
    for _ in range(2):
        result, status = mk.feedback_coefficients(hessian.clone(), 1)
        assert status == 0
        np.testing.assert_array_equal(np.triu(host(result), 1), np.triu(host(expected), 1))


@pytest.mark.parametrize("look_ahead", [False, True])
def test_captured_factorisation_equals_the_launch_by_launch_one(look_ahead, monkeypatch):
    """From the second matrix of a width on, the factorisation replays a captured graph.  Five
    different matrices of one width, with eager work and synchronisations between the replays and
    another width in between: every result equals the one computed launch by launch, bit for bit
    above the diagonal; an indefinite matrix reports its column through the graph as well."""
    import mlkit_amd as mk
    from mlkit_amd.quantization import feedback

    feedback.clear_factor_graphs()
    monkeypatch.setattr(feedback, "FACTORIZATION_PANEL", 512)
    monkeypatch.setattr(feedback, "LOOK_AHEAD_WIDTH", 1024 if look_ahead else 1 << 30)
    width = 1664
    generator = torch.Generator(device="cuda").manual_seed(11)

    def hessian_of(scale):
        inputs = torch.randn((2 * width, width), device="cuda", generator=generator) * scale
        inputs[:, ::9] *= 3
        return inputs.T @ inputs / inputs.shape[0]

    try:
        matrices = [hessian_of(1.0 + 0.5 * index) for index in range(5)]
        monkeypatch.setattr(feedback, "FACTOR_GRAPHS", False)
        expected = [mk.feedback_coefficients(matrix.clone(), 1)[0] for matrix in matrices]
        monkeypatch.setattr(feedback, "FACTOR_GRAPHS", True)
        other = hessian_of(2.0)[:1280, :1280].contiguous()
        for index, matrix in enumerate(matrices):
            result, status = mk.feedback_coefficients(matrix.clone(), 1)
            assert status == 0
            assert torch.equal(result.triu(1), expected[index].triu(1)), index
            busy = (matrix @ matrix).sum()            # eager work and a synchronisation between replays
            torch.cuda.synchronize()
            assert torch.isfinite(busy)
            if index == 2:
                mk.feedback_coefficients(other.clone(), 1)   # another width in between
        assert feedback._factor_graphs[(0, width)] is not None
        broken = matrices[0].clone()
        broken[900, 900] = -1e6
        assert mk.feedback_coefficients(broken, 1, damp=0.0)[1] != 0
        assert mk.feedback_coefficients(matrices[1].clone(), 1)[1] == 0   # the status starts from zero again
    finally:
        feedback.clear_factor_graphs()


@pytest.mark.parametrize("width,step", [(384, 1), (1152, 1), (1152, 8)])
def test_coefficients_from_several_threads(width, step):
    """Threads with streams of their own and matrices of one width, with another width in between (which may drop the
    width's graph): everyone receives the coefficients that one thread alone works out, bit for bit."""
    import threading

    import mlkit_amd as mk
    from mlkit_amd.quantization import feedback

    generator = torch.Generator(device="cuda").manual_seed(width + step)

    def hessian_of(columns):
        inputs = torch.randn((2 * columns, columns), device="cuda", generator=generator)
        return inputs.T @ inputs / inputs.shape[0]

    matrices = [[hessian_of(width), hessian_of(width), hessian_of(width + 128)] for _ in range(3)]
    expected = [[mk.feedback_coefficients(matrix.clone(), step)[0] for matrix in some] for some in matrices]
    torch.cuda.synchronize()
    feedback.clear_factor_graphs()
    wrong, failures = [], []

    def work(index):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for turn in range(6):
                    for matrix, right in zip(matrices[index], expected[index]):
                        result, status = mk.feedback_coefficients(matrix.clone(), step)
                        torch.cuda.current_stream().synchronize()
                        if status != 0 or not torch.equal(result.triu(step), right.triu(step)):
                            wrong.append((index, turn, matrix.shape[0]))
        except Exception as error:   # reported by the main thread
            failures.append(repr(error))

    threads = [threading.Thread(target=work, args=(index,)) for index in range(3)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join(timeout=60)
    feedback.clear_factor_graphs()
    assert not failures and not wrong, (failures, wrong)


def test_blocked_factorisation_reports_an_indefinite_matrix():
    import mlkit_amd as mk

    width = 1280
    rng = np.random.default_rng(3)
    inputs = rng.standard_normal((width // 2, width)).astype(np.float32)   # rank deficient
    hessian = (inputs.T @ inputs).astype(np.float32)
    hessian[700, 700] = -5000.0
    _, status = mk.feedback_coefficients(dev(hessian).clone(), 1, damp=0.0)
    assert status != 0
    quantizer = mk.gptq(mk.int(4, group=128))
    with pytest.raises(ValueError, match="positive definite"):
        quantizer(dev(np.zeros((8, width), dtype=np.float32)), mk.Ctx("layer", H=dev(hessian)))


def block_factor(matrix, size, first=0, entry="mk_cholesky_block"):
    """`mk_cholesky_block` on the first `size` rows of a matrix: (factor, block row, status)."""
    from mlkit_amd import native

    width = matrix.shape[0]
    work = dev(matrix)
    beside = width - size
    factor = torch.zeros((128, 128), device="cuda")
    status = torch.zeros((), dtype=torch.int32, device="cuda")
    native.check(getattr(native.library(), entry)(
        work.data_ptr(), width, size, first, beside, factor.data_ptr() if beside else None, status.data_ptr(),
        native.current_stream(work.device)))
    out = host(work)
    return (host(factor)[:size, :size] if beside else out[:size, :size]), out[:size, size:], int(status.item())


@pytest.mark.parametrize("size,beside", [(1, 0), (15, 0), (16, 1), (17, 64), (64, 63), (100, 130), (113, 0), (127, 200), (128, 0),
                                         (128, 1), (128, 65), (128, 700)])
def test_a_factored_block_and_its_block_row(size, beside):
    """Sizes at the edges of the 16-row panels and of the 64 columns a workgroup carries.  Normwise the factor of a
    well-conditioned matrix is as good as a few fp32 roundings per pivot: 1e-5 of its norm leaves a factor of ten."""
    rng = np.random.default_rng(size * 1000 + beside)
    width = size + beside
    inputs = rng.standard_normal((2 * width + 8, width))
    matrix = (inputs.T @ inputs / inputs.shape[0] + 0.05 * np.eye(width)).astype(np.float32)
    expected = np.linalg.cholesky(matrix[:size, :size].astype(np.float64)).T
    factor, row, status = block_factor(matrix, size)
    assert status == 0
    assert np.linalg.norm(factor - expected) <= 1e-5 * np.linalg.norm(expected)
    assert not np.tril(factor, -1).any()
    if beside:
        carried = np.linalg.solve(expected.T, matrix[:size, size:].astype(np.float64))
        assert np.linalg.norm(row - carried) <= 1e-5 * np.linalg.norm(carried)


@pytest.mark.parametrize("beside", [0, 200])
def test_a_factored_block_is_as_close_to_64_bits_as_the_two_column_kernel(beside):
    """Entries are subtracted from in panels of sixteen products, not product by product: summed over eight matrices the
    distance to the float64 factor is no larger than that of the kernel which subtracts two products at a time."""
    error = {"mk_cholesky_block": 0.0, "mk_cholesky_block_pairs": 0.0}
    for seed in range(8):
        rng = np.random.default_rng(seed)
        width = 128 + beside
        inputs = rng.standard_normal((2 * width, width))
        matrix = (inputs.T @ inputs / inputs.shape[0]).astype(np.float32)
        matrix += 0.01 * np.eye(width, dtype=np.float32)
        exact = np.linalg.cholesky(matrix[:128, :128].astype(np.float64)).T
        for entry in error:
            factor, row, status = block_factor(matrix, 128, entry=entry)
            assert status == 0
            error[entry] += np.linalg.norm(factor - exact) / np.linalg.norm(exact)
            if beside:
                carried = np.linalg.solve(exact.T, matrix[:128, 128:].astype(np.float64))
                error[entry] += np.linalg.norm(row - carried) / np.linalg.norm(carried)
    assert error["mk_cholesky_block"] <= error["mk_cholesky_block_pairs"], error


@pytest.mark.parametrize("size,beside", [(1, 3), (2, 0), (16, 64), (17, 65), (37, 5), (112, 1), (128, 0), (128, 130)])
def test_pairs_of_rows_are_taken_in_their_order(size, beside):
    """`mk_cholesky_block_pairs`, bit for bit: an entry loses fma(u_j, v_j, u_{j+1} v_{j+1}) for one pair of rows after another.
    Replayed with the factor's own rows (sums in extended precision: one more rounding, at 2^-40 of a 24-bit one); only the
    reciprocal root of a pivot is the device's, one of the numbers within two ulps."""
    f32, wide = np.float32, np.longdouble
    rng = np.random.default_rng(size + beside)
    width = size + beside
    inputs = rng.standard_normal((2 * width + 8, width))
    matrix = (inputs.T @ inputs / inputs.shape[0] + 0.05 * np.eye(width)).astype(f32)
    factor, row, status = block_factor(matrix, size, entry="mk_cholesky_block_pairs")
    assert status == 0 and not np.tril(factor, -1).any()
    upper = factor if not beside else np.concatenate([factor, row], 1)

    def fused(a, b, c):
        return (wide(a) * wide(b) + wide(c)).astype(f32)

    rest = matrix[:size].copy()
    for j in range(0, size, 2):
        for k in range(j, min(j + 2, size)):
            rest[k, k:] = rest[k, k:] if k == j else fused(-upper[j, k], upper[j, k:], rest[k, k:])
            root = f32(1 / np.sqrt(np.float64(rest[k, k])))
            near = [root, *(np.nextafter(root, f32(end)) for end in (0, 2 * root))]
            near += [np.nextafter(near[1], f32(0)), np.nextafter(near[2], f32(2 * root))]
            assert any(np.array_equal((rest[k, k:] * r).astype(f32), upper[k, k:]) for r in near), k
        if j + 1 < size:
            last = (upper[j + 1, :size, None] * upper[j + 1, None]).astype(f32)
            rest[j + 2:] -= fused(upper[j, :size, None], upper[j, None], last)[j + 2:]


@pytest.mark.parametrize("step", [2, 4, 8, 16])
@pytest.mark.parametrize("width", [16, 64, 80, 208, 1008])
def test_block_coefficients_are_those_of_a_forward_substitution(width, step):
    """`mk_blocks_upper_from_factor`: R blockdiag(R)^-1 by x_j = (r_j - x_0 d_0j - ...) / d_jj, fused and in ascending order (in
    extended precision here, rounded once each), whatever lies below the factor's diagonal."""
    from mlkit_amd.quantization import feedback

    f32, wide = np.float32, np.longdouble
    rng = np.random.default_rng(width + step)
    upper = np.triu(rng.standard_normal((width, width)) * 0.3).astype(f32)
    upper[np.arange(width), np.arange(width)] = 0.5 + rng.random(width).astype(f32)
    r = upper.T[::-1, ::-1]
    expected = np.zeros_like(r)
    for first in range(0, width, step):
        for j in range(first, first + step):
            rest = r[:, j].copy()
            for k in range(first, j):
                rest = (wide(rest) - wide(expected[:, k]) * wide(r[k, j])).astype(f32)
            expected[:, j] = rest / r[j, j]
    junk = upper + np.tril(np.full((width, width), np.nan, dtype=f32), -1)
    out = host(feedback._block_coefficients(dev(junk), step))
    np.testing.assert_array_equal(out, expected)


@pytest.mark.parametrize("beside", [0, 65])
@pytest.mark.parametrize("column", [0, 1, 15, 16, 47, 100, 127])
def test_pairs_of_rows_report_the_first_refused_pivot(column, beside):
    rng = np.random.default_rng(column)
    width = 128 + beside
    matrix = (rng.standard_normal((width, width)) * 0.01).astype(np.float32)
    matrix = matrix + matrix.T + np.diag(np.full(width, 4, dtype=np.float32))
    matrix[column, column] = -1.0
    matrix[127, 127] = -1.0
    assert block_factor(matrix, 128, first=256, entry="mk_cholesky_block_pairs")[2] == 256 + column + 1


@pytest.mark.parametrize("column", [0, 1, 15, 16, 47, 100, 126])
@pytest.mark.parametrize("value", [-1.0, float("nan"), float("inf")])
def test_a_factored_block_names_its_bad_pivot(column, value):
    matrix = np.eye(130, dtype=np.float32) * 2
    matrix[column, column] = value
    assert block_factor(matrix, 128, first=256)[2] == 256 + column + 1


@pytest.mark.parametrize("width,k_first,k_stop,row_first,row_stop", [
    (200, 0, 128, 128, 200), (129, 0, 128, 128, 129), (517, 128, 384, 384, 512), (1000, 0, 256, 256, 384), (4300, 0, 128, 128, 256)])
@pytest.mark.parametrize("one_chain", [0, 1])
def test_products_of_a_block_of_rows(width, k_first, k_stop, row_first, row_stop, one_chain):
    """`mk_factor_block_rows`: rows and columns that fill no tile, both tile widths; every sum within its rounding bound of 64
    bits ((k + 1) half ulps of the magnitudes added), everything else untouched."""
    check_products("mk_factor_block_rows", width, k_first, k_stop, row_first, row_stop, one_chain, triangular=False)


@pytest.mark.parametrize("width,k_first,k_stop,row_first,row_stop", [
    (130, 0, 64, 64, 130), (321, 64, 128, 128, 321), (600, 0, 256, 256, 600), (700, 0, 128, 128, 300), (1031, 512, 768, 768, 1031),
    (5700, 0, 64, 64, 5700), (5701, 0, 64, 64, 5701)])
@pytest.mark.parametrize("leave_room", [0, 1])
def test_products_behind_a_panel(width, k_first, k_stop, row_first, row_stop, leave_room):
    """`mk_factor_trailing`: both tile sizes, on 16-byte boundaries and off them, all rows behind the panel and a band of them."""
    check_products("mk_factor_trailing", width, k_first, k_stop, row_first, row_stop, leave_room, triangular=True)


def check_products(entry, width, k_first, k_stop, row_first, row_stop, option, triangular):
    from mlkit_amd import native

    generator = torch.Generator(device="cuda").manual_seed(width + k_stop)
    matrix = torch.randn((width, width), device="cuda", generator=generator)
    result = matrix.clone()
    native.check(getattr(native.library(), entry)(result.data_ptr(), width, k_first, k_stop, row_first, row_stop, option,
                                                  native.current_stream(matrix.device)))
    finished = matrix[k_first:k_stop].double()
    rows = finished[:, row_first:row_stop]
    expected = matrix[row_first:row_stop].double() - rows.T @ finished
    bound = (k_stop - k_first + 1) * 2.0**-24 * (matrix[row_first:row_stop].abs().double() + rows.abs().T @ finished.abs())
    column, row = torch.arange(width, device="cuda"), torch.arange(row_first, row_stop, device="cuda")[:, None]
    changed = column >= (row if triangular else torch.full_like(row, row_first))
    got = result[row_first:row_stop]
    assert ((got.double() - expected).abs() <= bound)[changed].all()
    if triangular:   # tiles below the diagonal are skipped; what lies below it inside a diagonal tile may change
        changed = column >= row_first + (row - row_first) // 128 * 128
    assert torch.equal(got[~changed], matrix[row_first:row_stop][~changed])
    assert torch.equal(result[:row_first], matrix[:row_first]) and torch.equal(result[row_stop:], matrix[row_stop:])


@pytest.mark.parametrize("width,step", [(128, 1), (129, 1), (255, 1), (384, 8), (640, 1), (896, 1), (1000, 2), (1023, 1)])
def test_blocked_factorisation_of_narrow_matrices(width, step):
    """The same comparison as for wide matrices, from the narrowest one that is factored by blocks."""
    test_blocked_factorisation_matches_the_float64_coefficients(width, step)
