"""fp32 / fp16 sparse_conv2d on the matrix cores (tuning.float_mfma) against the same sums in 64 bits, and the rule that
gives calls to it."""
import ctypes as C

import numpy as np
import pytest

from helpers import capi, workloads, pla, make_kernel, run_hip, run_oracle, oracle_pack

pytestmark = pytest.mark.gpu

AP = pla.ActivationParam
ACTS = {"none": AP(), "relu": AP("relu"), "relu6": AP("relu6", Relu_clipped_coef=6.0), "leaky": AP("leaky_relu", Leaky_relu_alpha=0.1), "hswish": AP("hard_swish")}
KINDS = {"fp32": capi.KIND_FP32, "fp16": capi.KIND_FP16}
ROWS = (64, 128, 256)
FORMS = ROWS + ("split",)  # of fp32
KIND_FORMS = [("fp16", rows) for rows in ROWS] + [("fp32", form) for form in FORMS]


def make_case(kind, batch, ic, oc, h, w, paired=False, act="none", sparsity=0.75, seed=0):
    c = workloads.make_fp32("t", batch, ic, oc, h, w, sparsity, paired, ACTS[act], seed=seed + ic + 3 * oc)
    c.kind = KINDS[kind]
    if kind == "fp16":
        c.x = c.x.astype(np.float16)
    return c


def chunk_form(kernel, batch, im_size):
    """(rows, positions, split) of the call's workgroups."""
    form = capi.ChunkForm()
    capi.check(capi.lib().pl_sparse_conv_chunk_form_for(kernel._handle, batch, im_size, C.byref(form)))
    return form.rows, form.positions, form.split


def forced(case, rows, paired=False):
    """A kernel that runs the dense product with `rows` rows per workgroup (0: the rule's; "split": wavefronts of their own for the inputs), which
    the library confirms."""
    how = dict(float_mfma_split=capi.TUNE_ALWAYS) if rows == "split" else dict(float_mfma_rows=rows)
    kernel = make_kernel(case, force_semi=paired, tuning=capi.tuning(float_mfma=capi.TUNE_ALWAYS, **how))[0]
    assert capi.lib().pl_sparse_conv_algo_for(kernel._handle, case.batch, case.im_size) == capi.ALGO_CHUNK_MFMA
    if rows != 0:
        assert chunk_form(kernel, case.batch, case.im_size) == ((256, 64, 1) if rows == "split" else (rows, 128, 0))
    return kernel


def sums(case):
    """Sums before the activation in 64 bits, and the same with every term's magnitude."""
    to = np.float16 if case.kind == capi.KIND_FP16 else np.float32
    w = case.dense.astype(to).astype(np.float64)
    bias = np.zeros(w.shape[0]) if case.bias is None else case.bias.astype(to).astype(np.float64)
    x = case.x.astype(np.float64).reshape(case.batch, w.shape[1], -1)
    shape = (case.batch, w.shape[0]) + tuple(case.x.shape[2:])
    return (np.matmul(w, x) + bias[:, None]).reshape(shape), (np.matmul(np.abs(w), np.abs(x)) + np.abs(bias)[:, None]).reshape(shape)


def activate(v, act, dtype):
    one = lambda t: np.asarray(t).astype(dtype)  # noqa: E731
    v = one(v)
    if act == "relu":
        return np.maximum(v, one(0))
    if act == "relu6":
        return np.minimum(np.maximum(v, one(0)), one(6))
    if act == "leaky":
        return np.where(v >= 0, v, one(v * one(0.1)))
    if act == "hswish":
        return one(one(v * one(1.0 / 6.0)) * np.minimum(np.maximum(one(v + one(3)), one(0)), one(6)))
    return v


def check(case, act, got):
    """fp32: pieces of 22 bits of both factors and of three of four products (4 units of 2^-23 of every term), and one
    cut sum per 16 channels.  fp16: one rounding of a sum that is fp32's, so at most the neighbouring binary16 value,
    then the activation's own roundings (hard_swish: two factors that follow the sum and three roundings)."""
    ref, mag = sums(case)
    assert got.shape == ref.shape
    if case.kind == capi.KIND_FP32:
        tol = (6 + case.x.shape[1] / 16.0) * 2.0 ** -23 * mag
        if act == "hswish":
            tol = 2 * tol + np.abs(ref) * tol
        assert (np.abs(got - activate(ref, act, np.float64)) <= tol + 1e-30).all()
        return
    assert got.dtype == np.float16
    tol = 2.0 ** -10 * np.abs(ref) + 2.0 ** -19 * mag + 1e-7
    if act == "hswish":
        tol = (3 + 2 * np.abs(ref)) * tol
    assert (np.abs(got.astype(np.float64) - activate(ref.astype(np.float16), act, np.float16).astype(np.float64)) <= tol).all()


# (batch, ic, oc, h, w): one quad; a single row; channels off the groups of eight and chunks of 64 (fewer than one, one more than a
# chunk, odd numbers of chunks); rows off the blocks of 32 and the workgroups' 64 / 128 / 256; maps off the quads
# (partial quads of 1, 2 and 3 positions, several images per tile); exactly one tile and one position more
SHAPES = [(1, 8, 1, 2, 2), (3, 9, 33, 5, 1), (2, 63, 31, 3, 3), (1, 65, 64, 9, 6), (5, 130, 65, 7, 7), (2, 203, 129, 11, 5), (1, 256, 257, 8, 16), (1, 64, 96, 3, 43), (2, 320, 40, 14, 14), (9, 100, 300, 1, 7)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("paired", [False, True], ids=["unstructured", "semi"])
@pytest.mark.parametrize("kind, rows", KIND_FORMS)
def test_against_64_bits(kind, paired, shape, rows):
    act = sorted(ACTS)[(sum(shape) + (3 if rows == "split" else rows // 64)) % len(ACTS)]
    case = make_case(kind, *shape, paired=paired, act=act)
    check(case, act, run_hip(case, kernel=forced(case, rows, paired)))


# Calls that the rule gives to the fp32 form with wavefronts of their own for the inputs (256 rows x 16 quads, 128 channels a chunk):
# four to eleven chunks, even and odd, and channels that end inside a step of 32, a group of 8 and a chunk; rows around 32 and 256;
# tiles that cross images, partial quads, one quad, exactly one tile
SPLIT = [(1, 385, 2100, 2, 2), (3, 390, 2049, 5, 1), (2, 511, 2305, 3, 3), (1, 513, 2111, 4, 16), (1, 700, 2080, 11, 5), (9, 420, 2060, 1, 7), (1, 1030, 2100, 4, 17), (1, 1281, 2090, 5, 5), (24, 500, 513, 13, 13)]


@pytest.mark.parametrize("shape", SPLIT, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("paired", [False, True], ids=["unstructured", "semi"])
def test_fp32_wavefronts_of_their_own_for_the_inputs(paired, shape):
    act = sorted(ACTS)[sum(shape) % len(ACTS)]
    case = make_case("fp32", *shape, paired=paired, act=act)
    kernel = forced(case, 0, paired)
    assert chunk_form(kernel, case.batch, case.im_size) == (256, 64, 1)
    check(case, act, run_hip(case, kernel=kernel))


@pytest.mark.parametrize("how", ["grow", "late", "tails", "binades", "inf", "many nan"])
def test_fp32_wavefronts_of_their_own_and_hard_inputs(how):
    """New scales in the middle of a sum, inputs too small for their pieces, also in the last chunk; infinities and NaNs in few
    and in most quads."""
    case = make_case("fp32", 2, 450, 2100, 9, 7, act="none", sparsity=0.9)
    case.bias = None
    rng = np.random.RandomState(3)
    if how == "grow":
        case.x *= (2.0 ** (np.arange(450) // 60 * 4 - 14)).astype(np.float32)[None, :, None, None]
    elif how == "late":
        case.x[:, :128] = 0
        case.x[1, :440] = 0
        case.x[0, 449, 2] = 1e9
    elif how == "tails":
        case.x *= np.exp(3 * rng.standard_normal(case.x.shape)).astype(np.float32)
    elif how == "binades":
        case.x = np.ldexp(case.x, rng.randint(-60, 1, size=case.x.shape)).astype(np.float32)
    elif how == "inf":
        case.x[0, 3, 2, 1], case.x[1, 449, 8, 6] = np.inf, np.nan
    else:
        case.x[:, 200, :, 1:] = np.nan
    got = run_hip(case, kernel=forced(case, "split"))
    bad = ~np.isfinite(case.x)
    if bad.any():
        hit = np.matmul(case.dense != 0, bad.reshape(2, 450, -1)).reshape(got.shape)
        assert np.array_equal(~np.isfinite(got), hit) and hit.any() and not hit.all()
        case.x[bad] = 0
        ref, mag = sums(case)
        assert (np.abs(got - ref)[~hit] <= ((6 + 450 / 16.0) * 2.0 ** -23 * mag)[~hit]).all()
    else:
        check(case, "none", got)


def test_fp32_wavefronts_of_their_own_are_as_exact():
    """2-norm against 64 bits beside the form with 128 rows that this call would take otherwise: both add two sums of half of the
    channels, whose errors differ by chance only (5 % is 50 times what the norm of 100 000 outputs' errors scatters by)."""
    case = make_case("fp32", 16, 640, 2100, 5, 5, act="none", sparsity=0.8)
    ref, _ = sums(case)
    off = [np.linalg.norm((run_hip(case, kernel=forced(case, rows)) - ref).ravel()) for rows in (128, "split")]
    assert off[1] <= 1.05 * off[0]


@pytest.mark.parametrize("act", sorted(ACTS))
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_activations_and_a_new_bias(kind, act):
    case = make_case(kind, 3, 96, 70, 6, 7, act=act)
    case.bias = None
    kernel = forced(case, 128)
    check(case, act, run_hip(case, kernel=kernel))
    case.bias = np.linspace(-0.7, 0.9, 70).astype(np.float32)
    capi.check(capi.lib().pl_sparse_conv_set_epilogue(kernel._handle, None, case.bias.ctypes.data, None))
    check(case, act, run_hip(case, kernel=kernel))


@pytest.mark.parametrize("rows", FORMS)
@pytest.mark.parametrize("how", ["images", "late", "grow", "tails", "small", "large"])
def test_fp32_magnitudes(how, rows):
    """The scales follow the inputs: images of very different size in one tile, positions that begin with a chunk of
    zeros, channels that grow from chunk to chunk (new scales in the middle of a sum), heavy tails, both ends of the
    exponent range."""
    case = make_case("fp32", 6, 330, 40, 5, 7)
    rng = np.random.RandomState(1)
    if how == "images":
        case.x *= (10.0 ** np.linspace(-9, 9, 6)).astype(np.float32)[:, None, None, None]
    elif how == "late":
        case.x[:, :64] = 0
        case.x[2, :200] = 0
    elif how == "grow":
        case.x *= (2.0 ** (np.arange(330) // 8 % 20 - 10)).astype(np.float32)[None, :, None, None]
    elif how == "tails":
        case.x *= np.exp(2 * rng.standard_normal(case.x.shape)).astype(np.float32)
    else:
        case.bias = None
        case.x *= np.float32(1e-30 if how == "small" else 1e30)
    check(case, "none", run_hip(case, kernel=forced(case, rows)))


@pytest.mark.parametrize("rows", FORMS)
@pytest.mark.parametrize("channels", [[5], [150], [329], list(range(3, 330, 9))], ids=["first", "middle", "last", "many"])
@pytest.mark.parametrize("size", [1e4, 1e6, 1e8, 1e12, 1e30])
def test_fp32_large_inputs_stay_with_the_rows_that_read_them(size, channels, rows):
    """Every output against the magnitudes of its own row: one that reads none of the large channels must be as exact as
    without them.  Half of the inputs are zero, some positions have no other input than a large one."""
    case = make_case("fp32", 2, 330, 70, 9, 7, act="none", sparsity=0.9)
    case.bias = None
    case.x = np.maximum(case.x, 0)
    case.x[1, :, 3:5] = 0
    case.x[:, channels] = np.where(case.x[:, channels] > 0.5, -size, size)
    case.x[0, channels, 2] = 0.25
    reads = (case.dense[:, channels] != 0).any(axis=1)
    assert not reads.all() and reads.any()
    check(case, "none", run_hip(case, kernel=forced(case, rows)))


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("channels", [[5], [329], list(range(3, 330, 9))], ids=["first", "last", "many"])
def test_fp16_large_inputs_stay_with_the_rows_that_read_them(channels, rows):
    """The largest numbers beside ordinary and subnormal ones: a product with a zero weight takes no bits from the others."""
    case = make_case("fp16", 2, 330, 70, 9, 7, act="none", sparsity=0.9)
    case.bias = None
    case.x[1] *= np.float16(1e-4)
    case.x[:, channels] = np.where(case.x[:, channels] > 0, np.float16(-65504), np.float16(65504))
    reads = (case.dense[:, channels] != 0).any(axis=1)
    case.dense[reads] *= np.float32(1e-3)  # sums of these stay below the largest number
    assert not reads.all() and reads.any()
    check(case, "none", run_hip(case, kernel=forced(case, rows)))


@pytest.mark.parametrize("rows", FORMS)
@pytest.mark.parametrize("binades", [24, 60, 230])
def test_fp32_inputs_of_all_magnitudes(binades, rows):
    """Exponents spread evenly, so every position holds values that its largest one leaves few bits."""
    case = make_case("fp32", 3, 200, 40, 5, 9, act="none", sparsity=0.95)
    case.bias = None
    rng = np.random.RandomState(2)
    case.x = np.ldexp(case.x, rng.randint(-binades, 1, size=case.x.shape) + (100 if binades > 100 else 0)).astype(np.float32)
    check(case, "none", run_hip(case, kernel=forced(case, rows)))


@pytest.mark.parametrize("paired", [False, True], ids=["unstructured", "semi"])
@pytest.mark.parametrize("size", [1.0, 1e4, 1e6, 1e8, 1e12, 1e30])
def test_fp32_weights_far_below_their_rows_largest(size, paired):
    """One weight of every row is large and meets zeros: what is left are the small ones.  Where the tiles would not hold
    these, the calls stay with the walks."""
    case = make_case("fp32", 2, 330, 70, 9, 7, paired=paired, act="none", sparsity=0.9)
    case.bias = None
    case.dense[:, 100] = size
    case.x[:, 100] = 0
    case.x[1, 100, ::2] = 1
    kernel = make_kernel(case, force_semi=paired, tuning=capi.tuning(float_mfma=capi.TUNE_ALWAYS))[0]
    check(case, "none", run_hip(case, kernel=kernel))
    taken = capi.lib().pl_sparse_conv_algo_for(kernel._handle, case.batch, case.im_size) == capi.ALGO_CHUNK_MFMA
    assert taken == (size <= 1e4)


def test_fp32_the_smallest_weights():
    """Rows of subnormal weights, rows that reach from the smallest to the largest number."""
    case = make_case("fp32", 1, 64, 40, 6, 6, act="none", sparsity=0.5)
    case.bias = None
    case.dense[:20] = np.where(case.dense[:20] != 0, np.float32(2.0 ** -140) * np.sign(case.dense[:20]), 0)
    kernel = forced(case, 64)
    case.x *= np.float32(1e30)
    check(case, "none", run_hip(case, kernel=kernel))
    case.dense[20, :2] = 3e38, 2.0 ** -149
    kernel = make_kernel(case, tuning=capi.tuning(float_mfma=capi.TUNE_ALWAYS))[0]
    assert capi.lib().pl_sparse_conv_algo_for(kernel._handle, 1, 36) == capi.ALGO_ROW_WALK


def test_fp32_error_is_not_above_the_walks():
    """2-norm against 64 bits of a deep layer (one sum for all products, which the matrix cores cut off, would be 1.4 times
    the walk's)."""
    case = make_case("fp32", 16, 512, 512, 14, 14, act="none", sparsity=0.85)
    ref, _ = sums(case)
    walk = make_kernel(case, tuning=capi.tuning(float_mfma=capi.TUNE_NEVER))[0]
    off = [np.linalg.norm((run_hip(case, kernel=k) - ref).ravel()) for k in [walk] + [forced(case, rows) for rows in FORMS]]
    assert max(off[1:]) <= off[0]


@pytest.mark.parametrize("paired", [False, True], ids=["unstructured", "semi"])
@pytest.mark.parametrize("kind, rows", KIND_FORMS)
def test_infinities_and_nans_reach_only_the_rows_that_read_them(kind, paired, rows):
    """A dense product would spread them through its zero weights.  Partial quads and every part of the channels."""
    case = make_case(kind, 3, 200, 70, 9, 5, paired=paired, act="leaky", sparsity=0.9)
    case.x[0, 3, 2, 1] = np.inf
    case.x[0, 150, 8, 4] = np.nan
    case.x[1, 70, 0, 0] = -np.inf
    case.x[2, 199, 4, 4] = np.inf
    got, want = run_hip(case, kernel=forced(case, rows, paired)), run_oracle(case, oracle_pack(case, force_semi=paired))
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any() and not np.isnan(want).all()
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]) and np.isinf(want).any()
    rest = np.isfinite(want)
    case.x[~np.isfinite(case.x)] = 0
    ref, mag = sums(case)
    tol = 2.0 ** -7 if kind == "fp16" else 2.0 ** -18  # the walk's own sums among them
    assert (np.abs(got.astype(np.float64) - np.where(ref >= 0, ref, 0.1 * ref))[rest] <= (tol * mag)[rest]).all()


@pytest.mark.parametrize("paired", [False, True], ids=["unstructured", "semi"])
@pytest.mark.parametrize("kind, rows", [("fp16", 128), ("fp32", 128), ("fp32", "split")])
def test_every_number_of_quads_to_walk(kind, rows, paired):
    """Positions with a NaN from one to all of a tile, partial quads among them: rows with few quads and with many take
    different ways.  The other positions keep the bits of a call without any."""
    case = make_case(kind, 2, 200, 70, 9, 9, paired=paired, act="relu", sparsity=0.8)
    kernel = forced(case, rows, paired)
    clean = run_hip(case, kernel=kernel)
    reads = case.dense[:, 3] != 0
    if paired:
        reads = np.repeat(reads.reshape(-1, 2).any(axis=1), 2)  # the walk of a pair of rows multiplies both of its weights
    whole = case.x.copy()
    for count in (1, 2, 5, 30, 36, 40, 80, 162):
        case.x = whole.copy()
        spoiled = np.zeros((2, 81), bool)
        spoiled.reshape(-1)[np.random.RandomState(count).permutation(162)[:count]] = True
        case.x[:, 3][spoiled.reshape(2, 9, 9)] = np.nan
        got = run_hip(case, kernel=kernel)
        hit = spoiled.reshape(2, 1, 9, 9) & reads[None, :, None, None]
        assert np.isfinite(got[~hit]).all()
        near = np.abs(got.astype(np.float64) - clean)[~hit]
        assert near.max() <= (2e-2 if kind == "fp16" else 2e-5)
        if kind == "fp32":
            quads = np.repeat(np.pad(spoiled, ((0, 0), (0, 3))).reshape(2, 21, 4).any(axis=2), 4, axis=1)[:, :81].reshape(2, 1, 9, 9)
            assert np.array_equal(got[np.broadcast_to(~quads, got.shape)], clean[np.broadcast_to(~quads, got.shape)])


def microseconds(kernel, x, out):
    import torch

    best = 1e9
    for _ in range(7):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(20):
            kernel.Run(x, out)
        end.record()
        end.synchronize()
        best = min(best, start.elapsed_time(end) * 50)
    return best


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_time_with_nans(kind):
    """One NaN, and one in every position: at most 4 and 10 times a call without (fp32 1.7 and 5 times; every lane for itself
    it was 8 and 31)."""
    import torch

    case = make_case(kind, 16, 512, 512, 14, 14, act="none", sparsity=0.85)
    kernel = forced(case, 0)
    x = torch.from_numpy(case.x).cuda()
    one, every = x.clone(), x.clone()
    one[3, 77, 4, 4] = float("nan")
    every[:, 77] = float("nan")
    out = kernel.Run(x)
    microseconds(kernel, x, out)
    clean = microseconds(kernel, x, out)
    times = microseconds(kernel, one, out), microseconds(kernel, every, out)
    print("clean %.1f us, one NaN %.1f, all %.1f" % ((clean,) + times))
    assert times[0] <= 4 * clean and times[1] <= 10 * clean, (clean, times)


@pytest.mark.parametrize("shape, sparsity, paired", [((1, 1712, 1933, 36, 36), 0.8, False), ((4, 662, 1530, 22, 22), 0.7, False), ((64, 1024, 1024, 7, 7), 0.7, True)], ids=["1712", "662", "1024"])
def test_time_with_nans_and_wavefronts_of_their_own_for_the_inputs(shape, sparsity, paired):
    """A call that the rule gives to that form, with one NaN and with one in every position: not above what it would take with 128 rows (0.84
    - 0.93 and 0.9 - 1.2 times; 1.2 - 1.6 and 1 - 1.5 when every row fetched its inputs from memory)."""
    import torch

    case = make_case("fp32", *shape, paired=paired, act="none", sparsity=sparsity)
    kernel, rows = forced(case, 0, paired), forced(case, 128, paired)
    assert chunk_form(kernel, case.batch, case.im_size) == (256, 64, 1)
    x = torch.from_numpy(case.x).cuda()
    one, every = x.clone(), x.clone()
    one[0, 77, 4, 4] = float("nan")
    every[:, 77] = float("nan")
    out = kernel.Run(x)
    microseconds(kernel, x, out)
    times = [[microseconds(k, t, out) for t in (x, one, every)] for k in (kernel, rows)]
    print(", ".join("clean %.1f us, one NaN %.1f, all %.1f" % tuple(t) for t in times))
    assert times[0][1] <= 1.15 * times[1][1] and times[0][2] <= 1.4 * times[1][2], times


@pytest.mark.parametrize("paired", [False, True], ids=["unstructured", "semi"])
@pytest.mark.parametrize("ic", [450, 1024, 2048, 2049, 2500])
def test_inputs_of_walked_quads_beside_the_lists(ic, paired):
    """Few quads with a NaN, whose inputs are brought to LDS up to 2048 channels at a time: every output of theirs that reads none is a sum
    over the whole row.  Channels at the ends of what is brought at a time, positions in either half of a quad, a partial quad, all rows of
    some wavefronts and few of the last; rows without nonzeros."""
    case = make_case("fp32", 2, ic, 300, 7, 9, paired=paired, act="none", sparsity=0.9)
    case.bias = np.linspace(-1, 1, 300).astype(np.float32)
    case.dense = np.sign(case.dense) * np.maximum(np.abs(case.dense), np.float32(1e-3))  # a weight far below its row's largest would keep the layer with the walks
    case.dense[40:44] = 0
    bad = np.zeros(case.x.shape, bool)
    for image, c, y, x in ((0, 0, 0, 0), (0, min(ic - 1, 2047), 3, 3), (0, ic - 1, 6, 8), (1, min(ic - 1, 2048), 2, 6), (1, 7, 2, 7), (1, ic // 2, 5, 1)):
        bad[image, c, y, x] = True
    case.x[bad] = np.nan
    got = run_hip(case, kernel=forced(case, "split", paired))
    reads = case.dense != 0
    if paired:
        reads = np.repeat(reads.reshape(-1, 2, ic).any(axis=1), 2, axis=0)  # the walk of a pair of rows multiplies both of its weights
    hit = np.matmul(reads, bad.reshape(2, ic, -1)).reshape(got.shape)
    assert np.array_equal(~np.isfinite(got), hit) and hit.any()
    case.x[bad] = 0
    ref, mag = sums(case)
    assert (np.abs(got - ref)[~hit] <= ((6 + ic / 16.0) * 2.0 ** -23 * mag)[~hit]).all()


def test_time_with_channels_of_different_size():
    """New scales in every position, but no output that is too small: at most 1.3 times a call without (1.03; with every marked
    quad looked at output by output it was 1.4 and 1.5)."""
    import torch

    case = make_case("fp32", 64, 512, 512, 14, 14, act="none", sparsity=0.85)
    kernel = forced(case, 256)
    x = torch.from_numpy(case.x).cuda()
    gains = torch.from_numpy(np.exp(1.5 * np.random.RandomState(0).standard_normal((1, 512, 1, 1))).astype(np.float32)).cuda()
    late = x.clone()
    late[:, :64] *= 1e-3
    out = kernel.Run(x)
    microseconds(kernel, x, out)
    clean = microseconds(kernel, x, out)
    times = microseconds(kernel, x * gains, out), microseconds(kernel, late, out)
    print("clean %.1f us, channel gains %.1f, first chunk small %.1f" % ((clean,) + times))
    assert max(times) <= 1.3 * clean, (clean, times)


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_tensors_off_the_16_byte_grid(kind):
    """Tensors that start one element behind a 16-byte boundary: the same bits as the aligned call, nothing written
    outside the output."""
    import torch

    case = make_case(kind, 3, 96, 40, 9, 7)
    kernel = forced(case, 64)
    want = run_hip(case, kernel=kernel)
    dtype = torch.float32 if kind == "fp32" else torch.float16
    flat_x = torch.zeros(case.x.size + 16, dtype=dtype, device="cuda")
    x = flat_x[1:1 + case.x.size].view(case.x.shape)
    x.copy_(torch.from_numpy(case.x))
    flat_o = torch.full((want.size + 16,), 77.0, dtype=dtype, device="cuda")
    out = flat_o[1:1 + want.size].view(want.shape)
    kernel.Run(x, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), want)
    host = flat_o.cpu().numpy()
    assert host[0] == 77.0 and (host[1 + want.size:] == 77.0).all()


def test_the_rule():
    """Which calls leave the walks: many nonzeros per row, not calls of few products, never those of a handle that asks for
    a walk; a layer with hardly any nonzeros holds no dense tiles."""
    L = capi.lib()

    def algo(case, batch, im_size, **tuning):
        kernel = make_kernel(case, tuning=capi.tuning(**tuning) if tuning else None)[0]
        return L.pl_sparse_conv_algo_for(kernel._handle, batch, im_size), kernel.info()["device_bytes"]

    for kind in KINDS:
        deep = make_case(kind, 1, 512, 512, 14, 14, sparsity=0.8)
        taken, size = algo(deep, 64, 196)
        assert taken == capi.ALGO_CHUNK_MFMA
        assert algo(deep, 1, 16)[0] == capi.ALGO_ROW_WALK
        assert algo(deep, 64, 196, walk_tiled=capi.TUNE_RULE, walk_pairs=capi.TUNE_ALWAYS)[0] == capi.ALGO_ROW_WALK
        never, walk_size = algo(deep, 64, 196, float_mfma=capi.TUNE_NEVER)
        assert never == capi.ALGO_ROW_WALK and walk_size < size
        assert algo(make_case(kind, 1, 512, 512, 4, 4, sparsity=0.98), 64, 196)[0] == capi.ALGO_ROW_WALK
    # few rows: the product takes longer than its times for more rows say
    assert algo(make_case("fp32", 1, 1184, 62, 9, 11, sparsity=0.82), 38, 99)[0] == capi.ALGO_ROW_WALK
    assert algo(make_case("fp32", 1, 800, 64, 33, 33, sparsity=0.88), 7, 1089)[0] == capi.ALGO_ROW_WALK
    assert algo(make_case("fp32", 1, 1624, 40, 8, 8, sparsity=0.76), 10, 2209)[0] == capi.ALGO_CHUNK_MFMA
    # by the time of the form that runs: 26 us with wavefronts of its own for the inputs, 30 without, 44 as a walk
    wide = make_case("fp32", 1, 1088, 736, 15, 15, sparsity=0.95)
    assert algo(wide, 19, 225)[0] == capi.ALGO_CHUNK_MFMA and algo(wide, 19, 225, float_mfma_split=capi.TUNE_NEVER)[0] == capi.ALGO_ROW_WALK
    # few nonzeros per row
    assert algo(make_case("fp32", 1, 96, 192, 8, 8, sparsity=0.9), 1, 3136)[0] == capi.ALGO_ROW_WALK
    assert algo(make_case("fp16", 1, 96, 200, 8, 8, sparsity=0.86), 102, 400)[0] == capi.ALGO_ROW_WALK
    with pytest.raises(capi.SparseConvError):
        make_kernel(make_case("fp32", 1, 16, 16, 4, 4), tuning=capi.tuning(float_mfma_rows=96))


def test_no_tiles_for_layers_that_no_call_can_use_them_with():
    """20000 x 14000 weights are beyond the kernel's 32-bit offsets: 1.1 GB of tiles otherwise."""
    oc, ic = 14000, 20000
    weights = pla.SparseWeights(np.zeros(0, np.float32), np.zeros(oc, np.uint32), np.zeros(0, np.int32), 0, 0, oc, ic, 49)
    kernel = pla.SparseConvKernel(pla.SparseConvParam(weights), tuning=capi.tuning(float_mfma=capi.TUNE_ALWAYS))
    kernel.PrepareForRun()
    assert kernel.info()["device_bytes"] < 2 ** 27  # the lists of 14000 empty rows take 35 MB
    assert capi.lib().pl_sparse_conv_algo_for(kernel._handle, 1, 49) == capi.ALGO_ROW_WALK
