"""The int8 kernel that takes the input channels chunk by chunk, against the CPU oracle through the C ABI, bit for
bit, at each of its three tile widths and in the form with wavefronts of its own for the activations: channel counts around a group of 16, a step of 64 and a chunk, one to 25 chunks
(each way the loop over the chunks can end), rows around a tile of 16 and a group of 128, maps of four positions and more
with every remainder modulo four, tiles of whole images and tiles that cross images; tensors off the 16-byte grid."""
import ctypes as C
import sys

import numpy as np
import pytest

from helpers import ALGO_NAMES, capi, workloads, pla, make_kernel, oracle_pack, run_hip, run_oracle, assert_same

pytestmark = pytest.mark.gpu

AP = pla.ActivationParam
KINDS = {"acc32": capi.KIND_INT8_ACC32, "fp32out": capi.KIND_INT8_FP32, "int8out": capi.KIND_INT8_INT8}
WIDTHS = (64, 128, 256)
# (batch, ic, oc, h, w).  64-position tiles hold chunks of 512 channels, 128: 256, 256: 128.
SMALL = [(1, 513, 17, 2, 2), (3, 520, 1, 1, 5), (5, 527, 127, 2, 3), (2, 600, 129, 7, 7), (1, 1024, 16, 14, 14), (1, 1025, 40, 9, 11), (9, 1536, 33, 3, 3), (1, 1900, 24, 5, 6),
         (1, 2049, 130, 5, 13), (2, 2561, 20, 8, 8), (1, 3100, 24, 1, 7), (4, 79, 140, 5, 9), (2, 65, 200, 3, 5), (1, 512, 512, 14, 14), (1, 200, 72, 12, 12)]
LARGE = [(16, 520, 4096, 8, 8), (3, 1030, 2200, 17, 17), (2, 130, 4096, 31, 33), (2, 330, 4096, 31, 33), (2, 900, 4096, 32, 32)]


def chunk_case(shape, kind, act, paired, seed):
    batch, ic, oc, h, w = shape
    case = workloads.make_int8("chunk", batch, ic, oc, h, w, 0.8, paired, AP() if kind == "acc32" else act, out_int8=(kind == "int8out"), seed=seed,
                               output_scale=0.2 * float(np.sqrt(ic / 64.0)) if kind == "int8out" else 1.0)
    case.kind = KINDS[kind]
    return case


def chunk_form(kernel, batch, im_size):
    """(rows, positions, split) of the call's workgroups."""
    form = capi.ChunkForm()
    capi.check(capi.lib().pl_sparse_conv_chunk_form_for(kernel._handle, batch, im_size, C.byref(form)))
    return form.rows, form.positions, form.split


def chunk_kernel(case, width):
    """A kernel that runs chunk by chunk on tiles of `width` positions (0: the rule's, "split": the form with wavefronts of its own for the
    activations), which the library confirms."""
    how = dict(chunk_split=capi.TUNE_ALWAYS) if width == "split" else dict(chunk_positions=width)
    kernel, _ = make_kernel(case, tuning=capi.tuning(chunk_mfma=capi.TUNE_ALWAYS, **how))
    assert capi.lib().pl_sparse_conv_algo_for(kernel._handle, case.batch, case.im_size) == capi.ALGO_CHUNK_MFMA
    if width != 0:
        assert chunk_form(kernel, case.batch, case.im_size) == ((256, 128, 1) if width == "split" else (128, width, 0))
    return kernel


def widths(case):
    return WIDTHS + (("split",) if case.im_size >= 16 else ())


def check(shape, kind, act, paired, seed):
    print("CASE chunk", shape, kind, file=sys.stderr, flush=True)
    batch, _, _, h, w = shape
    case = chunk_case(shape, kind, act, paired, seed)
    few = case.x[:1] if batch * h * w > 1000 else case.x
    want = run_oracle(case, oracle_pack(case), x=few)
    last = run_oracle(case, oracle_pack(case), x=case.x[-1:]) if len(few) != batch else None
    for width in (0,) + widths(case):
        got = run_hip(case, kernel=chunk_kernel(case, width))
        assert_same(case, got[:len(few)], want, "chunk %s %s, width %s" % (shape, kind, width))
        if last is not None:  # it ends the last tile
            assert_same(case, got[-1:], last, "chunk %s %s, width %s, last image" % (shape, kind, width))


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("shape", SMALL, ids=lambda s: "x".join(map(str, s)))
def test_small_calls(shape, kind):
    check(shape, kind, [AP("relu"), AP("hard_swish"), AP("leaky_relu", Leaky_relu_alpha=0.1), AP("relu6")][shape[1] % 4], shape[2] % 2 == 0, shape[1])


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("shape", LARGE, ids=lambda s: "x".join(map(str, s)))
def test_large_calls(shape, kind):
    check(shape, kind, AP("relu"), False, shape[1])


# The form with wavefronts of its own for the activations (256 rows x eight blocks of 16 positions, 256 channels a chunk):
# channels around a group of 16, a step of 64 and a chunk, each number of chunks that its loops can end with, rows around a tile of 16, a
# wavefront's 32 and a workgroup's 256, maps of one block, of blocks that overlap by 1 - 15 positions and of more than a tile, tiles that cross
# images and are not full.
SPLIT = [(1, 129, 1, 4, 4), (2, 191, 31, 1, 17), (3, 256, 33, 5, 5), (1, 257, 255, 1, 31), (5, 272, 256, 4, 8), (2, 320, 257, 3, 11), (9, 500, 15, 7, 7), (1, 513, 48, 14, 14),
         (3, 768, 17, 9, 15), (2, 770, 300, 1, 18), (1, 1000, 129, 10, 10), (7, 1025, 40, 4, 4), (1, 1281, 20, 12, 13), (2, 1601, 520, 6, 6)]


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("shape", SPLIT, ids=lambda s: "x".join(map(str, s)))
def test_wavefronts_of_their_own_for_the_activations(shape, kind):
    print("CASE chunk split", shape, kind, file=sys.stderr, flush=True)
    case = chunk_case(shape, kind, [AP("relu"), AP("leaky_relu", Leaky_relu_alpha=0.1)][shape[1] % 2], shape[2] % 2 == 0, shape[1])
    want = run_oracle(case, oracle_pack(case))
    for width in (0, "split"):
        assert_same(case, run_hip(case, kernel=chunk_kernel(case, width)), want, "chunk split %s %s, width %s" % (shape, kind, width))


# (batch, ic, oc, h, w) and the form the rule takes on 256 CUs: the widest tiles with four to eight chunks of 128 channels, on maps larger and
# smaller than a tile; calls of one round that the other form would and would not make shorter
RULE = [(121, 576, 320, 18, 18, (128, 256, 0)), (107, 420, 112, 18, 18, (128, 256, 0)), (120, 992, 672, 9, 9, (128, 256, 0)), (16, 500, 128, 35, 31, (128, 128, 0)), (16, 2048, 2048, 14, 14, (256, 128, 1)),
        (60, 900, 384, 13, 13, (256, 128, 1)), (1, 512, 512, 14, 14, (128, 64, 0)), (1, 1590, 1406, 40, 40, (128, 128, 0)), (9, 1905, 412, 33, 20, (128, 128, 0)),
        (20, 162, 1888, 11, 11, (256, 128, 1)), (18, 192, 142, 35, 35, (256, 128, 1))]


@pytest.mark.parametrize("kind", ["fp32out", "int8out"])
@pytest.mark.parametrize("call", RULE, ids=lambda c: "x".join(map(str, c[:5])))
def test_the_form_the_rule_takes(call, kind):
    """By the rule, with the form that the library names, and forced, where that is a tile width: the bits of the block kernel, and of the
    oracle on the first and the last image."""
    shape, form = call[:5], call[5]
    print("CASE chunk rule", shape, kind, file=sys.stderr, flush=True)
    case = chunk_case(shape, kind, AP("relu"), False, shape[1])
    kernel = chunk_kernel(case, 0)
    assert chunk_form(kernel, case.batch, case.im_size) == form
    got = run_hip(case, kernel=kernel)
    for image in (0, shape[0] - 1):
        assert_same(case, got[image:image + 1], run_oracle(case, oracle_pack(case), x=case.x[image:image + 1]), "chunk rule %s %s" % (shape, kind))
    assert_same(case, got, run_hip(case, algo=capi.ALGO_BLOCK_MFMA), "chunk rule %s %s, block kernel" % (shape, kind))
    # a width that a field names is that of the form with three widths, and the switch keeps the other one out
    for width in WIDTHS:
        assert chunk_form(chunk_kernel(case, width), case.batch, case.im_size) == (128, width, 0)
    never, _ = make_kernel(case, tuning=capi.tuning(chunk_mfma=capi.TUNE_ALWAYS, chunk_split=capi.TUNE_NEVER))
    assert chunk_form(never, case.batch, case.im_size)[2] == 0
    assert_same(case, run_hip(case, kernel=never), got, "chunk rule %s %s, chunk_split NEVER" % (shape, kind))
    # calls of other kernels have none
    block, _ = make_kernel(case, algo=capi.ALGO_BLOCK_MFMA)
    assert capi.lib().pl_sparse_conv_chunk_form_for(block._handle, case.batch, case.im_size, C.byref(capi.ChunkForm())) == capi.PL_ERR_UNSUPPORTED


# maps with every remainder modulo four, a last tile that is not full and rows that end inside a tile
@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("shape", [(3, 130, 37, 6, 6), (2, 200, 20, 5, 9), (3, 520, 129, 3, 6), (2, 77, 30, 3, 13)], ids=lambda s: "x".join(map(str, s)))
def test_tensors_off_the_grid_and_their_surroundings(shape, kind):
    """x and out start 1 - 3 elements behind a 16-byte boundary; the bytes around out stay as they were."""
    import torch

    print("CASE chunk off the grid", shape, kind, file=sys.stderr, flush=True)
    case = chunk_case(shape, kind, AP("relu"), False, shape[1])
    want = run_oracle(case, oracle_pack(case))
    batch, ic, oc, h, w = shape
    fill, dtype = (77, torch.int8) if kind == "int8out" else (77, torch.int32) if kind == "acc32" else (77.0, torch.float32)
    for width in widths(case):
        kernel = chunk_kernel(case, width)
        for shift in (1, 2, 3):
            guard = 64 + shift
            x = torch.randint(-127, 128, (case.x.size + 2 * guard,), dtype=torch.int8, device="cuda")
            x[guard:guard + case.x.size] = torch.from_numpy(case.x.reshape(-1)).cuda()
            out = torch.full((want.size + 2 * guard,), fill, dtype=dtype, device="cuda")
            kernel.Run(x[guard:guard + case.x.size].view(case.x.shape), out[guard:guard + want.size].view(want.shape))
            host = out.cpu().numpy()
            assert (host[:guard] == fill).all() and (host[guard + want.size:] == fill).all(), (width, shift)
            assert_same(case, host[guard:guard + want.size].reshape(want.shape), want, "chunk off the grid %s %s %s %d" % (shape, kind, width, shift))


def test_the_choice_is_reported_and_can_be_overridden():
    """pl_sparse_conv_algo_for names the kernel for the calls that the rule gives it out of each of the three others'
    range, and tuning.chunk_mfma forces it and keeps it out."""
    L = capi.lib()
    case = workloads.make_int8("chunk", 1, 512, 512, 14, 14, 0.85, False, AP(), out_int8=False, seed=3)
    never, _ = make_kernel(case, tuning=capi.tuning(chunk_mfma=capi.TUNE_NEVER))
    rule, _ = make_kernel(case)
    always, _ = make_kernel(case, tuning=capi.tuning(chunk_mfma=capi.TUNE_ALWAYS))
    for batch, im_size, other, by_rule in ((1, 196, "image_mfma", True), (64, 196, "image_mfma", False), (4, 50, "row_walk", True), (20, 50, "block_mfma", True), (64, 784, "block_mfma", False)):
        picked = [ALGO_NAMES[capi.check(L.pl_sparse_conv_algo_for(k._handle, batch, im_size))] for k in (never, rule, always)]
        assert picked == [other, "chunk_mfma" if by_rule else other, "chunk_mfma"], (batch, im_size, picked)
    assert L.pl_sparse_conv_algo_for(always._handle, 64, 3) == capi.ALGO_ROW_WALK  # no quad of positions
    assert np.array_equal(run_hip(case, kernel=always), run_hip(case, kernel=never))
    # a report only
    with pytest.raises(capi.SparseConvError) as e:
        make_kernel(case, capi.ALGO_CHUNK_MFMA)
    assert e.value.code == capi.PL_ERR_BAD_ARG


def test_a_kernel_that_a_tuning_field_names_keeps_its_calls():
    L = capi.lib()
    # (batch, ic, positions, the kernel without this one, fields that name its form)
    for batch, ic, im_size, other, fields in ((1, 512, 50, "row_walk", ("walk_tile", "walk_threads", "walk_slices")), (20, 512, 50, "block_mfma", ("mfma_stream", "mfma_sub_tiles", "mfma_tile_quads", "mfma_narrow_i8_stores", "wg_slots")),
                                              (1, 512, 196, "image_mfma", ("image_kernel", "image_min_items", "image_tr_regroup"))):
        case = workloads.make_int8("chunk", 1, ic, 512, 1, im_size, 0.85, False, AP(), out_int8=True, seed=3)
        for field in (None,) + fields:
            value = {"walk_tile": 64, "walk_threads": 256, "mfma_tile_quads": 16, "wg_slots": 512}.get(field, 1)  # 1: the switches' NEVER, one item, the first image kernel
            kernel, _ = make_kernel(case, tuning=capi.tuning(**({field: value} if field else {})))
            assert ALGO_NAMES[capi.check(L.pl_sparse_conv_algo_for(kernel._handle, batch, im_size))] == (other if field else "chunk_mfma"), (other, field)


# (batch, ic, oc, h, w, output, kernel)
BLOCKS = [(666, 424, 105, 16, 16, "fp32out", "block_mfma"), (2064, 357, 105, 8, 8, "fp32out", "block_mfma"), (65, 492, 101, 32, 32, "fp32out", "block_mfma"), (28, 453, 519, 36, 36, "fp32out", "block_mfma"),
          (28, 640, 1613, 25, 20, "fp32out", "block_mfma"), (155, 522, 865, 20, 20, "fp32out", "block_mfma"), (182, 443, 292, 14, 14, "int8out", "chunk_mfma"), (70, 320, 263, 12, 12, "fp32out", "chunk_mfma"), (28, 640, 1613, 25, 20, "int8out", "chunk_mfma"),
          (24, 512, 384, 28, 28, "fp32out", "block_mfma"), (12, 512, 384, 28, 28, "fp32out", "chunk_mfma"), (60, 512, 512, 18, 18, "fp32out", "chunk_mfma"), (40, 257, 768, 14, 16, "int8out", "chunk_mfma"), (5, 640, 900, 36, 36, "fp32out", "chunk_mfma"),
          (18, 352, 1152, 27, 27, "fp32out", "chunk_mfma"), (36, 320, 700, 30, 30, "fp32out", "block_mfma"), (12, 416, 876, 37, 37, "fp32out", "chunk_mfma"), (30, 422, 1004, 25, 25, "fp32out", "chunk_mfma"), (10, 1344, 896, 28, 28, "fp32out", "chunk_mfma"), (20, 700, 97, 40, 40, "fp32out", "chunk_mfma")]


@pytest.mark.parametrize("call", BLOCKS, ids=lambda c: "x".join(map(str, c[:6])))
def test_the_rule_beside_the_block_kernel(call):
    """More than 256 channels and 96 rows over many positions, on a device of 256 CUs."""
    batch, ic, oc, h, w, kind, chosen = call
    kernel, _ = make_kernel(chunk_case((1, ic, oc, h, w), kind, AP("relu"), False, 3))
    assert ALGO_NAMES[capi.check(capi.lib().pl_sparse_conv_algo_for(kernel._handle, batch, h * w))] == chosen


@pytest.mark.parametrize("batch, oc, chosen", [(32, 1024, "chunk_mfma"), (33, 1024, "image_mfma"), (64, 1024, "image_mfma"), (65, 1024, "chunk_mfma"), (33, 2048, "chunk_mfma"), (171, 384, "chunk_mfma"), (67, 1920, "image_mfma"), (85, 1408, "image_mfma"), (173, 640, "image_mfma"), (130, 1024, "chunk_mfma")])
@pytest.mark.parametrize("out_int8", [False, True], ids=["fp32", "int8"])
def test_1024_channels_on_maps_of_49_positions(batch, oc, chosen, out_int8):
    """More than one round of the image kernel's items and two thirds as many rounds here, or at most half of one, on a device of 256 CUs; the same bits as that kernel's."""
    case = workloads.make_int8("rounds", batch, 1024, oc, 7, 7, 0.9, False, AP(), out_int8=out_int8, seed=batch)
    rule, image = make_kernel(case)[0], make_kernel(case, tuning=capi.tuning(chunk_mfma=capi.TUNE_NEVER))[0]
    assert ALGO_NAMES[capi.check(capi.lib().pl_sparse_conv_algo_for(rule._handle, batch, 49))] == chosen
    assert ALGO_NAMES[capi.check(capi.lib().pl_sparse_conv_algo_for(image._handle, batch, 49))] == "image_mfma"
    assert_same(case, run_hip(case, kernel=rule), run_hip(case, kernel=image))


def test_weight_tiles_are_held_where_some_call_can_use_them():
    """Device memory of a handle: tiles of 16 rows x 64 channels in whole chunks of 512 channels, none where a tuning field
    gives every call to another kernel."""
    case = workloads.make_int8("chunk", 1, 520, 40, 7, 7, 0.85, False, AP(), out_int8=True, seed=3)

    def size(algo, **fields):
        return make_kernel(case, algo, tuning=capi.tuning(**fields))[0].info()["device_bytes"]

    assert size(capi.ALGO_AUTO) - size(capi.ALGO_AUTO, chunk_mfma=capi.TUNE_NEVER) == 3 * 16 * 1024  # 40 rows: three tiles
    assert size(capi.ALGO_BLOCK_MFMA, mfma_tile_quads=16) == size(capi.ALGO_BLOCK_MFMA, mfma_tile_quads=16, chunk_mfma=capi.TUNE_NEVER)
    assert size(capi.ALGO_AUTO, mfma_tile_quads=16) == size(capi.ALGO_AUTO)  # few positions: in place of the walk
