"""The int8 kernel that takes the input channels chunk by chunk, against the CPU oracle through the C ABI, bit for
bit: channel counts around a group of 16, a step of 64 and a chunk, one to seven chunks (each way the loop over the
chunks can end), rows around a tile of 16 and a group of 128, maps of four positions and more with every remainder
modulo four, tiles of whole images and tiles that cross images, and each of the three tile widths."""
import sys

import numpy as np
import pytest

from helpers import ALGO_NAMES, capi, workloads, pla, make_kernel, oracle_pack, run_hip, run_oracle, assert_same

pytestmark = pytest.mark.gpu

AP = pla.ActivationParam
KINDS = {"acc32": capi.KIND_INT8_ACC32, "fp32out": capi.KIND_INT8_FP32, "int8out": capi.KIND_INT8_INT8}
# (batch, ic, oc, h, w).  64-position tiles hold chunks of 512 channels, 128: 256, 256: 128.
NARROW = [(1, 513, 17, 2, 2), (3, 520, 1, 1, 5), (5, 527, 127, 2, 3), (2, 600, 129, 7, 7), (1, 1024, 16, 14, 14), (1, 1025, 40, 9, 11), (9, 1536, 33, 3, 3),
          (1, 2049, 130, 5, 13), (2, 2561, 20, 8, 8), (1, 3100, 24, 1, 7), (4, 79, 140, 5, 9), (2, 65, 200, 3, 5), (1, 512, 512, 14, 14), (1, 200, 72, 12, 12)]
MIDDLE = [(16, 520, 4096, 8, 8), (3, 1030, 2200, 17, 17)]
WIDE = [(2, 130, 4096, 31, 33), (2, 330, 4096, 31, 33), (2, 900, 4096, 32, 32)]


def check(shape, kind, act, paired, seed):
    print("CASE chunk", shape, kind, file=sys.stderr, flush=True)
    batch, ic, oc, h, w = shape
    k = KINDS[kind]
    case = workloads.make_int8("chunk", batch, ic, oc, h, w, 0.8, paired, AP() if kind == "acc32" else act, out_int8=(kind == "int8out"), seed=seed,
                               output_scale=0.2 * float(np.sqrt(ic / 64.0)) if kind == "int8out" else 1.0)
    case.kind = k
    got = run_hip(case, capi.ALGO_BLOCK_MFMA)
    few = case.x[:1] if batch * h * w > 1000 else case.x
    assert_same(case, got[:len(few)], run_oracle(case, oracle_pack(case), x=few), "chunk %s %s" % (shape, kind))
    if len(few) != batch:  # the last image too: it ends the last tile
        assert_same(case, got[-1:], run_oracle(case, oracle_pack(case), x=case.x[-1:]), "chunk %s %s, last image" % (shape, kind))


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("shape", NARROW, ids=lambda s: "x".join(map(str, s)))
def test_narrow_tiles(shape, kind):
    check(shape, kind, [AP("relu"), AP("hard_swish"), AP("leaky_relu", Leaky_relu_alpha=0.1), AP("relu6")][shape[1] % 4], shape[2] % 2 == 0, shape[1])


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("shape", MIDDLE + WIDE, ids=lambda s: "x".join(map(str, s)))
def test_wide_tiles(shape, kind):
    check(shape, kind, AP("relu"), False, shape[1])


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


def test_weight_tiles_are_held_where_some_call_can_use_them():
    """Device memory of a handle: tiles of 16 rows x 64 channels in whole chunks of 512 channels, none where a tuning field
    gives every call to another kernel."""
    case = workloads.make_int8("chunk", 1, 520, 40, 7, 7, 0.85, False, AP(), out_int8=True, seed=3)

    def size(algo, **fields):
        return make_kernel(case, algo, tuning=capi.tuning(**fields))[0].info()["device_bytes"]

    assert size(capi.ALGO_AUTO) - size(capi.ALGO_AUTO, chunk_mfma=capi.TUNE_NEVER) == 3 * 16 * 1024  # 40 rows: three tiles
    assert size(capi.ALGO_BLOCK_MFMA, mfma_tile_quads=16) == size(capi.ALGO_BLOCK_MFMA, mfma_tile_quads=16, chunk_mfma=capi.TUNE_NEVER)
    assert size(capi.ALGO_AUTO, mfma_tile_quads=16) == size(capi.ALGO_AUTO)  # few positions: in place of the walk
