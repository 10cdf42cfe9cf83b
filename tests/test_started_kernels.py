"""Which kernel a launch starts where it is another than the one that its records name (no GPU): both sides of every line of the rules."""
import pytest

from orinfer_amd import lib
from .started_util import BIG, MID_2, MID_4, RUNS, reported, started


def projection(codec, rows, n, k, **variant):
    variant = dict(dict(M=max(rows, 512), dynamic_rows=True, workspace=True), **variant)
    return lib.Kernel("e8p_q4_projection" if codec == "q4" else "int8_projection", N=n, K=k, **variant)


# by what the GEMV has for the codes: no replicated tables, eight lanes to a channel, sixteen
@pytest.mark.parametrize("packed_k,n,below,first", [
    (0, 4096, 2688, 2816), (0, 4097, 8064, 8320), (0, 8192, 8064, 8320), (0, 8193, 3968, 4224), (0, 12288, 3968, 4224), (0, 16385, 5504, 5760), (0, 20480, 5504, 5760),
    (128, 4096, 1280, 2304), (64, 16, 1280, 2304), (128, 4097, 2816, 3328), (128, 8192, 2304, 3328), (128, 8193, 3840, 4224),
    (128, 12289, 17280, None), (0, 12289, 17280, None), (0, 20481, 17280, None)])  # four blocks of channels to a CU, six
def test_one_row_of_codes_takes_the_channel_runs_from_a_k_on(packed_k, n, below, first):
    for rows in (1, 4):
        for k, runs in ((below, False), (first, True)):
            if k is not None:
                kernel = projection("q4", 1, n, k, M=rows, packed_k=packed_k, dynamic_rows=rows > 1, workspace=False)
                (only,) = started(kernel, 1)
                assert (only[1:] == (512, RUNS)) == runs and (only != reported(kernel, 1)) == runs, k


@pytest.mark.parametrize("codec,packed_k,n,inside,outside", [  # (rows, K) on both sides of a line
    ("q4", 0, 1030, (16, 2816), (16, 2688)), ("q4", 128, 1030, (17, 2304), (17, 2176)),                                         # one block of channels to a CU
    ("q4", 128, 4100, (16, 8192), (16, 8064)), ("q4", 128, 4100, (17, 12288), (17, 12160)),                                     # two
    ("q4", 0, 12288, (2, 4224), (2, 3968)), ("q4", 0, 8193, (2, 4224), (2, 4096)),                                              # three
    ("q4", 0, 8300, (96, 2048), (96, 1920)), ("q4", 64, 4300, (256, 2048), (256, 1920)), ("q4", 0, 8192, (270, 1536), (270, 1408)),
    ("w8", 0, 9000, (128, 8192), (128, 8320)), ("w8", 0, 9000, (128, 1024), (129, 1024)), ("w8", 0, 1000, (120, 8320), (121, 8320))])
def test_more_rows_that_take_the_channel_runs(codec, packed_k, n, inside, outside):
    for (rows, k), runs in ((inside, True), (outside, False)):
        kernel = projection(codec, rows, n, k, **({"packed_k": packed_k} if codec == "q4" else {}))
        assert (started(kernel, rows)[0][2] == RUNS) == runs, (rows, k)
        if runs:
            assert started(kernel, rows) != [reported(kernel, rows)]


@pytest.mark.parametrize("rows,n,k,instead", [(2, 12289, 1152, True), (2, 12288, 1152, False), (3, 12289, 1152, True), (4, 12289, 1152, True), (5, 12289, 1152, False)])
def test_few_rows_of_codes_that_take_the_streaming_kernel(rows, n, k, instead):
    kernel = projection("q4", rows, n, k)
    assert started(kernel, rows) == [(-(-n // 32), 512, 0)]  # (where it is not the rule's doing it is what the records name)
    assert (started(kernel, rows) != [reported(kernel, rows)]) == instead


@pytest.mark.parametrize("codec,rows,n,k,variant,tiles,parts", [  # tiles 0: not these tiles
    ("w8", 129, 8704, 256, {}, 136, 1), ("w8", 128, 8704, 256, {}, 0, 0),                                                          # above 128 rows
    ("w8", 512, 16384, 512, {}, 512, 1), ("w8", 513, 16384, 512, {}, 0, 0), ("w8", 2050, 2064, 256, {}, 289, 1),                   # two to a CU
    ("w8", 513, 528, 128, {}, 25, 1), ("w8", 513, 528, 192, {}, 0, 0), ("w8", 513, 528, 256, dict(algorithm="mfma"), 0, 0),        # whole steps, no kernel by name
    ("w8", 520, 250, 14336, {}, 10, 8), ("w8", 520, 250, 14336, dict(split_k=False), 10, 1), ("w8", 520, 250, 14336, dict(workspace=False), 10, 1),
    ("w8", 641, 1930, 14336, {}, 96, 5), ("q4", 770, 256, 8320, {}, 14, 8), ("q4", 513, 528, 512, {}, 25, 1), ("q4", 512, 528, 512, {}, 0, 0),
    ("q4", 513, 528, 512, dict(workspace=False), 0, 0), ("q4", 1100, 4112, 640, dict(packed_k=64), 297, 1),
    ("q4", 513, 6144, 10880, {}, 240, 1), ("q4", 513, 6144, 11008, {}, 0, 0)])                                                     # what the Workspace holds
def test_launches_that_take_the_128_by_128_tiles(codec, rows, n, k, variant, tiles, parts):
    kernel = projection(codec, rows, n, k, **variant)
    kernels = started(kernel, rows)
    if not tiles:
        assert not {shared for _, _, shared in kernels} & {MID_4, MID_2}
        return
    assert len(kernels) == (codec == "q4") + 1 + (parts > 1)  # decoded once, the tiles, the sum of their parts
    assert kernels[codec == "q4"] == (tiles * parts, 256, MID_4 if tiles * parts <= 256 else MID_2)
    if parts > 1:
        assert kernels[-1] == (4 * tiles, 256, 0)
    assert reported(kernel, rows) not in kernels
    assert kernel.workspace_bytes(rows) == (n * k if codec == "q4" else 0) + (tiles * parts * 65536 if parts > 1 else 0)


@pytest.mark.parametrize("experts,segments", [(4, 8), (8, 8), (9, 12), (16, 12), (17, 16), (1024, 16)])
def test_segmented_metadata_in_one_launch_up_to_a_line(experts, segments):
    kernel = lib.Kernel("route_metadata", M=40000, E=experts, top_k=1, block_m=32, slot_maps=True, workspace=True, dynamic_rows=True)
    assert started(kernel, 1024 * segments) == [(segments, 1024, 18 * experts * 4)]
    assert started(kernel, 1024 * segments + 1) == [(segments + 1, 1024, 16 * experts * 4), (segments + 1, 1024, 0)]


@pytest.mark.parametrize("rows,n,k,narrow", [  # tiles of the routed rows and half of the experts, eight XCDs
    (28 * 128 + 127, 2048, 1024, True), (29 * 128, 2048, 1024, False), (20 * 128, 2304, 512, True), (21 * 128, 2304, 512, False), (12 * 128, 4096, 256, True), (13 * 128, 4096, 256, False),
    (252 * 128, 256, 128, True), (253 * 128, 256, 128, False)])
def test_units_of_128_channels_up_to_a_line(rows, n, k, narrow):
    tiles = rows // 128 + 8
    kernel = lib.Kernel("e8p_decode_grouped", rows=rows, E=8, tiles=tiles, N=n, K=k, block_m=128, tile_units=True)
    assert [grid for grid, _, _ in started(kernel)] == [-(-tiles // 8) * 8 * -(-n // (128 if narrow else 256))]
    assert reported(kernel)[0] == -(-tiles // 8) * 8 * -(-n // 256)


def test_a_launch_by_record_starts_what_is_reported():
    """Kernels by name and rows that no rule takes elsewhere."""
    for kernel, rows in ((projection("w8", 513, 16384, 512), 513), (projection("q4", 40, 8300, 2048), 40), (projection("q4", 128, 8704, 512, algorithm="wide", M=128), 128),
                         (lib.Kernel("activation_quantization", K=512), 0)):
        assert started(kernel, rows) == [reported(kernel, rows)]
    assert started(projection("w8", 513, 16384, 512), 513) == [(192, 512, BIG)]
