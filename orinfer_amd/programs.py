"""Kernel programs: ordered launch lists for one quantized linear and for one MoE expert layer.

The engine runs a *program* -- an ordered list of kernel records whose buffers it owns
(crates/orinfer-engine/src/backend/cuda/executor.rs:1095-1124).  These classes are that list for
the paths of this library, with every buffer allocated once up front (torch is used only for
device memory and the stream), so `run()` only enqueues and can be captured in a graph.
Program order of the expert layer follows python/orinfer_build/models/flash_next (router top-k,
histogram, offsets, tiles, A8, dispatch, grouped gate_up, SwiGLU->A8, grouped down, combine).
"""
import math

import numpy as np
import torch

from . import codebook
from .lib import ORX_ERR_BAD_VARIANT, Kernel, OrxError, current_stream


def _dev(array):
    a = np.ascontiguousarray(array)
    view = {np.dtype(np.uint16): np.int16, np.dtype(np.uint32): np.int32}.get(a.dtype)
    return torch.from_numpy(a.view(view) if view else a).cuda()


PANEL_ROWS = 1024


def panels_pay(rows, n, k, cus):
    """Whether quantiser and projection of two-stage codes are faster over token panels than row-major (time of the pair over panels / row-major, 256 CUs,
    by blocks of 16 channels to a CU).
    65-128 rows: 4 to 5 blocks 0.65-0.84; more than 6 0.82-0.98 from 97 rows on, below 0.85-1.04; up to 2 blocks 0.77-0.96 above 112 rows, 0.81-0.98 above 96 up to
    K = 5120, 0.83-0.98 at K = 1024, otherwise to 1.3; 2 to 4 blocks 0.76-0.87 at K = 1024, 0.79-0.96 at K = 2048 above 80 rows, otherwise to 1.27; 5 to 6 1.0-1.1.
    Where the channel runs fill one round (up to 240 rows of up to 2 blocks, 257-384 of up to 1.3): up to one block 0.90-0.95 at K = 1024, 0.96-1.3 beyond;
    1.2 to 1.5 0.87-0.97 up to K = 2048, 0.96-1.12 beyond; 1.75 and 2 0.81-0.98; 257-384 rows 1.05-1.3.
    Elsewhere up to 512 rows: up to one block 1.1-2.2, wider 0.36-0.98 (5120 x 12288 1.01).  513-1024 rows: up to one block 0.44-1.02 up to K = 4096, 0.75-1.5
    beyond; wider 0.64-0.99 (5120 x 8192 and x 12288 at 640-768 rows 1.0-1.12, K below 2048 at 1024 rows 0.66-1.13).  Beyond 1024 rows decoding once is mostly faster
    (1280 rows 0.72-1.5)."""
    if not 64 < rows <= PANEL_ROWS:
        return False
    blocks = -(-n // 16)
    if rows <= 128:
        if blocks <= 2 * cus:
            return rows > 112 or k <= (5120 if rows > 96 else 1024)
        if blocks <= 4 * cus:
            return k <= (2048 if rows > 80 else 1024)
        return blocks <= 5 * cus or (blocks > 6 * cus and rows > 96)
    if rows > 512:
        if blocks <= cus:
            return k <= 4096
        return (rows <= 768 or k >= 2048) and (4 * blocks > 5 * cus or k <= 5120)
    row_tiles = -(-rows // 128)
    if blocks <= 2 * cus and row_tiles * -(-blocks // 4) <= cus and not (240 < rows <= 256 and blocks > cus):  # the channel runs in one round
        if rows > 256:
            return False
        return k <= 1024 or (blocks > cus and k <= 2048) or 2 * blocks > 3 * cus
    return blocks > cus


def int8_panels_pay(rows, n, k, cus):
    """The same for int8 weights (figures as above).
    65-128 rows: more than 5 blocks to a CU 0.55-0.94; 3 to 5 0.48-1.0 from 81 rows on, 1.0-1.3 below; 2 to 3 0.43-0.84 above 112 rows up to K = 8192, else 0.85-1.4; up to
    two 0.78-0.96 above 112 rows (up to one K to 8192, up to two K to 2048), otherwise 0.9-1.5.
    129-512 rows: where the channel runs fill one round 0.92-2.5 (K = 1024 of more than one block 0.39-0.5); elsewhere half to one block 0.46-0.99 up to K = 4096, 0.88-1.65
    beyond; to 1.5 blocks 0.4-0.96 up to K = 5120, 0.92-1.5 beyond; to two 0.39-1.01 up to K = 8192, 0.53-1.2 beyond; more 0.43-1.02 (17408 x 5120 at 130 / 512 rows 0.67 /
    0.82), but up to 256 rows of 2 to 3 blocks and K above 8192 0.83-1.1 and more than 5 blocks at 448-512 rows 0.7-1.2.
    513-768 rows: up to 1.5 blocks 0.44-0.87 up to K = 2048, 0.77-1.8 beyond; 1.75 to 3 0.62-1.0; more 0.73-1.25.  Above: half a block 0.53-0.73 up to K = 2048, others 0.71-2.1."""
    if not 64 < rows <= PANEL_ROWS:
        return False
    blocks = -(-n // 16)
    if rows <= 128:
        if blocks <= 3 * cus:
            return rows > 112 and k <= (2048 if cus < blocks <= 2 * cus else 8192)
        return blocks > 5 * cus or rows > 80
    if rows > 512:
        if 2 * blocks <= 3 * cus:
            return k <= 2048 and (rows <= 768 or 2 * blocks <= cus)
        return rows <= 768 and blocks <= 3 * cus
    row_tiles = -(-rows // 128)
    tile_rows = -(-rows // row_tiles)
    most = 5 if tile_rows <= 80 else 3 if tile_rows <= 112 else 2  # blocks of the widest run
    if row_tiles * -(-blocks // most) <= cus or 2 * blocks <= cus:
        return k <= 1024 and blocks > cus
    if blocks > 5 * cus:
        return rows <= 384
    if blocks > 2 * cus:
        return k <= 8192 or rows > 256 or blocks >= 3 * cus
    return k <= (4096 if blocks <= cus else 5120 if 2 * blocks <= 3 * cus else 8192)


def tiles_pay(codec, rows, n, k, cus):
    """Whether row-major rows over 128 x 128 tiles are faster than panels where these were the faster ones before the tiles (time of the pair over panels / row-major, 256 CUs,
    by blocks of 16 channels to a CU; 2600 shapes with weights in cache, both layouts of codes; median behind the range).
    Codes, 513-1024 rows: half to 1.5 blocks 0.94-1.60, 1.22, where the tiles are there (split_pays); to two blocks 0.90-1.33, 1.14 above 768 rows, 0.77-1.29, 1.02 below; wider 0.77-1.23, 0.97;
    up to half a block 0.96-1.11, 1.03 above 896 rows from K = 2048 on, 0.70-1.04, 0.86 otherwise.  Up to 512 rows panels (where they were) 0.56-0.98.
    int8, 129-256 rows: two to three blocks 1.01-1.12, 1.06 above 208 rows, up to 208 0.85-1.14, 0.99.  257-512 rows: up to two blocks 0.97-1.41, 1.15, wider 0.89-1.18, 1.05 up to K = 1024,
    0.84-1.26, 1.02 above.  513 rows and more: above half a block 1.07-1.67, 1.31; a third to half 0.97-1.26, 1.10 above 640 rows, 0.90-1.08, 0.98 below; up to a third 0.98-1.17, 1.06 above
    704, 0.88-1.05, 0.95 below."""
    if rows <= 128 or -(-rows // 128) * -(-n // 128) > 2 * cus:
        return False
    blocks = -(-n // 16)
    if codec == "q4":
        if rows <= 512:
            return False
        if 2 * blocks <= cus:
            return rows > 896 and k >= 2048
        return 2 * blocks <= 3 * cus or (rows > 768 and blocks <= 2 * cus)
    if rows <= 256:
        return rows > 208 and 2 * cus < blocks <= 3 * cus
    if rows <= 512:
        return blocks <= 2 * cus or k <= 1024
    return 2 * blocks > cus or rows > (640 if 3 * blocks > cus else 704)


def split_pays(rows, n, cus):
    """The same for codes without the 128 x 128 int8 tiles: these are decoded for them once, into a Workspace that is never larger than the launch's without them, and
    the older split tiles hold 64 MiB (513 to 896 rows of 5121 to 6144 channels and K from 11008 on).  Time over panels / split tiles: rows that fill 15/16 of their row tiles of up to
    22 channels to a CU 0.98-1.10, rows that fill less 0.90-1.06 there, wider 0.87-1.02."""
    return 16 * rows >= 15 * 128 * -(-rows // 128) and n <= 22 * cus


FEW_ROWS = 8  # rows that a projection of two-stage codes quantises itself


class QuantizedLinear:
    """A8 quantiser + one projection (E8P-Q4 or W8A8) with a dynamic row count up to `capacity`."""

    def __init__(self, codec, weight, scales, capacity, *, packed_k=0, algorithm="auto", block_m=0, book=None):
        if codec not in ("q4", "w8"):
            raise ValueError("codec must be q4 or w8")
        self.codec, self.capacity = codec, capacity
        scales = np.asarray(scales)
        self.n = scales.shape[0]
        weight = np.asarray(weight)
        if codec == "q4":
            self.k = weight.shape[1] * 8
            stored = codebook.q4_to_k_major(weight, 128) if packed_k == 128 else weight
        else:
            self.k = weight.shape[1]
            stored = weight
        self.weight = _dev(stored)
        self.scales = _dev(scales)
        self.book = _dev(codebook.book() if book is None else book)
        # rows over panels: the quantiser leaves the int8 rows a second time, in the order of the matrix operands
        top = min(capacity, PANEL_ROWS)
        self.over_panels = [False] * (top + 1)
        cus = self.cus = torch.cuda.get_device_properties(self.weight.device).multi_processor_count
        if algorithm == "auto" and not block_m and self.k % 128 == 0 and 256 <= self.k <= 32768 and self.n * self.k < 2**31:
            pays = panels_pay if codec == "q4" else int8_panels_pay
            self.over_panels = [pays(rows, self.n, self.k, cus) for rows in range(top + 1)]
        self.over_tiles = {}  # of row counts that have come: whether row-major is faster after all
        # (both copies in one allocation: a second one, new from the driver, took 2 ms of a construction)
        padded = (top + 15) // 16 * 16 if any(self.over_panels) else 0
        codes = torch.empty((capacity + padded, self.k), dtype=torch.int8, device="cuda")
        self.a_q, self.panels = codes[:capacity], codes[capacity:]
        self.a_s = torch.empty((capacity, 1), dtype=torch.float16, device="cuda")
        self.out = torch.empty((capacity, self.n), dtype=torch.float16, device="cuda")
        self.quantizer = Kernel("activation_quantization", K=self.k)
        if padded:
            self.sums = torch.empty(top, dtype=torch.int32, device="cuda")
            self.panel_quantizer = Kernel("activation_quantization", K=self.k, panels=True)
            variant = dict(M=top, N=self.n, K=self.k, dynamic_rows=True, panels=True)
            self.panel_projection = Kernel("e8p_q4_projection", packed_k=packed_k, **variant) if codec == "q4" else Kernel("int8_projection", **variant)
        # workspace=True: the projection takes a `Workspace` buffer (allocated below, once, at the size
        # orx_workspace_bytes reports) for split tiles and decode-once launches
        variant = dict(M=capacity, N=self.n, K=self.k, dynamic_rows=True, algorithm=algorithm, workspace=True)
        if block_m:
            variant["block_m"] = block_m
        if codec == "q4":
            if packed_k:
                variant["packed_k"] = packed_k
            self.projection = Kernel("e8p_q4_projection", **variant)
        else:
            self.projection = Kernel("int8_projection", **variant)
        # one row of two-stage codes, where the GEMV serves the shape: it quantises the fp16 row itself, one launch instead of two
        # (9728 x 2560: 8.7 -> 6.4 us)
        # (K-major codes of K = 512 i + 256 and at most 16 channels to a CU are as fast in two from K = 3072 on: 1392 x 3328 / 4352 / 5888 / 7424 7.8 / 8.9 / 11.0 / 12.4 us
        # in one, 7.3 / 7.8 / 8.4 / 9.2 in two)
        self.single = None
        two_are_faster = algorithm == "auto" and packed_k and self.k % 512 == 256 and self.k >= 3072 and self.n <= 16 * cus
        if codec == "q4" and algorithm in ("auto", "gemv") and not block_m and not two_are_faster:
            try:
                self.single = Kernel("e8p_q4_projection", M=1, N=self.n, K=self.k, algorithm=algorithm, packed_k=packed_k,
                                     input_dtype="float16", codes=True)
            except OrxError as error:
                if error.code != ORX_ERR_BAD_VARIANT:
                    raise
        # two to eight rows, where the loader-wave kernel serves the shape: it quantises the fp16 rows itself.  Time against quantiser and projection, 600 shapes of 1000 to 34816
        # channels, weights out of cache: 2 and 4 rows 0.65 (K = 512) to 0.93, 5 and 8 rows 0.68 to 0.98 (17408 x 5120 at 8 rows 17.1 -> 16.3 us, at 4 16.6 -> 14.5;
        # 9728 x 2560 9.4 -> 7.7)
        self.few = None
        if codec == "q4" and algorithm == "auto" and not block_m and capacity > 1:
            try:
                self.few = Kernel("e8p_q4_projection", M=min(capacity, FEW_ROWS), N=self.n, K=self.k, packed_k=packed_k, dynamic_rows=True, quantize=True)
            except OrxError as error:
                if error.code != ORX_ERR_BAD_VARIANT:
                    raise
        self.workspace = self.projection.workspace()

    def quantize(self, x16, stream=None):
        rows = x16.shape[0]
        self.quantizer(stream=stream, Mask=None, Q=self.a_q, S=self.a_s, X=x16, rows=rows)
        return rows

    def project(self, rows, stream=None):
        if self.codec == "q4":
            self.projection(stream=stream, A=self.a_q, AS=self.a_s, Book=self.book, Out=self.out, S=self.scales,
                            W=self.weight, Workspace=self.workspace, m=rows)
        else:
            self.projection(stream=stream, A=self.a_q, Output=self.out, TokenScale=self.a_s, Weight=self.weight,
                            WeightScale=self.scales, Workspace=self.workspace, m=rows)
        return self._rows(rows)

    def _rows(self, rows):
        """A tensor of the caller's own over the first rows of `out`: what it does to its shape stays with it.  (One view, 1.0 us of
        host time beside the launch, slicing 1.4; a kept slice and detach() take 0.5, but 12 more on a first call.)"""
        return self.out.as_strided((rows, self.n), (self.n, 1))

    def _row_major(self, rows):
        """Whether row-major rows are faster than panels, asked when such rows first come (0.2 us, of codes 1.5; for every row count at construction it was 3 ms)."""
        known = self.over_tiles.get(rows)
        if known is None:
            known = tiles_pay(self.codec, rows, self.n, self.k, self.cus)
            if known and self.codec == "q4" and self.projection.workspace_bytes(rows) < self.n * self.k:
                known = split_pays(rows, self.n, self.cus)
            self.over_tiles[rows] = known
        return known

    def run(self, x16, stream=None):
        if stream is None:
            stream = current_stream()
        if self.single is not None and x16.shape[0] == 1 and x16.data_ptr() % 16 == 0:  # (the quantiser takes any fp16 address)
            self.single(stream=stream, A=x16, AS=self.a_s, Book=self.book, Out=self.out, Q=self.a_q, S=self.scales, W=self.weight)
            return self._rows(1)
        rows = x16.shape[0]
        if 1 < rows <= FEW_ROWS and self.few is not None and x16.data_ptr() % 16 == 0:
            self.few(stream=stream, A=x16, AS=self.a_s, Book=self.book, Out=self.out, Q=self.a_q, S=self.scales, W=self.weight, m=rows)
            return self._rows(rows)
        if rows < len(self.over_panels) and self.over_panels[rows] and not self._row_major(rows):
            self.panel_quantizer(stream=stream, Mask=None, Panels=self.panels, Q=self.a_q, S=self.a_s, Sums=self.sums, X=x16, rows=rows)
            if self.codec == "q4":
                self.panel_projection(stream=stream, A=self.panels, AS=self.a_s, Book=self.book, Out=self.out, S=self.scales, Sums=self.sums,
                                      W=self.weight, m=rows)
            else:
                self.panel_projection(stream=stream, A=self.panels, Output=self.out, TokenScale=self.a_s, Weight=self.weight,
                                      WeightScale=self.scales, m=rows)
            return self._rows(rows)
        return self.project(self.quantize(x16, stream), stream)


BULK_ROWS = 128  # tile height of the routed projections of many rows
# Routed rows per expert from which they beat the seven-launch order over tiles of 32 rows whatever the shape (us, seven launches against six):
# 64 experts x top-6, H 3072, I 256: 73 / 76 at 24 rows, 87 / 85 at 48, 136 / 99 at 96; 16 x top-2, H 4096, I 1536: 85 / 88 at 32,
# 121 / 93 at 64, 325 / 171 at 256.
BULK_ROWS_PER_EXPERT = 48


def small_tile_work(routed, experts, hidden, intermediate):
    """Units of 32 rows (half a tile per expert more than the rows fill) x 512 channels that the projections of a layer come to, those of the second by the length of its rows."""
    return (routed / 32 + experts / 2) * (-(-2 * intermediate // 512) + -(-hidden // 512) * intermediate / hidden)


def routes_pay(routed, experts, hidden, intermediate, cus):
    """Whether the four launches over 32-row tiles whose first projection works out its tiles by itself are faster than the order over 128-row tiles where that was the faster one (time of the
    layer, the latter over the former; 75 layers of up to 4096 routes, popularity like 1 / rank^1.1, 256 CUs, by the small tiles' work to a CU).  Up to 1.5 units 0.96-1.36, median 1.08 (two of 58
    below 0.98); above 0.87-1.19, median 0.96."""
    return 2 * small_tile_work(routed, experts, hidden, intermediate) <= 3 * cus


def bulk_pays(routed, experts, hidden, intermediate, cus):
    """Whether the order over 128-row tiles is faster than the one over tiles of 32 rows, five launches of either kind (time of the layer, the latter over the former; 600 shapes
    with 6 to 48 routed rows per expert, popularity like 1 / rank^1.1, 256 CUs).  What counts is the small tiles' work: units of 32 rows (half a tile per expert more than the rows
    fill) x 512 channels to a CU, those of the second projection by the length of its rows.  From 24 rows per expert and half a unit on 0.95-1.64 (median 1.2), of up to 64 experts from 16 rows
    (32 experts: 12) and 0.7 on 0.97-1.35, of up to 32 experts with 896 and more channels between, where the small tiles of the second projection hold the fewest rows, from 7 rows and 0.4 on
    0.96-1.33; otherwise 0.64-1.1 (of 128 experts with fewer rows 0.75-1.29 without a line between)."""
    work = small_tile_work(routed, experts, hidden, intermediate)
    rows = routed / experts
    return (rows >= 24 and work >= 0.5 * cus or experts <= 64 and rows >= (12 if experts <= 32 else 16) and work >= 0.7 * cus
            or experts <= 32 and intermediate >= 896 and rows >= 7 and work >= 0.4 * cus)


def one_launch_routes(tokens, top_k, experts):
    """Whether router and metadata of few tokens are faster in one launch, whose workgroup has sixteen waves: a token to a wave at a time, top_k ranks one after another
    (time of the layer, one launch over two: up to 18 ranks a wave 0.79-0.99, 24 and 32 1.01-1.11)."""
    return tokens <= 64 and tokens * top_k <= 1024 and experts <= 512 and -(-tokens // 16) * top_k <= 18


def few_pays(tokens, top_k, experts, hidden, intermediate, cus):
    """Whether five launches over tiles of 32 rows (few_rows) are faster than the seven, where the resident kernel is not there (time of the layer, seven over five, 3700 shapes, popularity
    like 1 / rank^0.9, 256 CUs, the median behind the range; weights in cache, and in brackets out of it).  Every workgroup of their second projection quantises its tile's rows again,
    which few or short rows pay for.  Rows of all tiles together (routed x intermediate) up to 80000 0.85-1.80, 1.30 (0.98-1.72, 1.31); above, up to 640 channels between 0.87-1.55, 1.12
    (0.92-1.35, 1.11); up to 1152 where gate | up has at most seven workgroups of 64 channels to a CU 0.85-1.26, 1.02 (0.90-1.27, 1.05), beyond 0.77-1.31, 0.94 (0.82-1.25, 1.01); longer ones
    0.66-1.11, 0.89 (0.72-1.16, 0.97)."""
    routed = tokens * top_k
    if intermediate <= 640 or routed * intermediate <= 80000:
        return True
    tiles = max(experts * (1 - math.exp(-routed / experts)), routed / 32)  # of uniform popularity
    return intermediate <= 1152 and tiles * -(-intermediate // 32) <= 7 * cus


class MoeLayer:
    """Q2A8 expert layer: token-sort, grouped gate_up, SwiGLU->A8, grouped down, weighted combine."""

    def __init__(self, tokens, experts, top_k, hidden, intermediate, gate_up, gate_up_scales, down, down_scales,
                 block_m=32, packed_k=128, fused_metadata=None, fused_dispatch=True, signs=None, fused_stages=None,
                 keep_intermediates=False, grouped_algorithm="auto"):
        self.tokens, self.experts, self.top_k = tokens, experts, top_k
        self.hidden, self.inter, self.block_m = hidden, intermediate, block_m
        assignments = tokens * top_k
        self.assignments = assignments
        # capacity bound of the tile list (kernels/cuda/model/moe.py:263-264)
        self.tile_capacity = (assignments + block_m - 1) // block_m + min(experts, assignments)
        gate_up, down = np.asarray(gate_up), np.asarray(down)
        if packed_k == 128:
            gate_up, down = codebook.q2_to_k_major(gate_up), codebook.q2_to_k_major(down)
        self.w1, self.w2 = _dev(gate_up), _dev(down)
        self.s1, self.s2 = _dev(gate_up_scales), _dev(down_scales)
        self.book = _dev(codebook.book())
        i32 = dict(dtype=torch.int32, device="cuda")
        f16 = dict(dtype=torch.float16, device="cuda")
        i8 = dict(dtype=torch.int8, device="cuda")
        self.ids = torch.empty((tokens, top_k), **i32)
        self.prob = torch.empty((tokens, top_k), dtype=torch.float32, device="cuda")
        self.counts = torch.empty(experts, **i32)
        self.relative = torch.empty((tokens, top_k), **i32)
        self.row_offsets = torch.empty(experts, **i32)
        self.tile_offsets = torch.empty(experts, **i32)
        self.tile_count = torch.empty(1, **i32)
        self.tile_expert = torch.empty(self.tile_capacity, **i32)
        self.tile_row = torch.empty(self.tile_capacity, **i32)
        self.slot_map = torch.empty((tokens, top_k), **i32)
        self.a_q = torch.empty((tokens, hidden), **i8)
        self.a_s = torch.empty((tokens, 1), **f16)
        self.h_q = torch.empty((assignments, intermediate), **i8)
        self.h_s = torch.empty((assignments, 1), **f16)
        self.down_out = torch.empty((assignments, hidden), **f16)
        self.out = torch.empty((tokens, hidden), **f16)
        common = dict(M=tokens, E=experts, top_k=top_k)
        # one launch for all routing metadata where the fused kernel applies (kernels/cuda/model/moe.py:713-764),
        # the three-kernel form otherwise
        one_launch_refused = fused_metadata is False
        fused_metadata_asked = fused_metadata
        if fused_metadata is None:
            fused_metadata = experts <= 1024 and (16 * experts + 32 + 2 * tokens * top_k) * 4 <= 160 * 1024
        self.k_metadata = Kernel("route_metadata", block_m=block_m, **common) if fused_metadata else None
        self.k_router = Kernel("router_topk", renormalize=True, **common)
        self.k_histogram = Kernel("expert_histogram", **common)
        self.k_offsets = Kernel("expert_offsets", E=experts, block_m=block_m)
        self.k_tiles = Kernel("expert_tiles", block_m=block_m, **common)
        # the dispatch quantises the fp16 rows on its way (one launch instead of quantiser + copy) where
        # the row layout allows it
        self.fused_dispatch = fused_dispatch and hidden % 8 == 0
        self.k_a8 = Kernel("activation_quantization", K=hidden)
        self.k_dispatch = Kernel("expert_dispatch", H=hidden, scale_group=hidden, **common,
                                 **({"input_dtype": "float16"} if self.fused_dispatch else {}))
        # signs: the layer's input is rotated first (block-128 signed Hadamard); rotation, A8 and the
        # scatter to the expert-sorted slots are one launch (kernels/cuda/model/rotation_a8.py:558-604)
        self.signs = None if signs is None else _dev(np.asarray(signs, np.int8))
        self.k_rotate_dispatch = None
        if signs is not None:
            self.k_rotate_dispatch = Kernel("rotate_expert_a8", M=tokens, K=hidden, routing="scatter", top_k=top_k,
                                            experts=experts, hand_over="int8")
        grouped = dict(rows=assignments, E=experts, tiles=self.tile_capacity, block_m=block_m, packed_k=packed_k,
                       algorithm=grouped_algorithm)
        self.k_gate_up = Kernel("e8p_decode_grouped", N=2 * intermediate, K=hidden, **grouped)
        self.k_swiglu_a8 = Kernel("activation_quantization", K=intermediate, fused=True)
        self.k_down = Kernel("e8p_decode_grouped", N=hidden, K=intermediate, **grouped)
        # Five launches instead of seven where the resident expert kernel takes the shapes:
        #   router top-k that also quantises every token's row (once per token, not once per route),
        #   metadata that also writes SlotMap, its inverse and zeroed per-slot maxima,
        #   gate_up that gathers the int8 token rows by slot while it stages a tile (no dispatch copy) and
        #     whose epilogue writes fp16(silu(gate) * up) and raises every slot's largest magnitude,
        #   down that quantises those fp16 rows while it stages a tile (no SwiGLU->A8 launch),
        #   combine.
        # The library refuses the variants it does not serve that way, and the seven-launch program stays.
        # Four where gate_up also works out its tiles from the ids (up to 4096 routes): no launch for the metadata, which it leaves for down and combine; the router then
        # clears the maxima.
        self.fused_stages = self.routes_inside = False
        self.keep_intermediates = keep_intermediates
        if fused_stages is not False and fused_metadata and signs is None and hidden % 8 == 0:
            try:
                if fused_metadata_asked is None:
                    try:
                        self.k_gate_up_routes = Kernel("e8p_decode_grouped", N=2 * intermediate, K=hidden, gather=True, epilogue="swiglu", routes=True,
                                                       top_k=top_k, **grouped)
                        self.k_router_clear = Kernel("router_topk", renormalize=True, quantize_hidden=hidden, row_max=True, **common)
                        self.routes_inside = True
                    except OrxError as error:
                        if error.code != ORX_ERR_BAD_VARIANT:
                            raise
                if not self.routes_inside:
                    self.k_router_a8 = Kernel("router_topk", renormalize=True, quantize_hidden=hidden, **common)
                    self.k_metadata_slots = Kernel("route_metadata", block_m=block_m, slot_maps=True, **common)
                    self.k_gate_up_fused = Kernel("e8p_decode_grouped", N=2 * intermediate, K=hidden, gather=True,
                                                  epilogue="swiglu", **grouped)
                self.k_down_fused = Kernel("e8p_decode_grouped", N=hidden, K=intermediate, input_dtype="float16",
                                           tile_units=self.routes_inside, **grouped)
                self.fused_stages = True
            except OrxError as error:
                self.routes_inside = False
                if fused_stages or error.code != ORX_ERR_BAD_VARIANT:
                    raise
        # Many rows: six launches over tiles of 128 rows (`block_m` is the tile height of the orders above).
        #   router top-k + A8 of every token's row, metadata in segments (two launches above 16384 routes, of few experts above 8192 or 12288),
        #   gate_up that gathers the token rows and writes fp16(silu(gate) * up), A8, down, combine.
        # A caller who asked for the quantiser and the dispatch, or the metadata, as launches of their own gets them; `fused_stages` stays
        # true where the five launches are served too.
        self.bulk, bulk_tiles, bulk_kernels = False, 0, {}
        if (fused_stages is None and not keep_intermediates and signs is None and self.fused_dispatch
                and not one_launch_refused and packed_k == 128 and experts <= 1024 and grouped_algorithm == "auto"
                and (not self.fused_stages and assignments >= BULK_ROWS_PER_EXPERT * experts
                     or bulk_pays(assignments, experts, hidden, intermediate, torch.cuda.get_device_properties(self.w1.device).multi_processor_count))):
            try:
                bulk_tiles = (assignments + BULK_ROWS - 1) // BULK_ROWS + min(experts, assignments)
                bulk = dict(rows=assignments, E=experts, tiles=bulk_tiles, block_m=BULK_ROWS, tile_units=True)
                # (all of them before the first is kept: the five launches have kernels of the same names)
                bulk_kernels = dict(
                    k_router_a8=Kernel("router_topk", renormalize=True, quantize_hidden=hidden, **common),
                    k_metadata_slots=Kernel("route_metadata", block_m=BULK_ROWS, slot_maps=True, workspace=True, tile_units=True, **common),
                    k_gate_up_bulk=Kernel("e8p_decode_grouped", N=2 * intermediate, K=hidden, gather=True, epilogue="swiglu", **bulk),
                    k_act_a8=Kernel("activation_quantization", K=intermediate),
                    k_down_bulk=Kernel("e8p_decode_grouped", N=hidden, K=intermediate, **bulk))
                self.bulk = True
            except OrxError as error:
                if error.code != ORX_ERR_BAD_VARIANT:
                    raise
        # Few rows: where neither order applies, five launches over tiles of 32 rows, any hidden and intermediate width, where they are the faster ones.
        #   router top-k + A8 of every token's row, metadata with the tiles as units,
        #   gate_up that gathers the token rows, writes fp16(silu(gate) * up) and raises every slot's largest magnitude,
        #   down that quantises those rows on their way, combine.
        # A caller who asked for launches of their own, for the values in between (`keep_intermediates`) or for an algorithm gets them.
        self.few = False
        if (fused_stages is None and not self.bulk and not self.fused_stages and not keep_intermediates and signs is None and self.fused_dispatch
                and not one_launch_refused and packed_k == 128 and block_m == 32 and experts <= 1024 and grouped_algorithm == "auto"
                and few_pays(tokens, top_k, experts, hidden, intermediate, torch.cuda.get_device_properties(self.w1.device).multi_processor_count)):
            try:
                few = dict(rows=assignments, E=experts, tiles=self.tile_capacity, block_m=block_m, few_rows=True)
                # four where router and metadata are one
                self.k_routes = None
                if one_launch_routes(tokens, top_k, experts):
                    self.k_routes = Kernel("router_topk", renormalize=True, quantize_hidden=hidden, metadata=True, block_m=block_m, **common)
                self.k_router_a8 = Kernel("router_topk", renormalize=True, quantize_hidden=hidden, **common)
                self.k_metadata_slots = Kernel("route_metadata", block_m=block_m, slot_maps=True, workspace=True, tile_units=True, **common)
                self.k_gate_up_few = Kernel("e8p_decode_grouped", N=2 * intermediate, K=hidden, gather=True, epilogue="swiglu", **few)
                self.k_down_few = Kernel("e8p_decode_grouped", N=hidden, K=intermediate, input_dtype="float16", **few)
                self.few = True
            except OrxError as error:
                if error.code != ORX_ERR_BAD_VARIANT:
                    raise
        # The four launches also where nothing but the seven is left (1.06-1.28 times as fast, 11 layers), and over the order for many rows where they are the faster ones.  `bulk` says that that
        # one is served and would run; `routes_first` that these run before either.
        self.routes_first = False
        if (fused_stages is None and not self.few and not keep_intermediates and signs is None and self.fused_dispatch and fused_metadata and fused_metadata_asked is None
                and packed_k == 128 and block_m == 32 and grouped_algorithm == "auto"
                and (routes_pay(assignments, experts, hidden, intermediate, torch.cuda.get_device_properties(self.w1.device).multi_processor_count) if self.bulk
                     else not self.fused_stages)):
            if not self.routes_inside:
                try:
                    resident = dict(grouped, algorithm="resident")
                    served = dict(
                        k_gate_up_routes=Kernel("e8p_decode_grouped", N=2 * intermediate, K=hidden, gather=True, epilogue="swiglu", routes=True, top_k=top_k, **resident),
                        k_router_clear=Kernel("router_topk", renormalize=True, quantize_hidden=hidden, row_max=True, **common),
                        k_down_fused=Kernel("e8p_decode_grouped", N=hidden, K=intermediate, input_dtype="float16", tile_units=True, **resident))
                    vars(self).update(served)
                    self.routes_inside = True
                except OrxError as error:
                    if error.code != ORX_ERR_BAD_VARIANT:
                        raise
            self.routes_first = self.routes_inside
        # What the order that `run` takes needs between its launches, behind all decisions: orders that are served and not taken leave no buffer and no length of a list.
        takes_bulk = self.bulk and not self.routes_first
        if takes_bulk:
            vars(self).update(bulk_kernels)
        if takes_bulk or self.few or self.fused_stages or self.routes_first:
            tiles = bulk_tiles if takes_bulk else self.tile_capacity
            if tiles > self.tile_capacity:
                self.tile_expert, self.tile_row = torch.empty(tiles, **i32), torch.empty(tiles, **i32)
            if takes_bulk or self.few or self.routes_inside:
                self.tile_units = torch.empty((tiles, 4), **i32)
            if not takes_bulk:
                self.row_max = torch.empty(assignments, **i32)
            self.slot_token = torch.empty(assignments, **i32)
            self.act = torch.empty((assignments, intermediate), **f16)
        if takes_bulk or self.few:
            self.segments = self.k_metadata_slots.workspace()
        # the dispatched rows and the gate | up outputs, which the orders for long prompts and for few rows do without
        self.d = self.ds = self.gate_up_out = None
        if not self.bulk and not self.few and not self.routes_first:
            self.d = torch.empty((assignments, hidden), **i8)
            self.ds = torch.empty((assignments, 1), **f16)
            self.gate_up_out = torch.empty((assignments, 2 * intermediate), **f16)
        self.k_combine = Kernel("moe_combine", H=hidden, slots=assignments, **common)

    def run(self, x16, logits, stream=None):
        s = current_stream() if stream is None else stream
        if self.routes_first:
            return self._run_routes_inside(x16, logits, s)
        if self.bulk:
            return self._run_bulk(x16, logits, s)
        if self.fused_stages:
            return self._run_fused(x16, logits, s)
        if self.few:
            return self._run_few(x16, logits, s)
        self.k_router(stream=s, IDs=self.ids, Logits=logits, Prob=self.prob)
        if self.k_metadata is not None:
            self.k_metadata(stream=s, Counts=self.counts, IDs=self.ids, RelativeSlot=self.relative,
                            RowOffsets=self.row_offsets, TileCount=self.tile_count, TileExpert=self.tile_expert,
                            TileOffsets=self.tile_offsets, TileRow=self.tile_row)
        else:
            self.k_histogram(stream=s, Counts=self.counts, IDs=self.ids, RelativeSlot=self.relative)
            self.k_offsets(stream=s, Counts=self.counts, RowOffsets=self.row_offsets, TileCount=self.tile_count,
                           TileOffsets=self.tile_offsets)
            self.k_tiles(stream=s, Counts=self.counts, TileExpert=self.tile_expert, TileOffsets=self.tile_offsets,
                         TileRow=self.tile_row)
        if self.k_rotate_dispatch is not None:
            self.k_rotate_dispatch(stream=s, D=self.d, DS=self.ds, IDs=self.ids, Q=None, RelativeSlot=self.relative,
                                   RowOffsets=self.row_offsets, S=self.a_s, Signs=self.signs, SlotMap=self.slot_map,
                                   Sum=None, X=x16)
        elif self.fused_dispatch:
            self.k_dispatch(stream=s, A=x16, D=self.d, DS=self.ds, IDs=self.ids, RelativeSlot=self.relative,
                            RowOffsets=self.row_offsets, Scale=None, SlotMap=self.slot_map)
        else:
            self.k_a8(stream=s, Mask=None, Q=self.a_q, S=self.a_s, X=x16, rows=self.tokens)
            self.k_dispatch(stream=s, A=self.a_q, D=self.d, DS=self.ds, IDs=self.ids, RelativeSlot=self.relative,
                            RowOffsets=self.row_offsets, Scale=self.a_s, SlotMap=self.slot_map)
        routed = dict(Book=self.book, Counts=self.counts, Offsets=self.row_offsets, TileCount=self.tile_count,
                      TileExpert=self.tile_expert, TileRow=self.tile_row)
        self.k_gate_up(stream=s, A=self.d, AS=self.ds, C=self.gate_up_out, P=self.w1, WS=self.s1, **routed)
        self.k_swiglu_a8(stream=s, Mask=None, Q=self.h_q, S=self.h_s, X=self.gate_up_out, rows=self.assignments)
        self.k_down(stream=s, A=self.h_q, AS=self.h_s, C=self.down_out, P=self.w2, WS=self.s2, **routed)
        self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                       SlotMap=self.slot_map)
        return self.out

    def _run_bulk(self, x16, logits, s):
        self.k_router_a8(stream=s, IDs=self.ids, Logits=logits, Prob=self.prob, Q=self.a_q, S=self.a_s, X=x16)
        self.k_metadata_slots(stream=s, Counts=self.counts, IDs=self.ids, RelativeSlot=self.relative, RowMax=None,
                              RowOffsets=self.row_offsets, SlotMap=self.slot_map, SlotToken=self.slot_token,
                              TileCount=self.tile_count, TileExpert=self.tile_expert, TileOffsets=self.tile_offsets,
                              TileRow=self.tile_row, TileUnits=self.tile_units, Workspace=self.segments)
        routed = dict(Book=self.book, Counts=self.counts, Offsets=self.row_offsets, TileCount=self.tile_count,
                      TileExpert=self.tile_expert, TileRow=self.tile_row, TileUnits=self.tile_units)
        self.k_gate_up_bulk(stream=s, A=self.a_q, AS=self.a_s, Act=self.act, C=None, P=self.w1, RowMax=None,
                            SlotToken=self.slot_token, WS=self.s1, **routed)
        self.k_act_a8(stream=s, Mask=None, Q=self.h_q, S=self.h_s, X=self.act, rows=self.assignments)
        self.k_down_bulk(stream=s, A=self.h_q, AS=self.h_s, C=self.down_out, P=self.w2, WS=self.s2, **routed)
        self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                       SlotMap=self.slot_map)
        return self.out

    def _run_few(self, x16, logits, s):
        metadata = dict(Counts=self.counts, IDs=self.ids, RelativeSlot=self.relative, RowMax=self.row_max, RowOffsets=self.row_offsets,
                        SlotMap=self.slot_map, SlotToken=self.slot_token, TileCount=self.tile_count, TileExpert=self.tile_expert,
                        TileOffsets=self.tile_offsets, TileRow=self.tile_row, TileUnits=self.tile_units)
        if self.k_routes is not None:
            self.k_routes(stream=s, Logits=logits, Prob=self.prob, Q=self.a_q, S=self.a_s, X=x16, **metadata)
        else:
            self.k_router_a8(stream=s, IDs=self.ids, Logits=logits, Prob=self.prob, Q=self.a_q, S=self.a_s, X=x16)
            self.k_metadata_slots(stream=s, Workspace=self.segments, **metadata)
        routed = dict(Book=self.book, RowMax=self.row_max, TileCount=self.tile_count, TileUnits=self.tile_units)
        self.k_gate_up_few(stream=s, A=self.a_q, AS=self.a_s, Act=self.act, P=self.w1, SlotToken=self.slot_token, WS=self.s1, **routed)
        self.k_down_few(stream=s, A=self.act, C=self.down_out, P=self.w2, WS=self.s2, **routed)
        self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                       SlotMap=self.slot_map)
        return self.out

    def _run_fused(self, x16, logits, s):
        keep = self.keep_intermediates
        if self.routes_inside:
            return self._run_routes_inside(x16, logits, s)
        self.k_router_a8(stream=s, IDs=self.ids, Logits=logits, Prob=self.prob, Q=self.a_q, S=self.a_s, X=x16)
        self.k_metadata_slots(stream=s, Counts=self.counts, IDs=self.ids, RelativeSlot=self.relative, RowMax=self.row_max,
                              RowOffsets=self.row_offsets, SlotMap=self.slot_map, SlotToken=self.slot_token,
                              TileCount=self.tile_count, TileExpert=self.tile_expert, TileOffsets=self.tile_offsets,
                              TileRow=self.tile_row)
        routed = dict(Book=self.book, Counts=self.counts, Offsets=self.row_offsets, TileCount=self.tile_count,
                      TileExpert=self.tile_expert, TileRow=self.tile_row)
        self.k_gate_up_fused(stream=s, A=self.a_q, AS=self.a_s, Act=self.act, C=self.gate_up_out if keep else None,
                             P=self.w1, RowMax=self.row_max, SlotToken=self.slot_token, WS=self.s1, **routed)
        self.k_down_fused(stream=s, A=self.act, AS=self.h_s if keep else None, C=self.down_out, P=self.w2,
                          Q=self.h_q if keep else None, RowMax=self.row_max, WS=self.s2, **routed)
        self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                       SlotMap=self.slot_map)
        return self.out

    def _run_routes_inside(self, x16, logits, s):
        keep = self.keep_intermediates
        self.k_router_clear(stream=s, IDs=self.ids, Logits=logits, Prob=self.prob, Q=self.a_q, RowMax=self.row_max, S=self.a_s, X=x16)
        routed = dict(Book=self.book, Counts=self.counts, Offsets=self.row_offsets, RowMax=self.row_max, TileCount=self.tile_count,
                      TileExpert=self.tile_expert, TileRow=self.tile_row, TileUnits=self.tile_units)
        self.k_gate_up_routes(stream=s, A=self.a_q, AS=self.a_s, Act=self.act, C=self.gate_up_out if keep else None, IDs=self.ids, P=self.w1,
                              RelativeSlot=self.relative, SlotMap=self.slot_map, SlotToken=self.slot_token, TileOffsets=self.tile_offsets, WS=self.s1, **routed)
        self.k_down_fused(stream=s, A=self.act, AS=self.h_s if keep else None, C=self.down_out, P=self.w2, Q=self.h_q if keep else None, WS=self.s2, **routed)
        self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                       SlotMap=self.slot_map)
        return self.out


def combine_pays(routes, hidden, intermediate, cus):
    """Whether the second projection of one token with the SwiGLU in front and the sum over its routes behind is faster than projection and sum in two launches (time of the layer, one over
    two; 256 CUs; without the SwiGLU it also is where `MoeTokenLayer` says).  Every workgroup of 8 channels makes the codes of all routes itself, in turns of 512 values, and one route's are a wave's.
    Up to 512 values 0.78-0.97, with three workgroups to a CU 1.06-1.09 up to two routes and 0.79-0.96 above.  Up to 1024: one workgroup to a CU 0.92-0.98 up to four routes
    and 0.92-0.96 above (up to half of the CUs 1.0-1.03); two and three to a CU 0.98-1.22 up to four routes, 0.89-0.99 above.  Beyond mostly 1.0-1.33 (0.97 at best, 8 routes of
    4096 x 1536)."""
    per_cu = -(-hidden // (8 * cus))
    if intermediate <= 512:
        return per_cu <= 2 or routes > 2
    if intermediate <= 1024:
        return (routes <= 4 or hidden > 4 * cus) if per_cu == 1 else routes > 4
    return False


class MoeTokenLayer:
    """The same expert layer for ONE token: its routes index the expert banks directly
    (kernels/cuda/model/integer_vq.py:380-444), so there is no sorting, no tile list and no dispatch copy:
    router top-k, gate/up of every route from the shared row (quantised on the way), SwiGLU->A8 per route,
    down per route, weighted combine."""

    def __init__(self, experts, top_k, hidden, intermediate, gate_up, gate_up_scales, down, down_scales, fused=None):
        self.experts, self.top_k, self.hidden, self.inter = experts, top_k, hidden, intermediate
        self.w1 = _dev(codebook.q2_to_k_major(np.asarray(gate_up)))
        self.w2 = _dev(codebook.q2_to_k_major(np.asarray(down)))
        self.s1, self.s2 = _dev(gate_up_scales), _dev(down_scales)
        self.book = _dev(codebook.raw_book())
        f16 = dict(dtype=torch.float16, device="cuda")
        i8 = dict(dtype=torch.int8, device="cuda")
        self.ids = torch.empty((1, top_k), dtype=torch.int32, device="cuda")
        self.prob = torch.empty((1, top_k), dtype=torch.float32, device="cuda")
        self.a_s = torch.empty((1, 1), **f16)
        self.gate_up_out = torch.empty((top_k, 2 * intermediate), **f16)
        self.h_q = torch.empty((top_k, intermediate), **i8)
        self.h_s = torch.empty((top_k, 1), **f16)
        self.down_out = torch.empty((top_k, hidden), **f16)
        self.slot_map = torch.arange(top_k, dtype=torch.int32, device="cuda").view(1, top_k)  # route r is slot r
        self.out = torch.empty((1, hidden), **f16)
        common = dict(M=1, E=experts, top_k=top_k)
        self.k_router = Kernel("router_topk", renormalize=True, **common)
        # gate/up quantises the shared fp16 row itself (no launch for the A8 of one row)
        self.k_gate_up = Kernel("integer_e8p_gemv", E=experts, routes=top_k, N=2 * intermediate, K=hidden,
                                shared_input=True, input_dtype="float16")
        self.k_swiglu_a8 = Kernel("activation_quantization", K=intermediate, fused=True)
        self.k_down = Kernel("integer_e8p_gemv", E=experts, routes=top_k, N=hidden, K=intermediate, shared_input=False)
        self.k_combine = Kernel("moe_combine", H=hidden, slots=top_k, **common)
        # Fewer than five launches where the library has the forms (up to 512 experts): gate/up selects the token's
        # routes itself while it builds its tables (no router launch), down turns the fp16 gate|up rows into
        # SwiGLU -> A8 codes on their way into LDS (no launch in between).  These are three; two below.
        self.fused = False
        if fused is not False:
            try:
                routes = dict(E=experts, routes=top_k)
                self.k_gate_up_routing = Kernel("integer_e8p_gemv", N=2 * intermediate, K=hidden, shared_input=True,
                                                input_dtype="float16", route_logits=True, renormalize=True, **routes)
                self.k_down_swiglu = Kernel("integer_e8p_gemv", N=hidden, K=intermediate, shared_input=False,
                                            input_dtype="float16", fused_swiglu=True, **routes)
                self.fused = True
            except OrxError as error:
                if fused or error.code != ORX_ERR_BAD_VARIANT:
                    raise
        # Two launches where the sum over the routes joins the second projection: 13.8 -> 11.6 us for 8 of 128 experts, 2048 x 512, and 10.9 since the first one leaves
        # fp16(silu(gate) * up), which every workgroup of the second made again, beside gate | up.  Three launches over two (140 shapes of up to 2048 channels between): up to two workgroups to a CU
        # 0.99-1.37, median 1.13.  `k_down_combine` names it where it also paid with the SwiGLU in front.
        self.k_down_combine = self.k_down_act = None
        cus = torch.cuda.get_device_properties(self.w2.device).multi_processor_count
        pays = combine_pays(top_k, hidden, intermediate, cus)
        if self.fused and (pays or hidden <= 16 * cus):
            try:
                served = dict(
                    k_gate_up_act=Kernel("integer_e8p_gemv", N=2 * intermediate, K=hidden, shared_input=True, input_dtype="float16", route_logits=True,
                                         renormalize=True, epilogue="swiglu", **routes),
                    k_down_act=Kernel("integer_e8p_gemv", N=hidden, K=intermediate, shared_input=False, input_dtype="float16", combine=True, **routes))
                vars(self).update(served)
                self.act = torch.empty((top_k, intermediate), **f16)
                self.k_down_combine = self.k_down_act if pays else None
            except OrxError as error:
                if error.code != ORX_ERR_BAD_VARIANT:
                    raise

    def run(self, x16, logits, stream=None):
        s = current_stream() if stream is None else stream
        if self.k_down_act is not None:
            self.k_gate_up_act(stream=s, A=x16, AS=self.a_s, Act=self.act, Book=self.book, C=self.gate_up_out, IDs=self.ids,
                               Logits=logits, P=self.w1, Prob=self.prob, WS=self.s1)
            self.k_down_act(stream=s, A=self.act, AS=self.h_s, Book=self.book, C=self.down_out, IDs=self.ids,
                                Output=self.out, P=self.w2, Prob=self.prob, WS=self.s2)
            return self.out
        if self.fused:
            self.k_gate_up_routing(stream=s, A=x16, AS=self.a_s, Book=self.book, C=self.gate_up_out, IDs=self.ids,
                                   Logits=logits, P=self.w1, Prob=self.prob, WS=self.s1)
            self.k_down_swiglu(stream=s, A=self.gate_up_out, AS=self.h_s, Book=self.book, C=self.down_out, IDs=self.ids,
                               P=self.w2, WS=self.s2)
            self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                           SlotMap=self.slot_map)
            return self.out
        self.k_router(stream=s, IDs=self.ids, Logits=logits, Prob=self.prob)
        self.k_gate_up(stream=s, A=x16, AS=self.a_s, Book=self.book, C=self.gate_up_out, IDs=self.ids, P=self.w1,
                       WS=self.s1)
        self.k_swiglu_a8(stream=s, Mask=None, Q=self.h_q, S=self.h_s, X=self.gate_up_out, rows=self.top_k)
        self.k_down(stream=s, A=self.h_q, AS=self.h_s, Book=self.book, C=self.down_out, IDs=self.ids, P=self.w2,
                    WS=self.s2)
        self.k_combine(stream=s, Expert=self.down_out, Output=self.out, Prob=self.prob, Shared=None, SharedGate=None,
                       SlotMap=self.slot_map)
        return self.out
