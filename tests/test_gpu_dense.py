"""GPU parity: decode, A8 and the dense Q4A8 / W8A8 projections against the CPU oracle.

Integer results (decoded weights, int8 activations, int32 accumulators) must be bit-exact.
fp16/fp32 outputs are produced by the same two fp32 multiplies as the oracle, so they are
compared for equality as well; the contract tolerance (1e-3 relative / 1e-2 absolute) is
asserted separately so a reader sees the stated bar.
"""
import numpy as np
import pytest
import torch

from oracle import reference as orc
from orinfer_amd import codebook, lib, programs, workloads

from . import gpu_util as gu
from .started_util import MID_2, MID_4, RUNS, reported, started

pytestmark = pytest.mark.gpu
TABLE = orc.basis()
RTOL, ATOL = 1e-3, 1e-2  # fp16 output tolerance stated by the benchmark contract


def assert_close_fp16(got, want):
    got = np.asarray(got, np.float32)
    want = np.asarray(want, np.float32)
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= ATOL + RTOL * np.abs(want)).all()


def exhaustive_q4():
    first = np.arange(65536, dtype=np.uint32).reshape(4096, 16)
    second = (first * np.uint32(32771) + np.uint32(97)) & np.uint32(65535)
    return first | (second << np.uint32(16))


# ---- decode ---------------------------------------------------------------
@pytest.mark.parametrize("packed_k", [0, 64, 128])
def test_q4_unpack_every_code(packed_k):
    packed = exhaustive_q4()  # every coarse code once, residual by an LCG (test_e8p_q4.py:13-30)
    want = orc.q4_integers(packed, TABLE)
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    out = torch.zeros((4096, 128), dtype=torch.int8, device=gu.DEV)
    gu.kernel("e8p_q4_unpack", N=4096, K=128, packed_k=packed_k)(Book=gu.book(), Output=out, W=gu.dev(stored))
    np.testing.assert_array_equal(gu.host(out), want)


def test_q4_unpack_residual_every_code():
    # swap the halves so that every code also appears as the residual stage
    packed = exhaustive_q4()
    swapped = (packed >> np.uint32(16)) | (packed << np.uint32(16))
    out = torch.zeros((4096, 128), dtype=torch.int8, device=gu.DEV)
    gu.kernel("e8p_q4_unpack", N=4096, K=128)(Book=gu.book(), Output=out, W=gu.dev(swapped))
    np.testing.assert_array_equal(gu.host(out), orc.q4_integers(swapped, TABLE))


def test_q2_unpack_every_code():
    codes = np.arange(65536, dtype=np.uint16).reshape(4096, 16)
    out = torch.zeros((4096, 128), dtype=torch.int8, device=gu.DEV)
    gu.kernel("e8p_q2_unpack", N=4096, K=128)(Book=gu.book(), Output=out, W=gu.dev(codes))
    np.testing.assert_array_equal(gu.host(out), orc.q2_integers(codes, TABLE))
    k128 = orc.q2_pack_k128(codes)
    out.zero_()
    gu.kernel("e8p_q2_unpack", N=4096, K=128, packed_k=128)(Book=gu.book(), Output=out, W=gu.dev(k128))
    np.testing.assert_array_equal(gu.host(out), orc.q2_integers(codes, TABLE))


# ---- A8 -------------------------------------------------------------------
def test_a8_edges_and_random():
    rng = np.random.default_rng(orc.SEED)
    x = rng.normal(size=(67, 2560)).astype(np.float16)
    x[0] = 0
    x[1, :8] = [127, -127, 63.5, 0.5, 1.5, 2.5, -0.5, -2.5]
    x[1, 8:] = 0
    x[2] = 0
    x[2, 5] = 1e-7
    x[3, :8] = [254, 1, -1, 3, -3, 5, 127, -254]
    x[3, 8:] = 0
    x[4, 0] = 65504
    x[5] *= 20
    q, s = gu.a8(gu.dev(x))
    wq, ws = orc.a8(x)
    np.testing.assert_array_equal(gu.host(s), ws)
    np.testing.assert_array_equal(gu.host(q), wq)


@pytest.mark.parametrize("k,group", [(2560, 64), (384, 128), (100, 25), (7, 7), (5120, 5120), (16384, 8192), (9001, 9001),
                                     (1024, 512), (4096, 4096)])
def test_a8_groups_and_odd_shapes(k, group):
    rng = np.random.default_rng(orc.SEED + k)
    x = (rng.normal(size=(5, k)) * 3).astype(np.float16)
    q, s = gu.a8(gu.dev(x), group=group)
    wq, ws = orc.a8(x, group)
    np.testing.assert_array_equal(gu.host(s), ws)
    np.testing.assert_array_equal(gu.host(q), wq)


@pytest.mark.parametrize("rows,k,group", [(300, 17408, 17408), (260, 16384, 8192), (259, 5120, 5120), (257, 24576, 24576), (258, 24584, 24584)])
def test_a8_many_rows_of_long_groups(rows, k, group):
    # many rows of groups that four and eight waves hold in registers between the maximum and the codes
    rng = np.random.default_rng(orc.SEED + rows + k)
    x = (rng.normal(size=(rows, k)) * 2).astype(np.float16)
    x[1] = 0
    x[2, -1] = 1000
    q, s = gu.a8(gu.dev(x), group=group)
    wq, ws = orc.a8(x, group)
    np.testing.assert_array_equal(gu.host(s), ws)
    np.testing.assert_array_equal(gu.host(q), wq)


@pytest.mark.parametrize("fused", [False, True], ids=["rows", "swiglu"])
@pytest.mark.parametrize("rows,k,group", [
    (2049, 1016, 1016), (2048, 2048, 2048), (1023, 1536, 768),          # one wave to a group, units that do not divide by four
    (3, 520, 520), (5, 2048, 2048), (600, 2056, 2056), (514, 12288, 12288),   # four waves, at both ends of their pieces
    (2, 2056, 2056), (513, 12296, 12296), (1, 32768, 32768),            # eight waves
    (1, 32776, 32776), (3, 65536 + 4096, 65536 + 4096), (2, 90000, 45000),    # sixteen waves, longer than they hold
    (2, 2060, 2060), (2049, 1020, 1020), (2, 40004, 40004),             # rows that are not 16-byte aligned
])
def test_a8_held_forms(rows, k, group, fused):
    """The waves and pieces that hold a row follow its length and the row count; codes and scales do not."""
    rng = np.random.default_rng(orc.SEED + rows + k + fused)
    x = (rng.normal(size=(rows, 2 * k if fused else k)) * 2).astype(np.float16)
    x[0, -1] = 300
    q, s = gu.a8(gu.dev(x), group=group, fused=fused)
    values = x
    if fused:  # the device's own fp16 values (the exponential may differ from libm in the last place)
        y = torch.empty((rows, k), dtype=torch.float16, device=gu.DEV)
        gu.kernel("swiglu", I=k)(X=gu.dev(x), Y=y, rows=rows)
        values = gu.host(y)
    wq, ws = orc.a8(values, group)
    np.testing.assert_array_equal(gu.host(s), ws)
    np.testing.assert_array_equal(gu.host(q), wq)


@pytest.mark.parametrize("amax", [254.0, 127.0, 65504.0, 1.0, 3e-3, 2.0**-12, 300 * 2.0**-24, 190 * 2.0**-24, 3 * 2.0**-24])
def test_a8_every_value_up_to_the_largest(amax):
    """All fp16 values of a row with this largest one: ties at scales 1 and 2, quotients beyond 127 at subnormal scales."""
    every = np.arange(65536, dtype=np.uint16).view(np.float16)
    every = every[np.isfinite(every)]
    x = np.where(np.abs(every.astype(np.float32)) <= np.float32(np.float16(amax)), every, np.float16(0))[None]
    assert np.abs(x).max() == np.float16(amax)
    q, s = gu.a8(gu.dev(x), group=None)
    wq, ws = orc.a8(x)
    np.testing.assert_array_equal(gu.host(s), ws)
    np.testing.assert_array_equal(gu.host(q), wq)


def test_swiglu_gates_without_a_finite_sigmoid_product():
    """Gates at and beyond the ends of the exponential against the formula in fp32: a gate of minus infinity has no value
    (-inf * 0), the gates down to -104 keep a sigmoid above zero, and what the products make of infinities is theirs."""
    inf, nan = np.inf, np.nan
    gates = np.array([-inf, inf, nan, -65504, -104.0625, -104, -103.9375, -90, -87.5, -87, -20, -0.0, 0, 1, 88, 65504], np.float16)
    ups = np.array([1, -3, 65504, inf, -inf, nan, 0, -0.0], np.float16)
    g, u = (a.reshape(1, -1) for a in np.meshgrid(gates, ups))
    x = np.concatenate([g, u], axis=1)
    y = torch.empty(g.shape, dtype=torch.float16, device=gu.DEV)
    gu.kernel("swiglu", I=g.shape[1])(X=gu.dev(x), Y=y, rows=1)
    with np.errstate(invalid="ignore", over="ignore"):
        want = orc.swiglu_fp16(x)
    got = gu.host(y)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    known = ~np.isnan(want)
    np.testing.assert_array_equal(np.signbit(got[known]), np.signbit(want[known]))
    finite = np.isfinite(want)
    np.testing.assert_allclose(got[finite].astype(np.float32), want[finite].astype(np.float32), rtol=1e-3, atol=6e-8)


@pytest.mark.parametrize("rows,k", [
    (2048, 512), (4, 512),     # one wave to a row
    (4, 2048), (513, 12288),   # four waves
    (4, 12296),                # eight waves
    (4, 32776), (4, 2060),     # sixteen waves; rows that are not 16-byte aligned
])
def test_a8_of_gates_without_a_value(rows, k):
    """A gate that gives no number (minus infinity, NaN) leaves the row's scale and its other codes alone; an infinite value
    is the row's largest: the scale is infinite and every finite value's code is 0."""
    rng = np.random.default_rng(orc.SEED + rows + k)
    x = (rng.normal(size=(rows, 2 * k)) * 2).astype(np.float16)
    at = k // 2 + 3
    for row, gate in ((0, -np.inf), (1, np.nan), (2, np.inf), (3, -np.inf)):
        x[row, at] = gate
    x[3, at + 1] = np.inf  # both in one row: the infinity decides
    x[:, k + at] = 0.5
    x[:, k + at + 1] = 0.25
    y = torch.empty((rows, k), dtype=torch.float16, device=gu.DEV)
    gu.kernel("swiglu", I=k)(X=gu.dev(x), Y=y, rows=rows)
    values = gu.host(y)
    assert np.isnan(values[[0, 1, 3], at]).all() and values[2, at] == np.inf and values[3, at + 1] == np.inf
    for q, s in (gu.a8(gu.dev(x), fused=True), gu.a8(y)):
        q, s = gu.host(q), gu.host(s)
        plain = np.where(np.isfinite(values), values, np.float16(0))
        wq, ws = orc.a8(plain)
        live = np.isfinite(values)
        keep = [r for r in range(rows) if r not in (2, 3)]
        np.testing.assert_array_equal(s[keep], ws[keep])
        np.testing.assert_array_equal(q[keep][live[keep]], wq[keep][live[keep]])
        assert np.isinf(s[2:4]).all() and (q[2:4][live[2:4]] == 0).all()


@pytest.mark.parametrize("rows,k", [(2049, 512), (5, 8), (5, 2048), (5, 12296), (5, 32776)])
def test_a8_largest_beside_a_nan(rows, k):
    """The lane that holds a row's largest magnitude, a negative one, holds a NaN too (either sign, either half of a pair); rows of zeros and of NaN alone."""
    rng = np.random.default_rng(orc.SEED + rows + k)
    x = (rng.normal(size=(rows, k)) * 2).astype(np.float16)
    x[:3, -1] = -77
    x[0, -2], x[1, -3], x[2, -8] = np.nan, np.float16(-np.float32(np.nan)), np.nan
    x[3], x[4] = -0.0, np.nan
    q, s = (gu.host(t) for t in gu.a8(gu.dev(x)))
    live = ~np.isnan(x)
    wq, ws = orc.a8(np.where(live, x, np.float16(0)))
    np.testing.assert_array_equal(s, ws)
    np.testing.assert_array_equal(q[live], wq[live])


def test_swiglu_rounds_as_an_unbiased_exponential_does():
    """Share of fp16 results that differ from the correctly rounded product, where the exponential's argument is large: the
    fp32 roundings alone (sigmoid within 1.6e-7, two products) cost 0.85e-4 of them there, an exponential that is off by the
    error of one fp32 ln 2 times its argument 1.1e-4."""
    rng = np.random.default_rng(orc.SEED + 77)
    rows, k = 1024, 16384
    gate = rng.uniform(-18, -10, (rows, k)).astype(np.float16)
    up = np.exp2(rng.uniform(8, 15.9, (rows, k))).astype(np.float16)
    y = torch.empty((rows, k), dtype=torch.float16, device=gu.DEV)
    gu.kernel("swiglu", I=k)(X=gu.dev(np.concatenate([gate, up], axis=1)), Y=y, rows=rows)
    g = gate.astype(np.float64)
    want = (g / (1.0 + np.exp(-g)) * up).astype(np.float16)
    normal = np.abs(want) > 2.0**-14
    share = ((gu.host(y) != want) & normal).sum() / normal.sum()
    print("share of results rounded the other way:", share)
    assert share < 1.0e-4


def test_a8_masked_columns():
    rng = np.random.default_rng(orc.SEED)
    x = rng.normal(size=(9, 512)).astype(np.float16)
    mask = (rng.uniform(size=512) < 0.1).astype(np.uint8)
    x[:, 3] = 1000  # would dominate amax if the mask were ignored
    mask[3] = 7
    q, s = gu.a8(gu.dev(x), masked=gu.dev(mask))
    xm = x.copy()
    xm[:, mask != 0] = 0
    wq, ws = orc.a8(xm)
    np.testing.assert_array_equal(gu.host(s), ws)
    np.testing.assert_array_equal(gu.host(q), wq)


def test_swiglu_then_a8_and_fused_form_agree():
    rng = np.random.default_rng(orc.SEED)
    gu_in = (rng.normal(size=(33, 2 * 512)) * 2).astype(np.float16)
    x = gu.dev(gu_in)
    y = torch.empty((33, 512), dtype=torch.float16, device=gu.DEV)
    gu.kernel("swiglu", I=512)(X=x, Y=y, rows=33)
    want = orc.swiglu_fp16(gu_in)
    got = gu.host(y)
    # exp() differs by an ulp between libraries: tolerance on the fp16 boundary value
    np.testing.assert_allclose(got.astype(np.float32), want.astype(np.float32), rtol=2e-3, atol=1e-6)
    assert (got == want).mean() > 0.99
    q1, s1 = gu.a8(y)
    wq, ws = orc.a8(got)  # the quantiser itself must be exact on the GPU's own fp16 values
    np.testing.assert_array_equal(gu.host(q1), wq)
    np.testing.assert_array_equal(gu.host(s1), ws)
    q2, s2 = gu.a8(x, fused=True)
    assert torch.equal(q1, q2) and torch.equal(s1, s2)


# ---- signed block-128 rotation fused with A8 -------------------------------------------------
@pytest.mark.parametrize("m,k", [(1, 128), (3, 384), (5, 2560), (2, 5120), (1, 17408), (260, 2304)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_rotate_activation_a8_matches_oracle(m, k, swiglu):
    rng = np.random.default_rng(orc.SEED + m + k)
    x = rng.normal(size=(m, 2 * k if swiglu else k)).astype(np.float16)
    x[0, :3] = [0, 60000, -60000] if not swiglu else [3, -2, 0]
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    want_q, want_s = orc.rotate_a8(x, signs, swiglu=swiglu)
    variant = dict(M=m, K=k)
    if swiglu:
        variant["swiglu"] = True
    q = torch.full((m + 1, k), 77, dtype=torch.int8, device=gu.DEV)
    s = torch.full((m + 1,), 5.0, dtype=torch.float16, device=gu.DEV)
    gu.kernel("rotate_activation_a8", **variant)(Q=q, S=s, Signs=gu.dev(signs), X=gu.dev(x))
    if swiglu:
        # the exponential of the SwiGLU boundary may differ in the last place between libm and the
        # device: compare the codes on the device's own fp16 SwiGLU values
        mid = torch.empty((m, k), dtype=torch.float16, device=gu.DEV)
        gu.kernel("swiglu", I=k)(X=gu.dev(x), Y=mid, rows=m)
        want_q, want_s = orc.rotate_a8(gu.host(mid), signs)
    np.testing.assert_array_equal(gu.host(s)[:m], want_s[:, 0])
    np.testing.assert_array_equal(gu.host(q)[:m], want_q)
    assert (gu.host(q)[m:] == 77).all() and float(gu.host(s)[m]) == 5.0


def test_rotate_activation_a8_dynamic_rows_zero_row_and_graph():
    rng = np.random.default_rng(orc.SEED + 12)
    k = 1024
    x = rng.normal(size=(9, k)).astype(np.float16)
    x[4] = 0
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    kern = gu.kernel("rotate_activation_a8", M=16, K=k, dynamic_rows=True)
    d_x, d_signs = gu.dev(x), gu.dev(signs)
    q = torch.zeros((16, k), dtype=torch.int8, device=gu.DEV)
    s = torch.zeros((16,), dtype=torch.float16, device=gu.DEV)
    for rows in (9, 1):
        q.fill_(9)
        kern(Q=q, S=s, Signs=d_signs, X=d_x, m=rows)
        want_q, want_s = orc.rotate_a8(x[:rows], signs)
        np.testing.assert_array_equal(gu.host(q)[:rows], want_q)
        np.testing.assert_array_equal(gu.host(s)[:rows], want_s[:, 0])
        assert (gu.host(q)[rows:] == 9).all()
    assert float(gu.host(s)[0]) > 0
    kern(Q=q, S=s, Signs=d_signs, X=d_x, m=9)
    assert not gu.host(q)[4].any() and float(gu.host(s)[4]) == 1.0
    # rotated activations against rotated weights reproduce the un-rotated dot products
    w = rng.normal(size=(6, k)).astype(np.float32)
    rotated_w = orc.rotate(w, signs)
    codes, scales = gu.host(q)[:9].astype(np.float32), gu.host(s)[:9].astype(np.float32)
    approx = (codes * scales[:, None]) @ rotated_w.T
    np.testing.assert_allclose(approx, x.astype(np.float32) @ w.T, atol=0.6, rtol=0.05)


def ulps_fp16(a, b):
    """Distance in fp16 units in the last place (both finite)."""
    def key(v):
        bits = np.asarray(v, np.float16).view(np.int16).astype(np.int32)
        return np.where(bits < 0, -(bits & 0x7FFF), bits)
    return np.abs(key(a) - key(b))


@pytest.mark.parametrize("m,k,zero_centered", [(1, 256, True), (3, 1536, True), (5, 5120, True), (2, 5120, False),
                                               (1, 17408, True), (2, 2048, True), (256, 2304, True), (257, 2304, True)])
def test_residual_norm_rotate_a8_matches_oracle(m, k, zero_centered):
    rng = np.random.default_rng(orc.SEED + 3 * m + k)
    x = rng.normal(size=(m, k)).astype(np.float16)
    r = rng.normal(size=(m, k)).astype(np.float32)
    w = (rng.normal(size=k) * 0.1 + (0.0 if zero_centered else 1.0)).astype(np.float16)
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    variant = dict(M=m, K=k)
    if not zero_centered:
        variant["zero_centered"] = False
    # one spare row behind every output, as in the reference's check (check_rows.py:156-161,172)
    y = torch.full((m + 1, k), 91, dtype=torch.float16, device=gu.DEV)
    ro = torch.full((m + 1, k), 91, dtype=torch.float32, device=gu.DEV)
    q = torch.full((m + 1, k), 91, dtype=torch.int8, device=gu.DEV)
    s = torch.full((m + 1,), 91, dtype=torch.float16, device=gu.DEV)
    gu.kernel("residual_norm_rotate_a8", **variant)(Q=q, R=gu.dev(r), RO=ro, S=s, Signs=gu.dev(signs), W=gu.dev(w),
                                                    X=gu.dev(x), Y=y)
    want_y, want_ro, _, _ = orc.residual_norm_rotate_a8(x, r, w, signs, zero_centered=zero_centered)
    np.testing.assert_array_equal(gu.host(ro)[:m], want_ro)  # one fp32 add: exact
    got_y = gu.host(y)[:m]
    # fp16((sum * rsqrt(mean + eps)) * gain): the fp32 sum of squares and the reciprocal square root
    # may differ in the last place from the float64 restatement, which moves an fp16 rounding by
    # at most one unit in the last place
    distance = ulps_fp16(got_y, want_y)
    assert distance.max() <= 1 and (distance > 0).mean() < 0.02
    # the rotation and the quantiser read the fp16 row the kernel wrote: codes and scales are exact
    want_q, want_s = orc.rotate_a8(got_y, signs)
    np.testing.assert_array_equal(gu.host(q)[:m], want_q)
    np.testing.assert_array_equal(gu.host(s)[:m], want_s[:, 0])
    for spare in (y, ro, q, s):
        assert (gu.host(spare)[m:] == 91).all()


def test_residual_norm_rotate_a8_dynamic_rows_zero_rows_and_composition():
    rng = np.random.default_rng(orc.SEED + 77)
    k, cap = 5120, 32
    x = rng.normal(size=(17, k)).astype(np.float16)
    r = rng.normal(size=(17, k)).astype(np.float32)
    x[6], r[6] = 0, 0
    w = (rng.normal(size=k) * 0.1).astype(np.float16)
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    kern = gu.kernel("residual_norm_rotate_a8", M=cap, K=k, dynamic_rows=True)
    rotation = gu.kernel("rotate_activation_a8", M=cap, K=k, dynamic_rows=True)
    d = dict(R=gu.dev(r), Signs=gu.dev(signs), W=gu.dev(w), X=gu.dev(x))
    y = torch.zeros((cap, k), dtype=torch.float16, device=gu.DEV)
    ro = torch.zeros((cap, k), dtype=torch.float32, device=gu.DEV)
    q = torch.zeros((cap, k), dtype=torch.int8, device=gu.DEV)
    s = torch.zeros((cap,), dtype=torch.float16, device=gu.DEV)
    for rows in (17, 1, 8):
        for out in (y, ro, q, s):
            out.fill_(91)
        kern(Q=q, RO=ro, S=s, Y=y, m=rows, **d)
        # the reference's own check: the fused kernel equals the rotation kernel run on Y
        q2 = torch.zeros_like(q)
        s2 = torch.zeros_like(s)
        rotation(Q=q2, S=s2, Signs=d["Signs"], X=y, m=rows)
        assert torch.equal(q[:rows], q2[:rows]) and torch.equal(s[:rows], s2[:rows])
        assert (gu.host(q)[rows:] == 91).all() and (gu.host(y)[rows:] == 91).all()
        np.testing.assert_array_equal(gu.host(ro)[:rows], x[:rows].astype(np.float32) + r[:rows])
    kern(Q=q, RO=ro, S=s, Y=y, m=17, **d)
    # an all-zero row: zero codes, scale one (check_rows.py:186-190)
    assert not gu.host(q)[6].any() and float(gu.host(s)[6]) == 1.0 and not gu.host(y)[6].any()
    # unit RMS before the gain: mean(Y / (1 + w))^2 is 1 to fp16 accuracy
    unit = gu.host(y)[:17].astype(np.float64) / (1.0 + w.astype(np.float64))
    live = [i for i in range(17) if i != 6]
    np.testing.assert_allclose((unit[live] ** 2).mean(axis=1), 1.0, rtol=2e-3)


def test_residual_norm_rotate_a8_refuses_incomplete_tiles():
    for k in (128, 5120 + 128, 0, 32768 + 256):
        with pytest.raises(Exception):
            gu.kernel("residual_norm_rotate_a8", M=4, K=k)


@pytest.mark.parametrize("m,k,swiglu", [(1, 128, False), (3, 2560, False), (2, 5120, True), (4, 384, True)])
def test_rotate_activation_gives_the_values_the_fused_kernel_quantises(m, k, swiglu):
    # kernels/cuda/model/integer_vq.py:447-486
    rng = np.random.default_rng(orc.SEED + m + k)
    x = rng.normal(size=(m, 2 * k if swiglu else k)).astype(np.float16)
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    y = torch.full((m + 1, k), 7.0, dtype=torch.float16, device=gu.DEV)
    variant = dict(M=m, K=k, swiglu=True) if swiglu else dict(M=m, K=k)
    gu.kernel("rotate_activation", **variant)(Signs=gu.dev(signs), X=gu.dev(x), Y=y)
    values = x
    if swiglu:  # the device's own fp16 SwiGLU values (the exponential may differ from libm in the last place)
        mid = torch.empty((m, k), dtype=torch.float16, device=gu.DEV)
        gu.kernel("swiglu", I=k)(X=gu.dev(x), Y=mid, rows=m)
        values = gu.host(mid)
    want = orc.rotate(values.astype(np.float32), signs).astype(np.float16)
    np.testing.assert_array_equal(gu.host(y)[:m], want)
    assert (gu.host(y)[m] == 7).all()
    # A8 of these values is what rotate_activation_a8 writes
    q = torch.zeros((m, k), dtype=torch.int8, device=gu.DEV)
    s = torch.zeros((m,), dtype=torch.float16, device=gu.DEV)
    gu.kernel("rotate_activation_a8", **variant)(Q=q, S=s, Signs=gu.dev(signs), X=gu.dev(x))
    want_q, want_s = orc.a8(gu.host(y)[:m])
    np.testing.assert_array_equal(gu.host(q), want_q)
    np.testing.assert_array_equal(gu.host(s), want_s[:, 0])
    with pytest.raises(Exception):
        gu.kernel("rotate_activation", M=2, K=192)


@pytest.mark.parametrize("m,block_m", [(1, None), (3, None), (8, 8), (6, 2)])
def test_int8_small_projection_symbol(m, block_m):
    # kernels/cuda/model/int8_projection.py:65-107: same buffers and arithmetic as int8_projection
    rng = np.random.default_rng(orc.SEED + m)
    n, k = 136, 384
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    ts = rng.uniform(0.01, 0.03, m).astype(np.float16)
    variant = dict(M=m, N=n, K=k, block_n=8, output_stride=n + 8)
    if block_m:
        variant["block_m"] = block_m
    out = torch.full((m, n + 8), 9.0, dtype=torch.float16, device=gu.DEV)
    gu.kernel("int8_small_projection", **variant)(A=gu.dev(a), Output=out, TokenScale=gu.dev(ts), Weight=gu.dev(w),
                                                  WeightScale=gu.dev(ws))
    np.testing.assert_array_equal(gu.host(out)[:, :n], orc.project(a, ts, w, ws))
    assert (gu.host(out)[:, n:] == 9).all()
    for bad in (dict(block_m=9), dict(block_n=32), dict(block_m=0)):
        with pytest.raises(Exception):
            gu.kernel("int8_small_projection", M=4, N=n, K=k, **bad)


@pytest.mark.parametrize("n,k,packed_k", [(9728, 2560, 0), (17408, 5120, 0), (200, 1024, 0), (4096, 8192, 0),
                                          (17408, 5120, 128), (136, 2048, 128)])
def test_q4_gemv_quantises_fp16_input_itself(n, k, packed_k):
    """input_dtype=float16: one launch gives what activation_quantization + e8p_q4_projection give."""
    rng = np.random.default_rng(orc.SEED + n + k)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    stored = gu.dev(packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k))
    kern = gu.kernel("e8p_q4_projection", M=1, N=n, K=k, packed_k=packed_k, input_dtype="float16")
    weights = orc.q4_integers(packed, TABLE)
    out = torch.full((2, n), 9.0, dtype=torch.float16, device=gu.DEV)
    a_scale = torch.full((2,), 7.0, dtype=torch.float16, device=gu.DEV)
    for case in range(3):
        x = rng.normal(size=(1, k)).astype(np.float16)
        if case == 1:
            x[0, :4] = [900, -900, 0, 1e-7]  # a large maximum: most codes are zero
        if case == 2:
            x[:] = 0                              # zero row: scale one, zero output
        kern(A=gu.dev(x), AS=a_scale, Book=gu.book(), Out=out, S=gu.dev(scales), W=stored)
        a_q, a_s = orc.a8(x)
        np.testing.assert_array_equal(gu.host(a_scale)[:1], a_s[:, 0])
        np.testing.assert_array_equal(gu.host(out)[:1], orc.project(a_q, a_s, weights, scales))
        assert float(gu.host(a_scale)[1]) == 7.0 and (gu.host(out)[1] == 9).all()


@pytest.mark.parametrize("n,k,packed_k", [(9728, 2560, 0), (17408, 5120, 0), (200, 1024, 0), (17408, 5120, 128)])
def test_q4_gemv_rotates_and_quantises_fp16_input(n, k, packed_k):
    """input_dtype=float16, rotate=true: one launch gives what rotate_activation_a8 + e8p_q4_projection give."""
    rng = np.random.default_rng(orc.SEED + n + k + 1)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    stored = gu.dev(packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k))
    kern = gu.kernel("e8p_q4_projection", M=1, N=n, K=k, packed_k=packed_k, input_dtype="float16", rotate=True,
                     workspace=False)
    assert kern.arg_names == ["A", "AS", "Book", "Out", "S", "Signs", "W"]
    weights = orc.q4_integers(packed, TABLE)
    out = torch.full((2, n), 9.0, dtype=torch.float16, device=gu.DEV)
    a_scale = torch.full((2,), 7.0, dtype=torch.float16, device=gu.DEV)
    for case in range(3):
        x = rng.normal(size=(1, k)).astype(np.float16)
        if case == 1:
            x[0, :4] = [900, -900, 0, 1e-7]
        if case == 2:
            x[:] = 0
        kern(A=gu.dev(x), AS=a_scale, Book=gu.book(), Out=out, S=gu.dev(scales), Signs=gu.dev(signs), W=stored)
        a_q, a_s = orc.rotate_a8(x, signs)
        np.testing.assert_array_equal(gu.host(a_scale)[:1], a_s[:, 0])
        np.testing.assert_array_equal(gu.host(out)[:1], orc.project(a_q, a_s, weights, scales))
        assert float(gu.host(a_scale)[1]) == 7.0 and (gu.host(out)[1] == 9).all()
    with pytest.raises(Exception):
        gu.kernel("e8p_q4_projection", M=1, N=n, K=k, rotate=True)


@pytest.mark.parametrize("n,k,packed_k", [
    (1027, 5120, 128), (515, 5120, 64), (517, 3072, 128), (35, 6144, 128), (34, 8192, 64),                        # 32 lanes to a K-major channel: 5, 3, 6 and 8 steps
    (10240, 4096, 128), (10241, 4096, 128), (12289, 4096, 128), (20481, 3072, 128), (258, 3072, 0), (35, 6144, 0),  # both sides of its lines; six steps, which nothing holds
    (70, 1024, 128), (71, 1024, 64), (6144, 1024, 0), (6145, 1024, 0), (67, 2048, 0), (66, 2048, 128)])             # 8 lanes; 16 where 32 divide
def test_one_row_with_other_lanes_than_the_handle_says(n, k, packed_k):
    """The lanes to a channel that a launch takes by the channels that a CU gets, int8 and rotated fp16 rows, codes on both sides of the overflow plane."""
    rng = np.random.default_rng(orc.SEED + n + k)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    weights = orc.q4_integers(packed, TABLE)
    stored = gu.dev(packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k))
    q = rng.integers(-128, 128, (1, k), dtype=np.int8)
    q[0, k // 2 :] = np.clip(q[0, k // 2 :], -127, 119)  # (chunks without an overflow)
    ones = np.ones(1, np.float16)
    got = gu.q4_project(gu.dev(q), gu.dev(ones), stored, gu.dev(scales), algorithm="gemv", packed_k=packed_k)
    np.testing.assert_array_equal(gu.host(got), orc.project(q, ones[:, None], weights, scales))
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    x = rng.normal(size=(1, k)).astype(np.float16)
    kern = gu.kernel("e8p_q4_projection", M=1, N=n, K=k, packed_k=packed_k, input_dtype="float16", rotate=True)
    out = torch.full((2, n), 9.0, dtype=torch.float16, device=gu.DEV)
    scale = torch.empty(1, dtype=torch.float16, device=gu.DEV)
    kern(A=gu.dev(x), AS=scale, Book=gu.book(), Out=out, S=gu.dev(scales), Signs=gu.dev(signs), W=stored)
    a_q, a_s = orc.rotate_a8(x, signs)
    np.testing.assert_array_equal(gu.host(out)[:1], orc.project(a_q, a_s, weights, scales))
    assert (gu.host(out)[1] == 9).all()


@pytest.mark.parametrize("n,k,packed_k,single", [(200, 1024, 0, True), (136, 2048, 128, True), (48, 8192, 0, True), (40, 8704, 0, False), (64, 1152, 128, False)])
def test_one_row_program_gives_the_bits_of_two_launches(n, k, packed_k, single):
    """One launch quantises the row, publishes its codes and projects; shapes and addresses it does not take keep the two launches."""
    rng = np.random.default_rng(orc.SEED + n + k)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    linear = programs.QuantizedLinear("q4", packed, scales, 4, packed_k=packed_k)
    assert (linear.single is not None) == single
    weights = orc.q4_integers(packed, TABLE)
    for offset in (0, 1):  # the second row starts at an odd fp16
        padded = torch.zeros(k + 8, dtype=torch.float16, device=gu.DEV)
        x = padded[offset : offset + k].view(1, k)
        x.copy_(torch.from_numpy((rng.normal(size=(1, k)) * 3).astype(np.float16)))
        linear.a_q.fill_(99)
        out = gu.host(linear.run(x)).copy()
        a_q, a_s = orc.a8(gu.host(x))
        np.testing.assert_array_equal(gu.host(linear.a_q)[:1], a_q)
        assert (gu.host(linear.a_q)[1:] == 99).all()
        np.testing.assert_array_equal(gu.host(linear.a_s)[:1], a_s)
        np.testing.assert_array_equal(out, orc.project(a_q, a_s, weights, scales))


@pytest.mark.parametrize("n,k,packed_k", [
    (17, 512, 0), (300, 1536, 0), (4097, 2560, 0), (5, 4608, 0), (2000, 5120, 0),            # odd and even steps to a wave; fewer workgroups than steps
    (17, 1024, 128), (4200, 3072, 128), (33, 5120, 128), (258, 2048, 64), (8448, 5120, 64)])
@pytest.mark.parametrize("rows", [1, 2, 4, 5, 8])
def test_few_rows_quantised_by_the_projection(rows, n, k, packed_k):
    """One launch leaves the codes, scales and outputs of the quantiser and the projection, of rows with a NaN, an infinity and zeros too, and nothing behind its rows."""
    rng = np.random.default_rng(orc.SEED + rows + n + k)
    stored = torch.from_numpy(rng.integers(-(2**31), 2**31, n * k // 8).astype(np.int32)).to(gu.DEV)
    scales = gu.dev(rng.uniform(0.005, 0.02, n).astype(np.float16))
    x = (rng.normal(size=(rows, k)) * 3).astype(np.float16)
    x[rows - 1, -1] = 500
    if rows > 4:
        x[0], x[1, k // 2], x[2, 3], x[2, -2] = 0, np.inf, np.nan, -900
    f16 = dict(dtype=torch.float16, device=gu.DEV)
    out, a_s, a_q = torch.full((rows + 1, n + 8), 9.0, **f16), torch.full((rows + 1,), 7.0, **f16), torch.full((rows + 1, k), 99, dtype=torch.int8, device=gu.DEV)
    few = lib.Kernel("e8p_q4_projection", M=rows, N=n, K=k, packed_k=packed_k, output_stride=n + 8, quantize=True)
    few(A=gu.dev(x), AS=a_s, Book=gu.book(), Out=out, Q=a_q, S=scales, W=stored)
    want_q, want_s = gu.a8(gu.dev(x))
    want = gu.q4_project(want_q, want_s.view(-1), stored, scales, packed_k=packed_k)
    assert torch.equal(a_q[:rows], want_q) and torch.equal(a_s[:rows], want_s[:, 0])
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], gu.host(want))
    assert (a_q[rows:] == 99).all() and (a_s[rows:] == 7).all() and (out[rows:] == 9).all() and (out[:, n:] == 9).all()


@pytest.mark.parametrize("rows,n,k,packed_k", [(1, 40, 512, 0), (3, 300, 2560, 0), (4, 17, 1024, 128), (5, 272, 3072, 64), (8, 1000, 5120, 128), (7, 33, 4608, 0)])
def test_few_rows_quantised_by_the_projection_against_the_oracle(rows, n, k, packed_k):
    rng = np.random.default_rng(orc.SEED + rows + k)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    x = (rng.normal(size=(rows, k)) * np.where(rng.random((1, k)) < 0.01, 40, 1)).astype(np.float16)
    x[0, :64] = 0
    f16 = dict(dtype=torch.float16, device=gu.DEV)
    out, a_s, a_q = torch.empty((rows, n), **f16), torch.empty(rows, **f16), torch.empty((rows, k), dtype=torch.int8, device=gu.DEV)
    lib.Kernel("e8p_q4_projection", M=rows, N=n, K=k, packed_k=packed_k, quantize=True)(
        A=gu.dev(x), AS=a_s, Book=gu.book(), Out=out, Q=a_q, S=gu.dev(scales), W=gu.dev((orc.q4_pack_k(packed, packed_k) if packed_k else packed).view(np.int32)))
    want_q, want_s = orc.a8(x)
    np.testing.assert_array_equal(gu.host(a_q), want_q)
    np.testing.assert_array_equal(gu.host(a_s), want_s[:, 0])
    np.testing.assert_array_equal(gu.host(out), orc.project(want_q, want_s, orc.q4_integers(packed, TABLE), scales))


@pytest.mark.parametrize("k,packed_k,served", [(1024, 128, True), (2560, 0, True), (1536, 128, False), (5632, 0, False)])
def test_few_rows_of_a_linear(k, packed_k, served):
    """Which rows and addresses a linear hands to the projection as they are; all of them give the bits of two launches, rows after others as well."""
    rng = np.random.default_rng(orc.SEED + k)
    linear = programs.QuantizedLinear("q4", rng.integers(0, 2**32, (200, k // 8), dtype=np.uint32), rng.uniform(0.005, 0.02, 200).astype(np.float16), 12, packed_k=packed_k)
    assert (linear.few is not None) == served
    for rows, offset in ((2, 0), (9, 0), (8, 0), (3, 1), (4, 8)):
        x = torch.zeros(rows * k + 8, dtype=torch.float16, device=gu.DEV)[offset : offset + rows * k].view(rows, k)
        x.copy_(torch.from_numpy((rng.normal(size=(rows, k)) * 3).astype(np.float16)))
        got, codes, a_s = linear.run(x).clone(), linear.a_q[:rows].clone(), linear.a_s[:rows].clone()
        want = linear.project(linear.quantize(x))
        assert torch.equal(got, want) and torch.equal(codes, linear.a_q[:rows]) and torch.equal(a_s, linear.a_s[:rows])


def test_quantize_is_refused_beside_keys_of_other_kernels():
    good = dict(M=8, N=256, K=1024, quantize=True)
    lib.Kernel("e8p_q4_projection", **good)
    for other in (dict(M=9), dict(K=1152), dict(K=6144), dict(K=1536, packed_k=128), dict(workspace=True), dict(algorithm="runs"), dict(block_m=32), dict(panels=True),
                  dict(input_dtype="float16"), dict(split_k=True), dict(decode_in_gemm=True), dict(quantize=3)):
        with pytest.raises(Exception):
            lib.Kernel("e8p_q4_projection", **{**good, **other})


@pytest.mark.parametrize("codec", ["q4", "w8"])
def test_a_result_of_a_linear_is_the_callers_own_tensor(codec):
    """What a caller does to the shape of one result leaves the next one, and `out`, as they are."""
    rng = np.random.default_rng(orc.SEED + 5)
    weight = rng.integers(0, 2**32, (256, 64), dtype=np.uint32) if codec == "q4" else rng.integers(-127, 128, (256, 512), dtype=np.int8)
    linear = programs.QuantizedLinear(codec, weight, rng.uniform(0.005, 0.02, 256).astype(np.float16), 4)
    for rows in (1, 3, 4):
        x = gu.dev(rng.normal(size=(rows, 512)).astype(np.float16))
        first = linear.run(x)
        want = first.clone()
        first.t_()
        second = linear.run(x)
        assert second.shape == (rows, 256) and torch.equal(second, want) and second.data_ptr() == linear.out.data_ptr()
        second.resize_((1, 2))
        third = linear.project(rows)
        assert third.shape == (rows, 256) and torch.equal(third, want) and linear.out.shape == (4, 256)


def test_q4_fp16_input_is_refused_where_no_kernel_serves_it():
    for variant in (dict(M=2, N=256, K=1024), dict(M=1, N=256, K=1024, algorithm="mfma"), dict(M=1, N=256, K=16384),
                    dict(M=1, N=256, K=1024, input_dtype="bfloat16")):
        variant.setdefault("input_dtype", "float16")
        with pytest.raises(Exception):
            gu.kernel("e8p_q4_projection", **variant)


@pytest.mark.parametrize("codec,m,n,k,dtype", [("q4", 128, 8704, 512, "float16"), ("q4", 70, 8300, 384, "float16"),
                                               ("w8", 128, 8704, 256, "float16"), ("w8", 300, 8450, 384, "float32"),
                                               ("q4", 256, 17408, 256, "float16"), ("w8", 40, 2048, 1024, "float16"),
                                               ("w8", 17, 5120, 512, "float32")])
def test_mid_row_projections_split_k_steps_evenly(codec, m, n, k, dtype):
    """The 128-row tiles by name: the K steps of the tiles are dealt evenly to one workgroup per CU, runs that
    do not cover a whole tile meet as int32 partial sums.  Same bytes as whole tiles in one launch."""
    rng = np.random.default_rng(orc.SEED + m + n)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    a_s = rng.uniform(0.01, 0.03, m).astype(np.float16)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    torch_dtype = torch.float16 if dtype == "float16" else torch.float32
    stride = n + 8
    if codec == "q4":
        packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
        weights = orc.q4_integers(packed, TABLE)
        symbol, stored = "e8p_q4_projection", gu.dev(packed)
        call = lambda kern, out: kern(A=gu.dev(a), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=stored)
    else:
        weights = rng.integers(-128, 128, (n, k), dtype=np.int8)
        symbol, stored = "int8_projection", gu.dev(weights)
        call = lambda kern, out: kern(A=gu.dev(a), Output=out, TokenScale=gu.dev(a_s), Weight=stored, WeightScale=gu.dev(scales))
    variant = dict(M=m, N=n, K=k, output_dtype=dtype, output_stride=stride)
    # by name: `auto` gives few rows to the streaming kernel or the channel runs, and more int8 rows to the 128 x 128 tiles of k_mid.hip, split or not
    variant["algorithm"] = "mfma"
    split = gu.kernel(symbol, **variant)
    whole = gu.kernel(symbol, split_k=False, **variant)
    grid_split, grid_whole = tuple(split.geometry()[0]), tuple(whole.geometry()[0])
    assert grid_split[1] == 1 and grid_whole[0] == -(-n // 128) and grid_whole[1] == -(-m // 128)
    assert started(split, m)[0] == (grid_split[0], 256, 0) and len(started(split, m)) == 2  # the steps, the sums
    assert started(whole, m) == [(grid_whole[0], 256, 0)]
    out = torch.full((m + 1, stride), 9.0, dtype=torch_dtype, device=gu.DEV)
    other = torch.full((m + 1, stride), 9.0, dtype=torch_dtype, device=gu.DEV)
    call(split, out)
    call(whole, other)
    assert torch.equal(out, other)
    want = orc.project(a, a_s, weights, scales, out_dtype=np.float16 if dtype == "float16" else np.float32)
    np.testing.assert_array_equal(gu.host(out)[:m, :n], want)
    assert (gu.host(out)[m] == 9).all() and (gu.host(out)[:, n:] == 9).all()
    # again into the same buffers: the partial slots carry nothing over
    out.fill_(9)
    call(split, out)
    assert torch.equal(out, other)


@pytest.mark.parametrize("codec,m,n,k,dtype,pad,parts", [
    ("w8", 513, 144, 128, "float16", 0, 1), ("w8", 640, 257, 256, "float16", 3, 1),     # one and two K steps of four stages
    ("w8", 600, 1000, 384, "float32", 0, 1), ("q4", 521, 528, 512, "float16", 8, 1),    # three, and as many as there are stages
    ("w8", 700, 400, 640, "float16", 1, 1), ("q4", 650, 130, 1152, "float32", 5, 1),    # more of them
    ("w8", 2050, 2064, 256, "float16", 0, 1), ("q4", 1100, 4112, 640, "float16", 8, 1),  # two workgroups to a CU, two stages
    ("w8", 520, 250, 14336, "float16", 4, 8), ("q4", 770, 256, 8320, "float16", 0, 8), ("w8", 641, 1930, 14336, "float32", 2, 5)])  # tiles in parts of K
def test_tiles_of_128_by_128(codec, m, n, k, dtype, pad, parts):
    """The edges of tiles, steps and stages; rows that start at any address; nothing beyond the rows and channels is written."""
    rng = np.random.default_rng(orc.SEED + m + n)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    a_s = rng.uniform(0.01, 0.03, m).astype(np.float16)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    stride = n + pad
    variant = dict(M=m, N=n, K=k, output_dtype=dtype, output_stride=stride, workspace=True)
    if codec == "q4":
        packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
        weights, stored = orc.q4_integers(packed, TABLE), gu.dev(packed)
        kern = gu.lib.Kernel("e8p_q4_projection", **variant)
        call = lambda out: kern(A=gu.dev(a), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=stored, Workspace=kern.workspace())
    else:
        weights = rng.integers(-128, 128, (n, k), dtype=np.int8)
        stored, kern = gu.dev(weights), gu.lib.Kernel("int8_projection", **variant)
        call = lambda out: kern(A=gu.dev(a), Output=out, TokenScale=gu.dev(a_s), Weight=stored, WeightScale=gu.dev(scales), Workspace=kern.workspace())
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        tiles = -(-m // 128) * -(-n // 128)
        assert kern.workspace_bytes(m) == (n * k if codec == "q4" else 0) + (tiles * parts * 65536 if parts > 1 else 0)
        assert started(kern, m)[codec == "q4"] == (tiles * parts, 256, MID_4 if tiles * parts <= 256 else MID_2)
    threads, _ = kern.query(m)
    assert threads == np.prod(kern.geometry(m)[1])  # a record names the reported block
    want = orc.project(a, a_s, weights, scales, out_dtype=np.float16 if dtype == "float16" else np.float32)
    flat = torch.full(((m + 1) * stride + 1,), 9.0, dtype=torch.float16 if dtype == "float16" else torch.float32, device=gu.DEV)
    for shift in (0, 1):
        flat.fill_(9)
        call(flat[shift : shift + (m + 1) * stride])
        out = gu.host(flat[shift : shift + (m + 1) * stride].view(m + 1, stride))
        np.testing.assert_array_equal(out[:m, :n], want)
        assert (out[m] == 9).all() and (out[:, n:] == 9).all()


@pytest.mark.parametrize("m,n,k,dtype,pad", [
    (1224, 18784, 256, "float16", 0), (1224, 18784, 384, "float32", 0), (2100, 17000, 512, "float16", 3), (1224, 18784, 640, "float16", 0)])
def test_persistent_tiles_of_short_k(m, n, k, dtype, pad):
    """Two and three K steps, whose requests are spread over three phases, four and five, over two; more tiles than workgroups, ragged ones among them."""
    generator = torch.Generator(device=gu.DEV).manual_seed(orc.SEED + m + k)
    a, weights = (torch.randint(-128, 128, (rows, k), generator=generator, device=gu.DEV, dtype=torch.int8) for rows in (m, n))
    a_s, scales = (torch.rand(rows, generator=generator, device=gu.DEV).add(0.5).mul(0.01).half() for rows in (m, n))
    # sums of up to 640 products of 2^14 at most are integers below 2^24: exact in float32, in any order
    want = (((a.float() @ weights.float().t()) * scales.float()) * a_s.float()[:, None]).to(getattr(torch, dtype))
    kern = gu.kernel("int8_projection", M=m, N=n, K=k, output_dtype=dtype, output_stride=n + pad)
    out = torch.full((m + 1, n + pad), 9.0, dtype=want.dtype, device=gu.DEV)
    for _ in range(2):
        kern(A=a, Output=out, TokenScale=a_s, Weight=weights, WeightScale=scales)
        assert torch.equal(out[:m, :n], want)
        assert (out[m] == 9).all() and (out[:, n:] == 9).all()


@pytest.mark.parametrize("dtype,pad", [("float16", 0), ("float32", 3)])
@pytest.mark.parametrize("packed_k,n,k", [
    (0, 1, 2816), (0, 4096, 2816), (0, 4099, 8320), (0, 8208, 4224), (0, 40, 3584), (0, 16400, 5760),  # no tables, 16 lanes; one to five blocks
    (128, 33, 2304), (128, 4112, 3328), (128, 8208, 4352), (128, 70, 3584), (128, 4096, 2944), (64, 333, 9984)])
def test_one_row_of_codes_in_the_channel_runs(packed_k, n, k, dtype, pad):
    """At the edges of the rule; the record of the kernel before still launches, and nothing beyond the row is written."""
    rng = np.random.default_rng(orc.SEED + n + k)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    a = rng.integers(-127, 128, (1, k), dtype=np.int8)
    a_s, scales = rng.uniform(0.01, 0.03, 1).astype(np.float16), rng.uniform(0.005, 0.02, n).astype(np.float16)
    stored = gu.dev(codebook.q4_to_k_major(packed, packed_k) if packed_k else packed)
    want = orc.project(a, a_s, orc.q4_integers(packed, TABLE), scales, out_dtype=np.float16 if dtype == "float16" else np.float32)
    for rows in (1, 4):  # a handle of one row, and one that serves several
        variant = dict(M=rows, N=n, K=k, packed_k=packed_k, output_dtype=dtype, output_stride=n + pad, dynamic_rows=rows > 1)
        kern = gu.lib.Kernel("e8p_q4_projection", **variant)
        out = torch.full((2, n + pad), 9.0, dtype=torch.float16 if dtype == "float16" else torch.float32, device=gu.DEV)
        kern(A=gu.dev(a), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=stored, **({"m": 1} if rows > 1 else {}))
        got = gu.host(out)
        np.testing.assert_array_equal(got[:1, :n], want)
        assert (got[0, n:] == 9).all() and (got[1] == 9).all()
        assert started(kern, 1)[0][1:] == (512, RUNS)
        threads, _ = kern.query(1)
        assert threads == np.prod(kern.geometry(1)[1])


@pytest.mark.parametrize("codec,packed_k,rows,n,k", [
    ("q4", 0, 2, 4096, 2816), ("q4", 128, 16, 1030, 3456), ("q4", 128, 17, 333, 2304), ("q4", 0, 32, 70, 2432),      # one block of channels to a CU
    ("q4", 128, 16, 4112, 8192), ("q4", 0, 32, 4100, 12288), ("q4", 0, 2, 8208, 4224),                                  # two, three
    ("q4", 0, 2, 8200, 1152), ("q4", 0, 4, 16400, 1152), ("q4", 0, 3, 20500, 1408),                                     # the streaming kernel
    ("q4", 0, 96, 8300, 2048), ("q4", 128, 128, 4130, 2176), ("q4", 128, 247, 5904, 2304), ("q4", 64, 256, 4300, 2048), ("q4", 0, 270, 8192, 1536),
    ("w8", 0, 65, 14960, 1152), ("w8", 0, 128, 9000, 1024), ("w8", 0, 120, 1000, 8320),
    ("q4", 128, 24, 4100, 12288), ("q4", 0, 2, 12289, 1152), ("q4", 128, 82, 9928, 2176), ("w8", 0, 65, 23909, 256)])
def test_rows_that_leave_the_reported_kernel(codec, packed_k, rows, n, k):
    """Shapes at the edges of the rules by which a launch takes the channel runs or the streaming kernel while its records name another; of four the records name it too."""
    rng = np.random.default_rng(orc.SEED + rows + n + k)
    a = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_s, scales = rng.uniform(0.01, 0.03, rows).astype(np.float16), rng.uniform(0.005, 0.02, n).astype(np.float16)
    out = torch.full((rows + 1, n), 9.0, dtype=torch.float16, device=gu.DEV)
    if codec == "q4":
        packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
        weights = orc.q4_integers(packed, TABLE)
        kern = gu.kernel("e8p_q4_projection", M=512, N=n, K=k, packed_k=packed_k, dynamic_rows=True)
        kern(A=gu.dev(a), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=gu.dev(codebook.q4_to_k_major(packed, packed_k) if packed_k else packed),
             Workspace=kern.workspace(), m=rows)
    else:
        weights = rng.integers(-127, 128, (n, k), dtype=np.int8)
        kern = gu.kernel("int8_projection", M=512, N=n, K=k, dynamic_rows=True)
        kern(A=gu.dev(a), Output=out, TokenScale=gu.dev(a_s), Weight=gu.dev(weights), WeightScale=gu.dev(scales), Workspace=kern.workspace(), m=rows)
    got = gu.host(out)
    np.testing.assert_array_equal(got[:rows], orc.project(a, a_s, weights, scales, out_dtype=np.float16))
    assert (got[rows] == 9).all()
    (only,) = started(kern, rows)
    assert only[2] == RUNS or (only == (-(-n // 32), 512, 0) and rows <= 4)  # the channel runs, or the streaming kernel
    assert (only == reported(kern, rows)) == ((codec, rows, n, k) in {("q4", 32, 4100, 12288), ("q4", 2, 8200, 1152), ("q4", 128, 4130, 2176), ("w8", 65, 14960, 1152)})
    threads, _ = kern.query(rows)
    assert threads == np.prod(kern.geometry(rows)[1])


@pytest.mark.parametrize("packed_k", [128, 64])
def test_split_launches_serve_k_major_codes_and_dynamic_rows(packed_k):
    rng = np.random.default_rng(orc.SEED + 91)
    n, k, cap = 8704, 384, 256
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    weights = orc.q4_integers(packed, TABLE)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    # by name: `auto` gives 65 rows of so short a K to the channel runs over all rows
    kern = gu.kernel("e8p_q4_projection", M=cap, N=n, K=k, packed_k=packed_k, dynamic_rows=True, algorithm="mfma")
    stored = gu.dev(orc.q4_pack_k(packed, packed_k))
    for m in (200, 65, 130):
        a = rng.integers(-128, 128, (cap, k), dtype=np.int8)
        a_s = rng.uniform(0.01, 0.03, cap).astype(np.float16)
        out = torch.full((cap, n), 9.0, dtype=torch.float16, device=gu.DEV)
        assert tuple(kern.geometry(m)[0])[1] == 1 and kern.workspace_bytes(m) > 0  # one workgroup list: the split form
        kern(A=gu.dev(a), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=stored, m=m)
        np.testing.assert_array_equal(gu.host(out)[:m], orc.project(a[:m], a_s[:m], weights, scales))
        assert (gu.host(out)[m:] == 9).all()


def test_q4_embedding_gather_matches_oracle():
    rng = np.random.default_rng(orc.SEED + 40)
    vocab, hidden, cap = 50, 640, 16
    packed = rng.integers(0, 2**32, (vocab, hidden // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, vocab).astype(np.float16)
    signs = rng.choice(np.array([-1, 1], np.int8), hidden)
    ids = np.array([0, 49, 7, -1, 50, 7, 2**31 - 1, 13, 1], np.int32)
    kern = gu.kernel("e8p_q4_embedding", M=cap, vocab=vocab, hidden=hidden)
    out = torch.full((cap, hidden), 3.0, dtype=torch.float16, device=gu.DEV)
    padded = np.zeros(cap, np.int32)
    padded[: len(ids)] = ids
    kern(Book=gu.book(), IDs=gu.dev(padded), Output=out, Scale=gu.dev(scales), Signs=gu.dev(signs),
         Weight=gu.dev(orc.q4_pack_k(packed, 128)), m=len(ids))
    got = gu.host(out)
    np.testing.assert_array_equal(got[: len(ids)], orc.q4_embedding(ids, packed, TABLE, scales, signs))
    assert not got[3].any() and not got[4].any() and not got[6].any() and (got[len(ids):] == 3).all()


@pytest.mark.parametrize("m,n,k", [(1, 96, 256), (6, 200, 1024), (70, 130, 384), (300, 260, 256), (64, 512, 2048),
                                   (129, 64, 128)])
def test_int8_swiglu_gate_up_boundary(m, n, k):
    rng = np.random.default_rng(orc.SEED + m + n)
    a_q = rng.integers(-127, 128, (m, k), dtype=np.int8)
    a_s = rng.uniform(0.005, 0.02, m).astype(np.float16)
    gate, up = (rng.integers(-127, 128, (n, k), dtype=np.int8) for _ in range(2))
    gs, us = (rng.uniform(0.001, 0.004, n).astype(np.float16) for _ in range(2))
    out = torch.full((m + 1, n), 2.0, dtype=torch.float16, device=gu.DEV)
    gu.kernel("int8_swiglu", M=m, N=n, K=k)(A=gu.dev(a_q), Gate=gu.dev(gate), GateScale=gu.dev(gs), Output=out,
                                            TokenScale=gu.dev(a_s), Up=gu.dev(up), UpScale=gu.dev(us))
    got = gu.host(out)
    want = orc.int8_swiglu(a_q, a_s, gate, gs, up, us)
    # the two projections inside are exact integers rounded to fp16 as the oracle rounds them; only exp()
    # may differ in the last place between the device and libm: one fp16 step at most, rarely
    np.testing.assert_allclose(got[:m].astype(np.float32), want.astype(np.float32), rtol=1e-3, atol=1e-2)
    assert ulps_fp16(got[:m], want).max() <= 1
    assert np.mean(got[:m] == want) > 0.99 and (got[m:] == 2).all()


# ---- Q4A8 projections -----------------------------------------------------
def q4_case(rng, m, n, k):
    x = (rng.normal(size=(m, k))).astype(np.float16)
    a_q, a_s = orc.a8(x)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    return a_q, a_s[:, 0].copy(), packed, scales


@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k", [(65, 256), (257, 2560), (1024, 5120), (130, 17408), (33, 8192 + 512), (70, 1536)])
def test_q4_gemv_matches_oracle(m, n, k):
    rng = np.random.default_rng(orc.SEED + m + n)
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :4] = [-128, -1, 0, 127]  # extremes outside the A8 range must still be exact
    w = orc.q4_integers(packed, TABLE)
    acc = orc.int_dot(a_q, w)
    ones_n, ones_m = np.ones(n, np.float16), np.ones(m, np.float16)
    got_acc = gu.q4_project(gu.dev(a_q), gu.dev(ones_m), gu.dev(packed), gu.dev(ones_n), dtype=torch.float32,
                            algorithm="gemv")
    np.testing.assert_array_equal(gu.host(got_acc).astype(np.int64), acc.astype(np.int64))
    got = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), algorithm="gemv")
    want = orc.rescale(acc, scales, a_s)
    assert_close_fp16(gu.host(got), want)
    np.testing.assert_array_equal(gu.host(got), want)


@pytest.mark.parametrize("blocks_of", [128, 64])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k", [(65, 256), (257, 2560), (1024, 5120), (130, 16384), (33, 8192 + 512), (7, 1536), (17408, 5120),
                                 (40, 17408), (9, 768)])
def test_q4_gemv_k_major_codes_match_oracle(m, n, k, blocks_of):
    """The reference's storage layouts (K/128 blocks of N rows, or K/64: e8p_q4.py:78-80): 16 lanes per row and tasks of 4
    adjacent rows, or 8 lanes and 8 rows when K is a multiple of 256 only."""
    rng = np.random.default_rng(orc.SEED + 500 + m + n)
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :4] = [-128, -1, 0, 127]
    stored = orc.q4_pack_k(packed, blocks_of)
    w = orc.q4_integers(packed, TABLE)
    acc = orc.int_dot(a_q, w)
    ones_n, ones_m = np.ones(n, np.float16), np.ones(m, np.float16)
    planes_fit = 131072 + (1 if m == 1 else 2 if m == 2 else 4) * (k // 8) * 12 + 256 + k // 32 + 16 <= 160 * 1024
    if not planes_fit:  # the activation planes of so many rows do not fit beside the tables: refused at launch
        with pytest.raises(Exception, match="K-major"):
            gu.q4_project(gu.dev(a_q), gu.dev(ones_m), gu.dev(stored), gu.dev(ones_n), algorithm="gemv", packed_k=blocks_of)
        return
    got_acc = gu.q4_project(gu.dev(a_q), gu.dev(ones_m), gu.dev(stored), gu.dev(ones_n), dtype=torch.float32,
                            algorithm="gemv", packed_k=blocks_of)
    np.testing.assert_array_equal(gu.host(got_acc).astype(np.int64), acc.astype(np.int64))
    storage = torch.full((m + 1, n + 5), 91.0, dtype=torch.float16, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 5,
                  algorithm="gemv", packed_k=blocks_of)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.rescale(acc, scales, a_s))
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()
    if m <= 2:  # what `auto` picks for K-major codes at 1 and 2 rows
        auto = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), packed_k=blocks_of)
        np.testing.assert_array_equal(gu.host(auto), orc.rescale(acc, scales, a_s))


def test_q4_gemv_k_major_refuses_what_it_cannot_read():
    with pytest.raises(Exception, match="gemv"):
        gu.kernel("e8p_q4_projection", M=1, N=64, K=384, packed_k=128, algorithm="gemv")


@pytest.mark.parametrize("variant", [{}, {"gemv_passes": 1}], ids=["replicated-tables", "compact-tables"])
@pytest.mark.parametrize("m", [1, 2, 4])
@pytest.mark.parametrize("pattern", ["all_max", "band", "sparse", "negative"])
def test_q4_gemv_activation_extremes(m, pattern, variant):
    """Activations at and around the top of the int8 range: the GEMV splits them into signed
    nibbles, and values of 120..127 take a separate path that random data visits rarely."""
    n, k = 193, 5120
    rng = np.random.default_rng(orc.SEED + 77 + m)
    if pattern == "all_max":
        a_q = np.full((m, k), 127, np.int8)
    elif pattern == "band":                       # every boundary value, many times
        a_q = rng.choice(np.array([111, 112, 119, 120, 121, 126, 127, -120, -121, -127, -128, 7, 8, -8, -9, 0], np.int8),
                         size=(m, k))
    elif pattern == "sparse":                     # one overflow in the last chunk of the last row only
        a_q = rng.integers(-119, 120, (m, k)).astype(np.int8)
        a_q[m - 1, k - 1] = 124
    else:
        a_q = rng.integers(-128, -119, (m, k)).astype(np.int8)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    acc = orc.int_dot(a_q, orc.q4_integers(packed, TABLE))
    np.testing.assert_array_equal(acc, orc.int_dot_bruteforce(a_q[:, :256], orc.q4_integers(packed[:, :32], TABLE))
                                  + orc.int_dot(a_q[:, 256:], orc.q4_integers(packed[:, 32:], TABLE)))
    got = gu.q4_project(gu.dev(a_q), gu.dev(np.ones(m, np.float16)), gu.dev(packed), gu.dev(np.ones(n, np.float16)),
                        dtype=torch.float32, algorithm="gemv", **variant)
    np.testing.assert_array_equal(gu.host(got).astype(np.int64), acc.astype(np.int64))


@pytest.mark.parametrize("packed_k", [0, 64, 128])
@pytest.mark.parametrize("m", [1, 7, 32, 33, 64, 65, 128, 129, 300])
def test_q4_mfma_rows_tails_stride_and_sentinels(m, packed_k):
    # check_e8p_q4.py:123-193: N=65, K=256, fp32 out, stride N+3, sentinel 91 beyond the tails
    rng = np.random.default_rng(orc.SEED + m)
    n, k = 65, 256
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :2] = [-128, 127]
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    storage = torch.full((m + 2, n + 3), 91.0, dtype=torch.float32, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 3,
                  dtype=torch.float32, algorithm="mfma", packed_k=packed_k)
    got = gu.host(storage)
    want = orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), scales, np.float32)
    np.testing.assert_array_equal(got[:m, :n], want)
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()


@pytest.mark.parametrize("packed_k", [0, 64, 128])
@pytest.mark.parametrize("m", [5, 8, 31, 32, 33, 64])
def test_q4_stream_rows_tails_stride_and_sentinels(m, packed_k):
    # same construction as the MFMA tail test, through the weight-streaming kernel; K=640 gives the
    # eight K slices of a workgroup uneven shares (5 blocks over 8 waves, three of them empty)
    rng = np.random.default_rng(orc.SEED + 100 + m)
    n, k = 97, 640
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :2] = [-128, 127]
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    w = orc.q4_integers(packed, TABLE)
    storage = torch.full((m + 2, n + 3), 91.0, dtype=torch.float32, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 3,
                  dtype=torch.float32, algorithm="stream", packed_k=packed_k)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(a_q, a_s, w, scales, np.float32))
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()
    ones_n, ones_m = np.ones(n, np.float16), np.ones(m, np.float16)
    acc = gu.q4_project(gu.dev(a_q), gu.dev(ones_m), gu.dev(stored), gu.dev(ones_n), dtype=torch.float32,
                        algorithm="stream", packed_k=packed_k)
    np.testing.assert_array_equal(gu.host(acc).astype(np.int64), orc.int_dot(a_q, w).astype(np.int64))
    half = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), algorithm="stream", packed_k=packed_k)
    np.testing.assert_array_equal(gu.host(half), orc.project(a_q, a_s, w, scales))


# The resident two-stage kernels (K split over the waves of one workgroup per CU, channel blocks of
# 16; K up to 5120 in steps of 512 with loader waves, up to 8192 in steps of 1024 without): every K
# they take, one and two token tiles, channel counts that leave CUs
# without work, with a part block or with several rounds of held blocks, more than 32 rows (several
# launches), the contract shape, fp32 and fp16 outputs with a stride and sentinels around them.
@pytest.mark.parametrize("m,n,k", [(5, 97, 1024), (16, 300, 2048), (17, 1000, 3072), (8, 5000, 4096), (32, 17408, 5120),
                                   (9, 4100, 6144), (31, 600, 7168), (32, 9000, 8192), (33, 513, 1024), (128, 2050, 5120),
                                   (1, 40, 2048), (3, 9728, 2560), (20, 70, 512), (7, 1111, 1536), (32, 4099, 3584),
                                   (16, 257, 4608)])
def test_q4_resident_rows_blocks_and_tails(m, n, k):
    rng = np.random.default_rng(orc.SEED + 300 + m + n)
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :2] = [-128, 127]
    w = orc.q4_integers(packed, TABLE)
    storage = torch.full((m + 2, n + 3), 91.0, dtype=torch.float32, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), out=storage, stride=n + 3,
                  dtype=torch.float32, algorithm="resident")
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(a_q, a_s, w, scales, np.float32))
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()
    ones_n, ones_m = np.ones(n, np.float16), np.ones(m, np.float16)
    acc = gu.q4_project(gu.dev(a_q), gu.dev(ones_m), gu.dev(packed), gu.dev(ones_n), dtype=torch.float32,
                        algorithm="resident")
    np.testing.assert_array_equal(gu.host(acc).astype(np.int64), orc.int_dot(a_q, w).astype(np.int64))
    half = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), algorithm="resident")
    np.testing.assert_array_equal(gu.host(half), orc.project(a_q, a_s, w, scales))
    # launched again into the same buffers (the sums in LDS start from zero every time)
    again = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), algorithm="resident")
    assert torch.equal(half, again)


@pytest.mark.parametrize("m,n,k", [(3, 97, 1024), (16, 300, 2048), (17, 1000, 3072), (8, 5000, 4096), (32, 17408, 5120),
                                   (64, 2050, 5120), (5, 40, 2048)])
@pytest.mark.parametrize("blocks_of", [128, 64])
def test_q4_resident_k_major_codes(m, n, k, blocks_of):
    """The loader/decoder kernel on the reference's storage layouts (K/128 blocks of N rows x 64 bytes, K/64 x 32)."""
    rng = np.random.default_rng(orc.SEED + 400 + m + n)
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :2] = [-128, 127]
    stored = orc.q4_pack_k(packed, blocks_of)
    w = orc.q4_integers(packed, TABLE)
    storage = torch.full((m + 2, n + 3), 91.0, dtype=torch.float32, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 3,
                  dtype=torch.float32, algorithm="resident", packed_k=blocks_of)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(a_q, a_s, w, scales, np.float32))
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()
    half = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), packed_k=blocks_of)  # what `auto` picks
    np.testing.assert_array_equal(gu.host(half), orc.project(a_q, a_s, w, scales))


def test_q4_resident_dynamic_rows_and_refusals():
    rng = np.random.default_rng(orc.SEED + 77)
    n, k = 777, 2048
    a_q, a_s, packed, scales = q4_case(rng, 100, n, k)
    w = orc.q4_integers(packed, TABLE)
    for rows in (5, 32, 33, 64, 100):
        got = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), rows=rows, dynamic=True,
                            capacity=100, algorithm="resident")
        np.testing.assert_array_equal(gu.host(got)[:rows], orc.project(a_q[:rows], a_s[:rows], w, scales))
    for bad in (dict(K=1280), dict(K=9216), dict(packed_k=128, K=1536), dict(M=129)):
        variant = dict(M=8, N=256, K=1024, algorithm="resident")
        variant.update(bad)
        with pytest.raises(Exception, match="resident"):
            gu.kernel("e8p_q4_projection", **variant)
    with pytest.raises(Exception, match="resident"):
        gu.kernel("int8_projection", M=8, N=256, K=1024, algorithm="resident")


@pytest.mark.parametrize("m,n,k", [(7, 48, 2560), (40, 65, 128), (64, 129, 640)])
def test_w8_stream_matches_oracle(m, n, k):
    rng = np.random.default_rng(orc.SEED + m)
    x = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    ws = rng.uniform(0.001, 0.01, n).astype(np.float16)
    ts = rng.uniform(0.001, 0.01, m).astype(np.float16)
    out = torch.full((m + 1, n), 99.0, dtype=torch.float16, device=gu.DEV)
    gu.w8_project(gu.dev(x), gu.dev(ts), gu.dev(w), gu.dev(ws), out=out, algorithm="stream")
    got = gu.host(out)
    np.testing.assert_array_equal(got[:m], orc.project(x, ts, w, ws))
    assert (got[m] == 99).all()


@pytest.mark.parametrize("hints", [dict(algorithm="dp4a", block_m=4, block_n=8), dict(algorithm="tensor_core", block_m=8),
                                   dict(algorithm="int4_direct", block_m=16), dict(algorithm="tensor_core", block_m=96),
                                   dict(block_m=192)], ids=lambda h: "-".join(str(v) for v in h.values()))
def test_reference_schedule_names_and_row_tiles_give_the_same_outputs(hints):
    """The reference's schedule names and row tiles (e8p_q4.py:143-215, int8_projection.py:15-48) choose among this
    library's kernels; whichever kernel a launch then runs, the output is the oracle's to the bit."""
    rng = np.random.default_rng(orc.SEED + 77)
    n, k, capacity = 449, 1024, 300
    a_q, a_s, packed, scales = q4_case(rng, capacity, n, k)
    w = orc.q4_integers(packed, TABLE)
    want = orc.project(a_q, a_s, w, scales)
    x8 = rng.integers(-128, 128, (capacity, k), dtype=np.int8)
    w8 = rng.integers(-128, 128, (n, k), dtype=np.int8)
    want8 = orc.project(x8, a_s, w8, scales)
    for rows in (1, 2, 4, 5, 20, 33, 100, 129, 200, 300):
        got = gu.q4_project(gu.dev(a_q[:rows]), gu.dev(a_s[:rows]), gu.dev(packed), gu.dev(scales), dynamic=True,
                            capacity=capacity, **hints)
        np.testing.assert_array_equal(gu.host(got), want[:rows], err_msg=f"q4 rows {rows}")
        got = gu.w8_project(gu.dev(x8[:rows]), gu.dev(a_s[:rows]), gu.dev(w8), gu.dev(scales), dynamic=True,
                            capacity=capacity, **hints)
        np.testing.assert_array_equal(gu.host(got), want8[:rows], err_msg=f"w8 rows {rows}")


@pytest.mark.parametrize("block_m", [32, 64, 128, 256])
def test_q4_mfma_tiles_and_accumulators(block_m):
    rng = np.random.default_rng(orc.SEED + block_m)
    m, n, k = 300, 384 + 65, 1024
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    acc = orc.int_dot(a_q, orc.q4_integers(packed, TABLE))
    got = gu.q4_project(gu.dev(a_q), gu.dev(np.ones(m, np.float16)), gu.dev(packed), gu.dev(np.ones(n, np.float16)),
                        dtype=torch.float32, algorithm="mfma", block_m=block_m)
    np.testing.assert_array_equal(gu.host(got).astype(np.int64), acc.astype(np.int64))
    got16 = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), algorithm="mfma", block_m=block_m)
    np.testing.assert_array_equal(gu.host(got16), orc.rescale(acc, scales, a_s))


def test_q4_dynamic_rows_one_handle_many_lengths():
    rng = np.random.default_rng(orc.SEED)
    n, k, cap = 257, 640 + 128, 128
    _, _, packed, scales = q4_case(rng, 1, n, k)
    w = orc.q4_integers(packed, TABLE)
    for m in (1, 2, 4, 5, 31, 64, 127, 128):
        x = rng.normal(size=(m, k)).astype(np.float16)
        a_q, a_s = orc.a8(x)
        out = torch.full((cap + 1, n), 7.0, dtype=torch.float16, device=gu.DEV)
        gu.q4_project(gu.dev(a_q), gu.dev(a_s[:, 0].copy()), gu.dev(packed), gu.dev(scales), dynamic=True,
                      capacity=cap, out=out)
        got = gu.host(out)
        np.testing.assert_array_equal(got[:m], orc.project(a_q, a_s[:, 0], w, scales))
        assert (got[m:] == 7).all()


# ---- W8A8 -----------------------------------------------------------------
@pytest.mark.parametrize("m,n,k", [(1, 48, 2560), (3, 65, 128), (17, 129, 640)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("algorithm", ["auto", "mfma"])
def test_w8_power_of_two_scales_exact(m, n, k, dtype, algorithm):
    # tests/cuda/operators/int8_projection.py:25-41
    rng = np.random.default_rng(orc.SEED + m)
    x = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    ws = np.full(n, 0.015625, np.float16)
    ts = np.full(m, 0.0078125, np.float16)
    out = torch.full((m + 1, n), 99.0, dtype=dtype, device=gu.DEV)
    gu.w8_project(gu.dev(x), gu.dev(ts), gu.dev(w), gu.dev(ws), out=out, dtype=dtype, algorithm=algorithm)
    want = orc.project(x, ts, w, ws, np.float32 if dtype == torch.float32 else np.float16)
    got = gu.host(out)
    np.testing.assert_array_equal(got[:m], want)
    assert (got[m] == 99).all()


@pytest.mark.parametrize("m", [1, 3, 17, 63, 65, 129, 511])
def test_w8_dynamic_capacity_stride_extremes(m):
    # int8_projection.py:125-193: capacity 512, N=257, stride 272, forced extremes, ws[0]=0
    rng = np.random.default_rng(orc.SEED + m)
    n, k, stride = 257, 640, 272
    x = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    x[:, :4] = [-128, -1, 0, 127]
    ws = (rng.uniform(size=n) * 0.003).astype(np.float16)
    ts = (rng.uniform(size=m) * 0.005).astype(np.float16)
    ws[0] = 0
    storage = torch.full((m + 2, stride), 99.0, dtype=torch.float16, device=gu.DEV)
    gu.w8_project(gu.dev(x), gu.dev(ts), gu.dev(w), gu.dev(ws), dynamic=True, capacity=512, out=storage, stride=stride)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(x, ts, w, ws))
    assert (got[m:] == 99).all() and (got[:m, n:] == 99).all()


@pytest.mark.parametrize("k", [64, 192, 2752])
@pytest.mark.parametrize("m", [1, 5, 33, 100, 200, 500])
def test_w8_k_ends_in_half_a_step(m, k):
    # int8_projection.py:29 takes any K that is a multiple of 64; the last K step is then half empty.
    # A sentinel row sits right behind the activations and the weights, so a read past K would change the sums.
    rng = np.random.default_rng(orc.SEED + m + k)
    n, stride = 130, 136
    x = rng.integers(-128, 128, (m + 1, k), dtype=np.int8)
    w = rng.integers(-128, 128, (n + 1, k), dtype=np.int8)
    x[m], w[n] = 127, 127
    ws = (rng.uniform(0.2, 1.0, n) * 0.003).astype(np.float16)
    ts = (rng.uniform(0.2, 1.0, m) * 0.005).astype(np.float16)
    storage = torch.full((m + 2, stride), 99.0, dtype=torch.float32, device=gu.DEV)
    gu.w8_project(gu.dev(x)[:m], gu.dev(ts), gu.dev(w)[:n], gu.dev(ws), dynamic=True, capacity=512, out=storage, stride=stride,
                  dtype=torch.float32)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(x[:m], ts, w[:n], ws, np.float32))
    assert (got[m:] == 99).all() and (got[:m, n:] == 99).all()


# Channel runs per CU over the whole K (`algorithm=wide`): one and two row passes, a last pass of one row,
# runs of 2, 97 (two channel passes, the second with one channel) and 100 channels per CU, a K of one step
# and of many, both code layouts, strided fp32 output with sentinels, extremes outside the A8 range.
@pytest.mark.parametrize("packed_k", [0, 128, 64])
@pytest.mark.parametrize("m,n,k", [(33, 300, 384), (64, 24832, 128), (100, 1000, 640), (128, 300, 5120), (129, 515, 256),
                                   (200, 25600, 256), (256, 300, 1024)])
def test_q4_channel_run_kernel(m, n, k, packed_k):
    rng = np.random.default_rng(orc.SEED + m + n + k)
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :4] = [-128, -1, 0, 127]
    a_q[m - 1, -2:] = [127, -128]
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    storage = torch.full((m + 2, n + 3), 91.0, dtype=torch.float32, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 3, dtype=torch.float32,
                  algorithm="wide", packed_k=packed_k)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), scales, np.float32))
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()
    out16 = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), algorithm="wide", packed_k=packed_k)
    np.testing.assert_array_equal(gu.host(out16), orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), scales))


@pytest.mark.parametrize("packed_k", [0, 64, 128])
def test_q4_big_tile_tails_stride_sentinels(packed_k):
    rng = np.random.default_rng(orc.SEED + 9)
    m, n, k = 257 + 130, 300, 384
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :2] = [-128, 127]
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    storage = torch.full((m + 2, n + 5), 91.0, dtype=torch.float32, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 5,
                  dtype=torch.float32, algorithm="mfma", packed_k=packed_k, block_m=256)
    got = gu.host(storage)
    np.testing.assert_array_equal(got[:m, :n], orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), scales, np.float32))
    assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()


@pytest.mark.parametrize("packed_k", [0, 64, 128])
@pytest.mark.parametrize("m,n,k", [(512, 256, 512), (500, 333, 640), (700, 130, 256), (3, 128, 384), (300, 17400, 256)])
def test_q4_tall_tiles_decode_in_the_k_loop(m, n, k, packed_k):
    """512 rows x channel runs with the decode in the K loop (`algorithm=tall`): K of an even and an odd number of
    128-blocks, one and two row tiles, ragged rows and channels, runs of one block and (N = 17400 on 256 CUs) of four
    and five blocks with a ragged last block, every layout, fp16 and fp32 output with a stride and sentinels."""
    rng = np.random.default_rng(orc.SEED + m + n + k + packed_k)
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    a_q[0, :2] = [-128, 127]
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    weights = orc.q4_integers(packed, TABLE)
    for dtype, np_dtype in ((torch.float16, np.float16), (torch.float32, np.float32)):
        storage = torch.full((m + 2, n + 8), 91.0, dtype=dtype, device=gu.DEV)
        gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(scales), out=storage, stride=n + 8, dtype=dtype,
                      algorithm="tall", packed_k=packed_k)
        got = gu.host(storage)
        np.testing.assert_array_equal(got[:m, :n], orc.project(a_q, a_s, weights, scales, np_dtype))
        assert (got[m:] == 91).all() and (got[:m, n:] == 91).all()


def test_q4_tall_tiles_two_rounds_of_units_and_graph_replay():
    """More blocks of 16 channels than five per CU: the units come in two rounds.  One handle, live rows from a trailing
    scalar, replayed from a graph while the weight bits change in place and the row count changes between captures."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n, k = 16 * (5 * cus + 9) + 3, 256
    rng = np.random.default_rng(orc.SEED + 123)
    a_q, a_s, packed, scales = q4_case(rng, 512, n, k)
    other = rng.integers(0, 2**32, packed.shape, dtype=np.uint32)
    kern = gu.lib.Kernel("e8p_q4_projection", M=512, N=n, K=k, dynamic_rows=True, algorithm="tall")
    assert kern.geometry(300)[0] == (2 * cus, 1, 1)
    d_a, d_as, d_s, d_book, d_w = gu.dev(a_q), gu.dev(a_s), gu.dev(scales), gu.book(), gu.dev(packed)
    out = torch.full((512, n), 7.0, dtype=torch.float16, device=gu.DEV)
    side = torch.cuda.Stream()
    for rows in (300, 512):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            with torch.cuda.graph(graph, stream=side):
                kern(stream=side.cuda_stream, A=d_a, AS=d_as, Book=d_book, Out=out, S=d_s, W=d_w, m=rows)
        for bits in (other, packed, other):
            d_w.copy_(gu.dev(bits))
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got = gu.host(out)
            np.testing.assert_array_equal(got[:rows], orc.project(a_q[:rows], a_s[:rows], orc.q4_integers(bits, TABLE), scales))
            assert (got[rows:] == 7).all()


@pytest.mark.parametrize("workspace", [False, True])
def test_q4_auto_takes_channel_runs_from_257_rows_of_a_wide_matrix(workspace):
    """257..512 rows of a matrix with at least 2.25 blocks of 16 channels per CU: `auto` decodes in the K loop of the
    512-row channel runs and leaves the Workspace alone; 256 rows and a narrow matrix keep the other kernels."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n, k = 16 * (9 * cus // 4) + 16 + 8, 256
    rng = np.random.default_rng(orc.SEED + 77 + workspace)
    a_q, a_s, packed, scales = q4_case(rng, 512, n, k)
    weights = orc.q4_integers(packed, TABLE)
    variant = dict(M=512, N=n, K=k, dynamic_rows=True, output_stride=n + 8)
    if workspace:
        variant["workspace"] = True
    kern = gu.lib.Kernel("e8p_q4_projection", **variant)
    by_name = gu.lib.Kernel("e8p_q4_projection", **variant, algorithm="tall")
    narrow = [gu.lib.Kernel("e8p_q4_projection", **dict(variant, N=16 * 2 * cus), **extra) for extra in ({}, {"algorithm": "tall"})]
    scratch = torch.zeros(max(kern.workspace_bytes(0), 16), dtype=torch.uint8, device=gu.DEV) if workspace else None
    assert narrow[0].geometry(257) != narrow[1].geometry(257)      # two blocks per CU: the 128 x 128 tiles
    out = torch.full((513, n + 8), 7.0, dtype=torch.float16, device=gu.DEV)
    for rows in (257, 400, 512, 256):
        same = kern.geometry(rows) == by_name.geometry(rows)
        assert same == (rows > 256)
        if rows > 256:
            assert kern.workspace_bytes(rows) == 0
        out.fill_(7.0)
        args = dict(A=gu.dev(a_q), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=gu.dev(packed), m=rows)
        if workspace:
            args["Workspace"] = scratch
        kern(**args)
        got = gu.host(out)
        np.testing.assert_array_equal(got[:rows, :n], orc.project(a_q[:rows], a_s[:rows], weights, scales))
        assert (got[rows:] == 7).all() and (got[:rows, n:] == 7).all()


@pytest.mark.parametrize("codec", ["w8", "q4"])
def test_a_few_tiles_more_than_cus_go_to_split_tiles(codec):
    """A handful of 256 x 256 tiles beyond one round of the persistent kernel: it takes the column tiles that fill the
    round and the channels behind them run as split 128 x 128 tiles from the same Workspace (behind the decoded weights
    of two-stage codes).  Ragged last tile, output stride, sentinels; rows checked in every row tile."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rows, k = 1000, 256
    row_tiles = -(-rows // 256)
    main_columns = cus // row_tiles
    n = main_columns * 256 + 2 * 256 + 70          # two whole column tiles and a ragged one behind the round
    assert cus < row_tiles * -(-n // 256) <= cus + cus // 8
    rng = np.random.default_rng(orc.SEED + 91)
    scales = rng.uniform(0.005, 0.02, n).astype(np.float16)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_s = rng.uniform(0.005, 0.02, rows).astype(np.float16)
    out = torch.full((rows + 1, n + 5), 7.0, dtype=torch.float16, device=gu.DEV)
    variant = dict(M=rows, N=n, K=k, output_stride=n + 5, workspace=True)
    if codec == "q4":
        packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
        weights = orc.q4_integers(packed, TABLE)
        kern = gu.lib.Kernel("e8p_q4_projection", **variant)
        decoded = n * k
        args = dict(A=gu.dev(a_q), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(scales), W=gu.dev(packed))
    else:
        weights = rng.integers(-128, 128, (n, k), dtype=np.int8)
        kern = gu.lib.Kernel("int8_projection", **variant)
        decoded = 0
        args = dict(A=gu.dev(a_q), Output=out, TokenScale=gu.dev(a_s), Weight=gu.dev(weights), WeightScale=gu.dev(scales))
    assert kern.geometry(rows)[0][0] == row_tiles * main_columns     # the persistent launch: one round
    assert kern.workspace_bytes(rows) > decoded                        # partial tiles of the split launch behind it
    assert gu.lib.Kernel(kern.symbol, **dict(variant, split_k=False)).workspace_bytes(rows) == decoded
    kern(**args)
    got = gu.host(out)
    sample = np.unique(np.concatenate([np.arange(0, rows, 37), [127, 128, 255, 256, 511, 512, 767, 768, rows - 1]]))
    want = orc.project(a_q[sample], a_s[sample], weights, scales)
    np.testing.assert_array_equal(got[sample, :n], want)
    assert (got[rows:] == 7).all() and (got[:rows, n:] == 7).all()
    # every row and channel was written, and column sums agree with the oracle's on the sampled rows' complement check
    assert not (got[:rows, :n] == 7).all(axis=0).any()
    # the whole-tile launch of the same handle family gives the same bits
    whole = torch.full_like(out, 7.0)
    other = gu.lib.Kernel(kern.symbol, **dict(variant, split_k=False))
    other(**dict(args, **({"Out": whole} if codec == "q4" else {"Output": whole})))
    np.testing.assert_array_equal(gu.host(whole), got)
    # a dynamic handle of larger capacity: one Workspace sized for any row count serves this launch and a shorter one
    dynamic = gu.lib.Kernel(kern.symbol, **dict(variant, M=1024, dynamic_rows=True))
    space = torch.empty(dynamic.workspace_bytes(0), dtype=torch.uint8, device=gu.DEV)
    assert dynamic.workspace_bytes(0) >= dynamic.workspace_bytes(rows) == kern.workspace_bytes(rows)
    for live in (rows, 300):
        again = torch.full_like(out, 7.0)
        dynamic(**dict(args, Workspace=space, m=live, **({"Out": again} if codec == "q4" else {"Output": again})))
        result = gu.host(again)
        np.testing.assert_array_equal(result[:live], got[:live])
        assert (result[live:] == 7).all()


@pytest.mark.parametrize("packed_k", [0, 64, 128])
@pytest.mark.parametrize("decode_in_gemm", [False, True], ids=["decode-once", "decode-in-gemm"])
def test_q4_many_rows_both_decode_paths(packed_k, decode_in_gemm):
    """From 512 rows on the two-stage weights are decoded once into the caller's Workspace and the
    int8 kernel runs on them; `decode_in_gemm` keeps the decode inside the GEMM.  Same bits either
    way, also when the weights change between launches of one handle and under graph replay."""
    rng = np.random.default_rng(orc.SEED + 31 + packed_k)
    m, n, k = 700, 333, 640
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    other = rng.integers(0, 2**32, packed.shape, dtype=np.uint32)
    store = (lambda p: p) if packed_k == 0 else (lambda p: orc.q4_pack_k(p, packed_k))
    # split_k=False: so few 256-row tiles would otherwise go to the split 128-row tiles
    variant = dict(M=1024, N=n, K=k, dynamic_rows=True, output_stride=n + 3, split_k=False)
    if packed_k:
        variant["packed_k"] = packed_k
    if decode_in_gemm:
        variant["decode_in_gemm"] = True
    kern = gu.lib.Kernel("e8p_q4_projection", workspace=True, **variant)
    assert kern.workspace_bytes(700) == (0 if decode_in_gemm else n * k) and kern.workspace_bytes(3) == 0
    d_a, d_as, d_s, d_book = gu.dev(a_q), gu.dev(a_s), gu.dev(scales), gu.book()
    d_w = gu.dev(store(packed))
    out = torch.full((1024, n + 3), 7.0, dtype=torch.float16, device=gu.DEV)
    for rows in (700, 512, 511, 3):        # 511 and 3 take the other kernels of the same handle
        out.fill_(7.0)
        kern(A=d_a, AS=d_as, Book=d_book, Out=out, S=d_s, W=d_w, m=rows)
        got = gu.host(out)
        want = orc.project(a_q[:rows], a_s[:rows], orc.q4_integers(packed, TABLE), scales)
        np.testing.assert_array_equal(got[:rows, :n], want)
        assert (got[rows:] == 7).all() and (got[:rows, n:] == 7).all()
    # same handle, new weight bits in the same buffer, replayed from a graph
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            kern(stream=side.cuda_stream, A=d_a, AS=d_as, Book=d_book, Out=out, S=d_s, W=d_w, m=700)
    for bits in (other, packed, other):
        d_w.copy_(gu.dev(store(bits)))
        out.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = orc.project(a_q, a_s, orc.q4_integers(bits, TABLE), scales)
        np.testing.assert_array_equal(gu.host(out)[:700, :n], want)


@pytest.mark.parametrize("m,n,k", [(384, 512, 4096), (1000, 777, 640)])
def test_w8_mid_size_accumulators(m, n, k):
    rng = np.random.default_rng(orc.SEED)
    x = rng.integers(-127, 128, (m, k), dtype=np.int8)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    got = gu.w8_project(gu.dev(x), gu.dev(np.ones(m, np.float16)), gu.dev(w), gu.dev(np.ones(n, np.float16)),
                        dtype=torch.float32)
    acc = orc.int_dot(x, w)
    assert np.abs(acc).max() < 2**24
    np.testing.assert_array_equal(gu.host(got).astype(np.int64), acc.astype(np.int64))


# ---- launch contract -------------------------------------------------------
def test_graph_capture_replays_with_changed_contents():
    # Every reference operator test captures once and replays after mutating inputs in place.
    rng = np.random.default_rng(orc.SEED)
    m, n, k = 3, 129, 512
    a_q, a_s, packed, scales = q4_case(rng, m, n, k)
    ta, ts_, tw, tsc = gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales)
    book = gu.book()
    out = torch.empty((m, n), dtype=torch.float16, device=gu.DEV)
    for algorithm in ("gemv", "mfma"):
        kern = gu.kernel("e8p_q4_projection", M=m, N=n, K=k, algorithm=algorithm)
        args = dict(A=ta, AS=ts_, Book=book, Out=out, S=tsc, W=tw)
        kern(**args)  # warm-up outside capture
        gu.sync()
        stream = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            with torch.cuda.graph(graph, stream=stream):
                kern(stream=stream.cuda_stream, **args)
        w = orc.q4_integers(packed, TABLE)
        for step in range(3):
            out.fill_(float("nan"))
            graph.replay()
            gu.sync()
            np.testing.assert_array_equal(gu.host(out), orc.project(gu.host(ta), gu.host(ts_), w, gu.host(tsc)))
            ta.copy_(gu.dev(rng.integers(-127, 128, (m, k), dtype=np.int8)))  # new contents, same addresses
            tsc.mul_(1.5)
        ta.zero_()
        graph.replay()
        gu.sync()
        assert bool((out == 0).all())  # zero-input replay (backend/cuda/mod.rs:649-678)
        ta.copy_(gu.dev(a_q))
        tsc.copy_(gu.dev(scales))


def test_launch_rejects_bad_geometry_rows_and_alignment():
    from orinfer_amd import lib

    kern = gu.kernel("e8p_q4_projection", M=8, N=128, K=256, dynamic_rows=True)
    a = torch.zeros((8, 256), dtype=torch.int8, device=gu.DEV)
    s = torch.ones(8, dtype=torch.float16, device=gu.DEV)
    w = torch.zeros((128, 32), dtype=torch.int32, device=gu.DEV)
    ws = torch.ones(128, dtype=torch.float16, device=gu.DEV)
    out = torch.zeros((8, 128), dtype=torch.float16, device=gu.DEV)
    values = [a, s, gu.book(), out, ws, w, None, 8]    # 8 rows use no Workspace: a null one is taken
    grid, block, shared = kern.geometry(8)
    stream = torch.cuda.current_stream().cuda_stream
    with pytest.raises(lib.OrxError) as e:
        kern.launch_raw((grid[0] + 1, 1, 1), block, shared, stream, values)
    assert e.value.code == lib.ORX_ERR_BAD_GEOMETRY
    with pytest.raises(lib.OrxError) as e:
        kern.launch_raw(grid, block, shared, stream, values[:-1] + [9])
    assert e.value.code == lib.ORX_ERR_ROWS
    with pytest.raises(lib.OrxError) as e:
        kern.launch_raw(grid, block, shared, stream, [a.data_ptr() + 1] + values[1:])
    assert e.value.code == lib.ORX_ERR_BAD_ARGUMENT
    kern.launch_raw(grid, block, shared, stream, values)
    gu.sync()


# ---- benchmark configurations at full size ---------------------------------
def test_config0_full_size_bit_exact():
    c = workloads.config0()
    x = gu.dev(c["x"])
    a_q, a_s = gu.a8(x)
    wq, ws = orc.a8(c["x"])
    np.testing.assert_array_equal(gu.host(a_q), wq)
    np.testing.assert_array_equal(gu.host(a_s), ws)
    out = gu.q4_project(a_q, a_s, gu.dev(c["packed"]), gu.dev(c["scales"]))
    w = orc.q4_integers(c["packed"], TABLE)
    want = orc.project(wq, ws[:, 0], w, c["scales"])
    assert_close_fp16(gu.host(out), want)
    np.testing.assert_array_equal(gu.host(out), want)


@pytest.mark.parametrize("rows", [1, 8, 32, 128, 512])
def test_config1_full_size_bit_exact(rows):
    c = workloads.config1(rows)
    a_q, a_s = gu.a8(gu.dev(c["x"]))
    wq, ws = orc.a8(c["x"])
    np.testing.assert_array_equal(gu.host(a_q), wq)
    out = gu.q4_project(a_q, a_s, gu.dev(c["packed"]), gu.dev(c["scales"]))
    w = _config1_weights(c)
    want = orc.project(wq, ws[:, 0], w, c["scales"])
    assert_close_fp16(gu.host(out), want)
    np.testing.assert_array_equal(gu.host(out), want)


def test_config1_full_size_512_rows_without_scratch():
    """The same 512 rows through a handle without a Workspace: the same 512-row channel runs with the decode in the K
    loop (one workgroup per CU), K-major codes as the package stores them, against the oracle on every row."""
    c = workloads.config1(512)
    a_q, a_s = gu.a8(gu.dev(c["x"]))
    wq, ws = orc.a8(c["x"])
    stored = orc.q4_pack_k(c["packed"], 128)
    kern = gu.lib.Kernel("e8p_q4_projection", M=512, N=c["n"], K=c["k"], packed_k=128)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert kern.geometry(512)[1] == (512, 1, 1) and kern.geometry(512)[0] == (min(c["n"] // 16, cus), 1, 1)
    out = torch.empty((512, c["n"]), dtype=torch.float16, device=gu.DEV)
    kern(A=a_q, AS=a_s, Book=gu.book(), Out=out, S=gu.dev(c["scales"]), W=gu.dev(stored))
    np.testing.assert_array_equal(gu.host(out), orc.project(wq, ws[:, 0], _config1_weights(c), c["scales"]))


_weights_cache = {}


def _config1_weights(c):
    if "w" not in _weights_cache:
        _weights_cache["w"] = orc.q4_integers(c["packed"], TABLE)
    return _weights_cache["w"]


def test_config2_full_size_sampled_rows_and_linearity():
    c = workloads.config2()
    a_q, a_s = gu.a8(gu.dev(c["x"]))
    out = gu.w8_project(a_q, a_s, gu.dev(c["weight"]), gu.dev(c["scales"]))
    rows = np.random.default_rng(0).choice(c["rows"], 96, replace=False)
    wq, ws = orc.a8(c["x"][rows])
    np.testing.assert_array_equal(gu.host(a_q)[rows], wq)
    want = orc.project(wq, ws[:, 0], c["weight"], c["scales"])
    np.testing.assert_array_equal(gu.host(out)[rows], want)
    # size-independent property on ALL rows: the int32 accumulators are linear in the activations,
    # so acc(a) + acc(-a) == 0 and acc(a) with unit scales summed over N equals a . colsum(W)
    ones_m = torch.ones(c["rows"], dtype=torch.float16, device=gu.DEV)
    ones_n = torch.ones(c["n"], dtype=torch.float16, device=gu.DEV)
    acc = gu.w8_project(a_q, ones_m, gu.dev(c["weight"]), ones_n, dtype=torch.float32)
    neg = gu.w8_project(-a_q, ones_m, gu.dev(c["weight"]), ones_n, dtype=torch.float32)
    assert bool((acc + neg == 0).all())
    colsum = c["weight"].astype(np.int64).sum(0)
    checksum = gu.host(a_q).astype(np.int64) @ colsum
    np.testing.assert_array_equal(gu.host(acc.double().sum(1)).astype(np.int64), checksum)


# ---- configuration 4: one decoder layer's four projections at M = 8192 --------------------------
_config4_cache = {}


def _config4():
    if "c" not in _config4_cache:
        _config4_cache["c"] = workloads.config4()
    return _config4_cache["c"]


@pytest.mark.parametrize("name", [p[0] for p in workloads.LAYER_PROJECTIONS])
def test_config4_full_size_sampled_rows_and_checksums(name):
    """A8 with outlier channels + projection of every linear of the layer at M = 8192: the codes and
    scales of the quantiser and the fp16 output bit-exact on 96 sampled rows x all N (oracle in
    column blocks: the float64 form of the gate/up matrix alone would be 1.4 GB), and on ALL rows
    acc(a) + acc(-a) == 0, row sums == a . colsum(W), column sums == colsum(a) . W."""
    spec = _config4()[name]
    rows_total, n, k = spec["rows"], spec["n"], spec["k"]
    x = gu.dev(spec["x"])
    a_q, a_s = gu.a8(x)
    del x
    rng = np.random.default_rng(4)
    rows = np.sort(rng.choice(rows_total, 96, replace=False))
    rows[0], rows[-1] = 0, rows_total - 1
    wq, ws = orc.a8(spec["x"][rows])
    got_q = gu.host(a_q)
    np.testing.assert_array_equal(got_q[rows], wq)
    np.testing.assert_array_equal(gu.host(a_s)[rows], ws)
    # the outlier channels (x20) are where the row maxima sit: they must be the +-127 codes
    outliers = np.argsort(np.abs(spec["x"][:64].astype(np.float32)).mean(0))[-max(1, k // 1000):]
    assert (np.abs(got_q[rows][:, outliers]).max(1) == 127).all()
    if spec["codec"] == "q4":
        w_int = orc.q4_integers(spec["packed"], TABLE)
        w_dev, s_dev = gu.dev(spec["packed"]), gu.dev(spec["scales"])
        project = lambda a, s_tok, s_w, **kw: gu.q4_project(a, s_tok, w_dev, s_w, **kw)
    else:
        w_int = spec["weight"]
        w_dev, s_dev = gu.dev(spec["weight"]), gu.dev(spec["scales"])
        project = lambda a, s_tok, s_w, **kw: gu.w8_project(a, s_tok, w_dev, s_w, **kw)
    out = project(a_q, a_s, s_dev)
    got = gu.host(out[torch.from_numpy(rows).to(gu.DEV)])
    del out
    for first in range(0, n, 4096):
        want = orc.project(wq, ws[:, 0], w_int[first:first + 4096], spec["scales"][first:first + 4096])
        assert_close_fp16(got[:, first:first + 4096], want)
        np.testing.assert_array_equal(got[:, first:first + 4096], want)
    # size-independent properties over ALL rows, on the int32 accumulators (fp32 output, unit scales)
    ones_m = torch.ones(rows_total, dtype=torch.float16, device=gu.DEV)
    ones_n = torch.ones(n, dtype=torch.float16, device=gu.DEV)
    acc = project(a_q, ones_m, ones_n, dtype=torch.float32)
    assert float(acc.abs().max()) < 2.0 ** 24  # every accumulator is an exact fp32 value
    neg = project(-a_q, ones_m, ones_n, dtype=torch.float32)
    assert bool((acc + neg == 0).all())
    del neg
    row_sums = gu.host(acc.sum(1, dtype=torch.float64)).astype(np.int64)
    col_sums = gu.host(acc.sum(0, dtype=torch.float64)).astype(np.int64)
    del acc
    w_colsum = np.zeros(k, np.int64)
    for first in range(0, n, 4096):
        w_colsum += w_int[first:first + 4096].sum(0, dtype=np.int64)
    np.testing.assert_array_equal(row_sums, got_q.astype(np.int64) @ w_colsum)
    a_colsum = got_q.sum(0, dtype=np.int64).astype(np.float64)
    want_cols = np.concatenate([(w_int[first:first + 4096].astype(np.float64) @ a_colsum)
                                for first in range(0, n, 4096)]).astype(np.int64)
    np.testing.assert_array_equal(col_sums, want_cols)
    torch.cuda.empty_cache()


# ---- scratch is the caller's ---------------------------------------------------------------------
def test_resolving_handles_takes_no_device_memory():
    torch.cuda.synchronize()
    gu.lib.Kernel("int8_projection", M=8, N=128, K=128)  # the library's one-time set-up, if any
    free_before = torch.cuda.mem_get_info()[0]
    handles = [gu.lib.Kernel("e8p_q4_projection", M=4096 + i, N=17408, K=5120, dynamic_rows=True, workspace=True)
               for i in range(1000)]
    handles += [gu.lib.Kernel("int8_swiglu", M=512 + i, N=1024, K=2048, dynamic_rows=True) for i in range(100)]
    assert torch.cuda.mem_get_info()[0] == free_before
    # the decoded int8 weights, and at 1024 rows (272 tiles of 256 for 256 CUs) the partial tiles of the channels that
    # the persistent launch leaves to the split tiles behind them
    assert handles[0].workspace_bytes(4096) == 17408 * 5120
    assert 17408 * 5120 <= handles[0].workspace_bytes(0) <= 17408 * 5120 + 512 * 2 * 128 * 128 * 4


def test_two_handles_on_two_streams_with_their_own_workspaces_stay_bit_exact():
    """Launches of different handles (and of one handle) overlap on distinct streams as long as their
    buffers, the Workspace included, are distinct: split tiles on one stream, decode-once on the other."""
    rng = np.random.default_rng(orc.SEED + 77)
    cases = []
    for m, n, k in ((256, 5120, 1024), (640, 777, 640)):
        a_q, a_s, packed, scales = q4_case(rng, m, n, k)
        kern = gu.lib.Kernel("e8p_q4_projection", M=m, N=n, K=k, workspace=True)
        assert kern.workspace_bytes(m) > 0
        want = orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), scales)
        cases.append((kern, gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(scales), want))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    # two launches of each handle in flight at once: each (handle, stream) pair has its own workspace and output
    outs, spaces = {}, {}
    for c, (kern, a, s, w, ws, want) in enumerate(cases):
        for t in range(2):
            outs[c, t] = torch.zeros(want.shape, dtype=torch.float16, device=gu.DEV)
            spaces[c, t] = torch.empty(kern.workspace_bytes(0), dtype=torch.uint8, device=gu.DEV)
    torch.cuda.synchronize()
    for repeat in range(6):
        for c, (kern, a, s, w, ws, want) in enumerate(cases):
            for t in range(2):
                kern(stream=streams[t].cuda_stream, A=a, AS=s, Book=gu.book(), Out=outs[c, t], S=ws, W=w,
                     Workspace=spaces[c, t])
    torch.cuda.synchronize()
    for c, (kern, a, s, w, ws, want) in enumerate(cases):
        for t in range(2):
            np.testing.assert_array_equal(gu.host(outs[c, t]), want)


@pytest.mark.parametrize("m,k,block_k,swiglu,planes", [(3, 5120, 512, False, False), (1, 17408, 2048, False, False),
                                                       (5, 640, 256, True, False), (4, 1152, 1024, True, True),
                                                       (2, 128, 128, False, False)])
def test_rotation_in_tiles_gives_the_one_launch_codes(m, k, block_k, swiglu, planes):
    # kernels/cuda/model/rotation_a8.py:266-365: rotate_activation_tiles then quantize_rotation_tiles
    rng = np.random.default_rng(orc.SEED + m + k)
    x = (rng.normal(size=(m, 2 * k if swiglu else k)) * rng.uniform(0.2, 3.0, (m, 1))).astype(np.float16)
    signs = rng.choice(np.array([-1, 1], np.int8), k)
    cap = m + 2
    blocks = (k + block_k - 1) // block_k
    plane_rows = cap + 1 if planes else 0
    if planes:  # gate rows, then the up rows as a second plane
        stacked = np.zeros((cap + plane_rows, k), np.float16)
        stacked[:m], stacked[plane_rows:plane_rows + m] = x[:, :k], x[:, k:]
        d_x = gu.dev(stacked)
    else:
        d_x = gu.dev(np.concatenate([x, np.zeros((cap - m, x.shape[1]), np.float16)]))
    rotated = torch.full((cap, k), 9.0, dtype=torch.float16, device=gu.DEV)
    maxima = torch.full((m, blocks), -1.0, dtype=torch.float32, device=gu.DEV)
    variant = dict(M=cap, K=k, block_k=block_k, dynamic_rows=True)
    gu.kernel("rotate_activation_tiles", swiglu=swiglu, plane_rows=plane_rows, **variant)(
        Maxima=maxima, Rotated=rotated, Signs=gu.dev(signs), X=d_x, m=m)
    single = torch.empty((m, k), dtype=torch.float16, device=gu.DEV)
    gu.kernel("rotate_activation", M=m, K=k, swiglu=swiglu)(Signs=gu.dev(signs), X=gu.dev(x), Y=single)
    assert torch.equal(rotated[:m], single) and bool((rotated[m:] == 9).all())
    values = np.abs(gu.host(single).astype(np.float32))
    padded = np.zeros((m, blocks * block_k), np.float32)
    padded[:, :k] = values
    np.testing.assert_array_equal(gu.host(maxima), padded.reshape(m, blocks, block_k).max(axis=2))
    q = torch.full((cap, k), 77, dtype=torch.int8, device=gu.DEV)
    s = torch.full((cap,), 5.0, dtype=torch.float16, device=gu.DEV)
    gu.kernel("quantize_rotation_tiles", **variant)(Maxima=maxima, Q=q, Rotated=rotated, S=s, m=m)
    want_q = torch.empty((m, k), dtype=torch.int8, device=gu.DEV)
    want_s = torch.empty((m,), dtype=torch.float16, device=gu.DEV)
    gu.kernel("rotate_activation_a8", M=m, K=k, swiglu=swiglu)(Q=want_q, S=want_s, Signs=gu.dev(signs), X=gu.dev(x))
    assert torch.equal(q[:m], want_q) and torch.equal(s[:m], want_s)
    assert bool((q[m:] == 77).all()) and bool((s[m:] == 5).all())
    if not swiglu:
        oracle_q, oracle_s = orc.rotate_a8(x, signs)
        np.testing.assert_array_equal(gu.host(q)[:m], oracle_q)
        np.testing.assert_array_equal(gu.host(s)[:m], oracle_s[:, 0])


def test_rotation_tiles_refuse_what_the_reference_refuses():
    for bad in (dict(block_k=384), dict(K=192), dict(plane_rows=8), dict(swiglu=True, plane_rows=2), dict(threads=256),
                dict(registers=True, threads=512, block_k=1024), dict(registers=True, threads=96)):
        with pytest.raises(Exception):
            gu.kernel("rotate_activation_tiles", **{**dict(M=4, K=1024), **bad})
    gu.kernel("rotate_activation_tiles", M=4, K=1024, registers=True, threads=256, block_k=1024)
    with pytest.raises(Exception):
        gu.kernel("quantize_rotation_tiles", M=4, K=1024, block_k=64)


@pytest.mark.parametrize("m,n,k,symbol", [(3, 333, 640, "q4_projection"), (3, 333, 640, "q4_gemv"), (1, 9728, 2560, "q4_gemv"),
                                          (2, 333, 640, "q4_gemv"), (1, 129, 128, "q4_projection"), (2, 5000, 3200, "q4_projection"),
                                          (33, 200, 1024, "q4_projection"), (64, 129, 256, "q4_projection"),
                                          (65, 260, 384, "q4_projection"), (130, 1000, 1280, "q4_projection"),
                                          (700, 300, 512, "q4_projection")])
def test_scalar_q4_projection_at_every_row_range(m, n, k, symbol):
    # kernels/cuda/model/q4_projection.py; the check of python/orinfer_build/quantization/check_e8p_q4.py:195-214
    # (random u16 words, rows in -128..127, unit token scales, fp32 out) plus fp16 with scales, strides and live rows
    rng = np.random.default_rng(orc.SEED + m + n)
    words = rng.integers(0, 65536, (n, k // 4), dtype=np.uint16)
    weights = orc.row_q4_integers(words)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    cap, stride = m + 3, n + 5
    pad = np.concatenate([a, np.zeros((cap - m, k), np.int8)])
    ones = np.ones(cap, np.float16)
    extra = {} if symbol == "q4_gemv" else dict(workspace=True)
    kern = gu.kernel(symbol, M=cap, N=n, K=k, dynamic_rows=True, output_dtype="float32", output_stride=stride, **extra)
    out = torch.full((cap, stride), -7.0, dtype=torch.float32, device=gu.DEV)
    args = dict(A=gu.dev(pad), AS=gu.dev(ones), Out=out, S=gu.dev(ws), W=gu.dev(words), m=m)
    kern(**args)
    got = gu.host(out)
    np.testing.assert_array_equal(got[:m, :n], orc.project(a, ones[:m], weights, ws, np.float32))
    assert (got[m:] == -7).all() and (got[:, n:] == -7).all()
    # unit weight scales: the int32 accumulators themselves
    args["S"] = gu.dev(np.ones(n, np.float16))
    kern(**args)
    np.testing.assert_array_equal(gu.host(out)[:m, :n], (a.astype(np.int64) @ weights.astype(np.int64).T).astype(np.float32))
    scales = rng.uniform(0.01, 0.03, cap).astype(np.float16)
    half = torch.full((cap, n), 9.0, dtype=torch.float16, device=gu.DEV)
    plain = gu.kernel(symbol, M=cap, N=n, K=k, dynamic_rows=True)
    plain(A=gu.dev(pad), AS=gu.dev(scales), Out=half, S=gu.dev(ws), W=gu.dev(words), m=m)
    np.testing.assert_array_equal(gu.host(half)[:m], orc.project(a, scales[:m], weights, ws))
    assert bool((half[m:] == 9).all())


def test_scalar_q4_other_magnitudes_extremes_and_unpack():
    rng = np.random.default_rng(orc.SEED + 77)
    n, k, m = 160, 512, 5
    magnitudes = [1, 2, 5, 9, 33, 64, 100, 127]
    words = rng.integers(0, 65536, (n, k // 4), dtype=np.uint16)
    words[0] = 0xFFFF  # -127 everywhere
    words[1] = 0x7777  # +127 everywhere
    weights = orc.row_q4_integers(words, magnitudes)
    assert (weights[0] == -127).all() and (weights[1] == 127).all()
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    a[0] = -128
    out = torch.empty((m, n), dtype=torch.float32, device=gu.DEV)
    gu.kernel("q4_projection", M=m, N=n, K=k, magnitudes=magnitudes, output_dtype="float32")(
        A=gu.dev(a), AS=gu.dev(np.ones(m, np.float16)), Out=out, S=gu.dev(np.ones(n, np.float16)), W=gu.dev(words))
    np.testing.assert_array_equal(gu.host(out), (a.astype(np.int64) @ weights.astype(np.int64).T).astype(np.float32))
    assert gu.host(out)[0, 0] == 128 * 127 * k
    unpacked = torch.full((n + 1, k), 55, dtype=torch.int8, device=gu.DEV)
    gu.kernel("unpack_q4", N=n, K=k, magnitudes=magnitudes)(Output=unpacked, W=gu.dev(words))
    np.testing.assert_array_equal(gu.host(unpacked)[:n], weights)
    assert bool((unpacked[n] == 55).all())


# ---- channel runs with K split over the waves -------------------------------------------------------------------
# Token blocks of 16 (1 to 8 to a tile, up to four tiles), channel blocks (1 to 5 to a run, partly filled, a short last run),
# fewer K chunks than waves and remainders of the ring.
@pytest.mark.parametrize("rows,n,k", [(1, 16, 128), (2, 40, 256), (16, 1000, 1152), (17, 5120, 384), (33, 4112, 640), (48, 12288, 256),
                                      (63, 20480, 128), (64, 768, 2304), (65, 7168, 384), (96, 2048, 1280), (112, 5136, 256),
                                      (113, 300, 896), (128, 1024, 1152), (131, 2560, 1408), (200, 7168, 256), (257, 1000, 384),
                                      (512, 520, 256)])
@pytest.mark.parametrize("packed_k", [128, 64, 0])
def test_channel_runs_two_stage_codes(rows, n, k, packed_k):
    rng = np.random.default_rng(orc.SEED + rows + n + k)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_q[0, :2] = [-128, 127]
    a_s = rng.uniform(0.005, 0.02, rows).astype(np.float16)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    got = gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(stored), gu.dev(ws), packed_k=packed_k, algorithm="runs")
    np.testing.assert_array_equal(gu.host(got), orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), ws))


@pytest.mark.parametrize("rows,n,k", [(1, 16, 128), (2, 40, 256), (16, 1000, 1152), (17, 5120, 384), (33, 4112, 640), (48, 12288, 256),
                                      (63, 20480, 128), (64, 768, 2304), (65, 7168, 384), (96, 2048, 1280), (112, 5136, 256),
                                      (128, 1024, 1152), (131, 2560, 1408), (200, 7168, 256), (257, 1000, 384), (512, 520, 256)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32-strided"])
def test_channel_runs_int8_weights(rows, n, k, dtype):
    rng = np.random.default_rng(orc.SEED + rows + n + k)
    weight = rng.integers(-128, 128, (n, k), dtype=np.int8)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_s = rng.uniform(0.005, 0.02, rows).astype(np.float16)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    stride = n if dtype == torch.float16 else n + 3
    out = torch.full((rows + 1, stride), 91, dtype=dtype, device=gu.DEV)
    gu.w8_project(gu.dev(a_q), gu.dev(a_s), gu.dev(weight), gu.dev(ws), out=out, rows=rows, stride=stride, dtype=dtype, algorithm="runs")
    want = orc.project(a_q, a_s, weight, ws, out_dtype=np.float16 if dtype == torch.float16 else np.float32)
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], want)
    assert (gu.host(out)[rows] == 91).all() and (gu.host(out)[:, n:] == 91).all()


# Remainders of the ring with one wave to a SIMD (slices of 3, 5 and 7 chunks), all heights of a tile from five blocks on, channels that
# end in the middle of a store, rows of outputs at every alignment of a store.
@pytest.mark.parametrize("rows,n,k", [(72, 5000, 1536), (96, 5000, 2560), (104, 7000, 2688), (112, 5001, 3584), (128, 12000, 1664), (240, 7000, 2560),
                                      (130, 2562, 3456)])
@pytest.mark.parametrize("dtype,pad", [(torch.float16, 1), (torch.float16, 4), (torch.float32, 3)], ids=["fp16-odd", "fp16-8-bytes", "fp32"])
def test_channel_runs_two_stage_codes_remainders_and_strides(rows, n, k, dtype, pad):
    rng = np.random.default_rng(orc.SEED + rows + n + k + pad)
    a_q, a_s, packed, ws = q4_case(rng, rows, n, k)
    a_q[0, :], a_q[1, :] = 127, -128  # the largest sums either way
    stride = n + pad
    out = torch.full((rows + 1, stride), 91, dtype=dtype, device=gu.DEV)
    gu.q4_project(gu.dev(a_q), gu.dev(a_s), gu.dev(packed), gu.dev(ws), out=out, rows=rows, stride=stride, dtype=dtype, algorithm="runs")
    want = orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), ws, out_dtype=np.float16 if dtype == torch.float16 else np.float32)
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], want)
    assert (gu.host(out)[rows] == 91).all() and (gu.host(out)[:, n:] == 91).all()


# Either side of the lines where `auto` changes between the batched-decode kernels, the channel runs and the streaming kernel
@pytest.mark.parametrize("packed_k,n,k", [(128, 1000, 3968), (128, 1000, 4096 + 128), (0, 1000, 3200), (0, 1000, 4224), (64, 1000, 4224), (128, 4112, 3072),
                                          (128, 4112, 4608), (0, 4112, 6144), (128, 8208, 4224), (0, 8208, 6272)])
def test_two_to_32_rows_of_codes_on_either_side_of_a_rule(packed_k, n, k):
    rng = np.random.default_rng(orc.SEED + n + k)
    a_q, a_s, packed, scales = q4_case(rng, 32, n, k)
    a_q[0, :2] = [-128, 127]
    want = orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), scales)
    stored = gu.dev(packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k))
    for rows in (2, 3, 4, 8, 9, 16, 17, 24, 32):
        out = torch.full((33, n), 55, dtype=torch.float16, device=gu.DEV)
        gu.q4_project(gu.dev(a_q), gu.dev(a_s), stored, gu.dev(scales), out=out, rows=rows, dynamic=True, capacity=32, packed_k=packed_k)
        np.testing.assert_array_equal(gu.host(out)[:rows], want[:rows], err_msg=str(rows))
        assert (gu.host(out)[rows:] == 55).all()


@pytest.mark.parametrize("n,k", [(512, 2048), (4112, 3072), (4112, 2944), (8192, 1152), (17400, 256)])
def test_few_int8_rows_on_either_side_of_a_rule(n, k):
    rng = np.random.default_rng(orc.SEED + n + k)
    weight = rng.integers(-128, 128, (n, k), dtype=np.int8)
    a_q = rng.integers(-127, 128, (64, k), dtype=np.int8)
    a_s = rng.uniform(0.005, 0.02, 64).astype(np.float16)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    want = orc.project(a_q, a_s, weight, ws)
    for rows in (1, 2, 3, 16, 17, 33, 64):
        out = torch.full((65, n), 55, dtype=torch.float16, device=gu.DEV)
        gu.w8_project(gu.dev(a_q), gu.dev(a_s), gu.dev(weight), gu.dev(ws), out=out, rows=rows, dynamic=True, capacity=64)
        np.testing.assert_array_equal(gu.host(out)[:rows], want[:rows], err_msg=str(rows))
        assert (gu.host(out)[rows:] == 55).all()


def test_channel_runs_refuse_what_they_do_not_serve():
    for bad in (dict(M=513), dict(K=192)):
        with pytest.raises(gu.lib.OrxError):
            gu.kernel("int8_projection", **{**dict(M=8, N=256, K=256, algorithm="runs"), **bad})


# The last request of a tile (8 rows) or of a run (8 channels) is left out where it would hold no row; a short last tile or run
# beside full ones; rows of fp16 outputs that start at odd elements.
@pytest.mark.parametrize("rows,n", [(1, 5120), (7, 6144), (8, 5120), (9, 6144), (24, 5130), (25, 6400), (40, 2048), (137, 2600)])
@pytest.mark.parametrize("algorithm", ["auto", "runs"])
def test_channel_runs_int8_weights_short_requests(rows, n, algorithm):
    k = 2176  # 17 chunks: two to a wave, three to the last
    rng = np.random.default_rng(orc.SEED + rows * n)
    weight = rng.integers(-128, 128, (n, k), dtype=np.int8)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_s = rng.uniform(0.005, 0.02, rows).astype(np.float16)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    out = torch.full((rows + 1, n + 1), 91, dtype=torch.float16, device=gu.DEV)
    gu.w8_project(gu.dev(a_q), gu.dev(a_s), gu.dev(weight), gu.dev(ws), out=out, rows=rows, stride=n + 1, algorithm=algorithm)
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], orc.project(a_q, a_s, weight, ws))
    assert (gu.host(out)[rows] == 91).all() and (gu.host(out)[:, n] == 91).all()


# Runs of 37, 38 and 19 channels: rows of a run start at every multiple of 2 or 4 bytes, and its last lane holds one to seven channels.
@pytest.mark.parametrize("codec", ["q4", "w8"])
@pytest.mark.parametrize("n", [9472, 9728, 4752, 9701])
@pytest.mark.parametrize("rows,dtype,pad", [(3, torch.float16, 0), (20, torch.float16, 1), (40, torch.float16, 0), (100, torch.float16, 3), (130, torch.float16, 0), (64, torch.float32, 1)])
def test_channel_runs_whose_rows_start_anywhere(codec, n, rows, dtype, pad):
    k = 256
    rng = np.random.default_rng(orc.SEED + n + rows)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_s, ws = rng.uniform(0.005, 0.02, rows).astype(np.float16), rng.uniform(0.005, 0.02, n).astype(np.float16)
    weight = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32) if codec == "q4" else rng.integers(-128, 128, (n, k), dtype=np.int8)
    out = torch.full((rows + 1, n + pad), 91, dtype=dtype, device=gu.DEV)
    variant = dict(M=rows, N=n, K=k, algorithm="runs", workspace=False, output_stride=n + pad, output_dtype="float16" if dtype == torch.float16 else "float32")
    if codec == "q4":
        gu.kernel("e8p_q4_projection", **variant)(A=gu.dev(a_q), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(ws), W=gu.dev(weight))
    else:
        gu.kernel("int8_projection", **variant)(A=gu.dev(a_q), Output=out, TokenScale=gu.dev(a_s), Weight=gu.dev(weight), WeightScale=gu.dev(ws))
    want = orc.project(a_q, a_s, orc.q4_integers(weight, TABLE) if codec == "q4" else weight, ws, out_dtype=np.float16 if dtype == torch.float16 else np.float32)
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], want)
    assert (gu.host(out)[rows] == 91).all() and (gu.host(out)[:, n:] == 91).all()


# Row counts at which `auto` hands a projection to the channel runs: handles with a Workspace and without, both codecs, either side
# of a row tile, one and two rounds of the CUs.
@pytest.mark.parametrize("rows,n,k", [(17, 1040, 5120), (80, 8208, 1152), (81, 8208, 1152), (129, 8208, 1152), (200, 8208, 1152), (201, 8208, 1152),
                                      (240, 4096, 1152), (256, 4096, 1152), (257, 1040, 1024), (512, 1040, 1152)])
def test_auto_rows_around_the_channel_runs(rows, n, k):
    rng = np.random.default_rng(orc.SEED + 3 * rows + n)
    packed = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    weight = rng.integers(-128, 128, (n, k), dtype=np.int8)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_s = rng.uniform(0.005, 0.02, rows).astype(np.float16)
    ws = rng.uniform(0.005, 0.02, n).astype(np.float16)
    want4 = orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), ws)
    want8 = orc.project(a_q, a_s, weight, ws)
    for scratch in (False, True):
        variant = dict(M=rows, N=n, K=k, dynamic_rows=True, workspace=scratch)
        q4, w8 = gu.lib.Kernel("e8p_q4_projection", **variant), gu.lib.Kernel("int8_projection", **variant)
        out = torch.full((rows, n), 9.0, dtype=torch.float16, device=gu.DEV)
        extra = {"Workspace": q4.workspace()} if scratch else {}
        q4(A=gu.dev(a_q), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(ws), W=gu.dev(packed), m=rows, **extra)
        np.testing.assert_array_equal(gu.host(out), want4)
        out.fill_(9.0)
        extra = {"Workspace": w8.workspace()} if scratch else {}
        w8(A=gu.dev(a_q), Output=out, TokenScale=gu.dev(a_s), Weight=gu.dev(weight), WeightScale=gu.dev(ws), m=rows, **extra)
        np.testing.assert_array_equal(gu.host(out), want8)


# ---- token panels -----------------------------------------------------------------------------------------------------
# Every number of waves and pieces the quantiser has, a panel that is not full, several rounds of panels over the XCDs, and rows whose
# address leaves no 16-byte loads.
@pytest.mark.parametrize("rows,k,shift", [(1, 128, 0), (16, 256, 0), (37, 512, 1), (130, 1280, 0), (129, 2048, 0), (2049, 2048, 0), (2100, 384, 1), (600, 5120, 0),
                                          (200, 8192, 1), (17, 17408, 0), (3, 32768, 0)])
def test_a8_panels(rows, k, shift):
    rng = np.random.default_rng(orc.SEED + rows + k)
    x = torch.empty(rows * k + 8, dtype=torch.float16, device=gu.DEV)
    x16 = x[shift:shift + rows * k].view(rows, k)
    x16.copy_(gu.dev(rng.normal(0, 1, (rows, k)).astype(np.float16)))
    x16[0] = 0
    padded = (rows + 15) // 16 * 16
    panels = torch.full((padded + 1, k), 91, dtype=torch.int8, device=gu.DEV)
    q = torch.empty((rows, k), dtype=torch.int8, device=gu.DEV)
    s = torch.empty((rows, 1), dtype=torch.float16, device=gu.DEV)
    sums = torch.full((rows + 1,), 91, dtype=torch.int32, device=gu.DEV)
    gu.kernel("activation_quantization", K=k, panels=True)(Mask=None, Panels=panels, Q=q, S=s, Sums=sums, X=x16, rows=rows)
    want_q, want_s = gu.a8(x16)
    assert torch.equal(q, want_q) and torch.equal(s.view(-1), want_s.view(-1))
    assert torch.equal(sums[:rows].long(), q.long().sum(1)) and int(sums[rows]) == 91
    rest = torch.full((padded, k), 91, dtype=torch.int8, device=gu.DEV)
    rest[:rows] = q
    # block of 16 rows, chunk of 128, half, quarter, row, 16 bytes: the bytes [32 quarter + 16 half, +16) of a chunk
    order = rest.view(padded // 16, 16, k // 128, 4, 2, 16).permute(0, 2, 4, 3, 1, 5).reshape(padded, k)
    assert torch.equal(panels[:padded], order) and bool((panels[padded] == 91).all())


# One to five channel blocks to a workgroup (the last ones short), two to four row blocks to a wave with rows missing, one to three row
# tiles, phases that end early (1 to 8 chunks), and the largest sums either way.
@pytest.mark.parametrize("rows,n,k", [(1, 16, 256), (17, 24, 384), (129, 4099, 1152), (255, 5000, 896), (257, 8200, 1280), (256, 12290, 640), (300, 9728, 384), (384, 17408, 256),
                                      (385, 20480, 768), (512, 20600, 256), (513, 300, 1024), (1030, 1000, 640), (449, 16000, 512)])
@pytest.mark.parametrize("packed_k", [128, 64, 0])
def test_q4_over_panels(rows, n, k, packed_k):
    rng = np.random.default_rng(orc.SEED + rows + n + k)
    a_q, a_s, packed, ws = q4_case(rng, rows, n, k)
    a_q[0, :], a_q[-1, :] = 127, -128
    out = torch.full((rows + 1, n), 91, dtype=torch.float16, device=gu.DEV)
    project_over_panels(a_q, a_s, packed, ws, packed_k, out)
    np.testing.assert_array_equal(gu.host(out)[:rows], orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), ws))
    assert (gu.host(out)[rows] == 91).all()


@pytest.mark.parametrize("rows,n,k", [(1, 16, 256), (17, 24, 384), (100, 4099, 1152), (255, 5000, 896), (257, 8200, 1280), (256, 12290, 640), (300, 9728, 384), (384, 17408, 256),
                                      (385, 20480, 768), (512, 20600, 256), (513, 300, 1024), (1030, 1000, 640), (449, 16000, 512)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32-strided"])
def test_w8_over_panels(rows, n, k, dtype):
    rng = np.random.default_rng(orc.SEED + rows + n + k)
    weight = rng.integers(-128, 128, (n, k), dtype=np.int8)
    a_q = rng.integers(-127, 128, (rows, k), dtype=np.int8)
    a_q[0, :], a_q[-1, :], weight[-1, :] = 127, -128, -128
    a_s, ws = rng.uniform(0.005, 0.02, rows).astype(np.float16), rng.uniform(0.005, 0.02, n).astype(np.float16)
    stride = n if dtype == torch.float16 else n + 3
    out = torch.full((rows + 1, stride), 91, dtype=dtype, device=gu.DEV)
    gu.kernel("int8_projection", M=rows, N=n, K=k, panels=True, workspace=False, output_stride=stride, output_dtype="float16" if dtype == torch.float16 else "float32")(
        A=gu.dev(in_panels(a_q)), Output=out, TokenScale=gu.dev(a_s), Weight=gu.dev(weight), WeightScale=gu.dev(ws))
    want = orc.project(a_q, a_s, weight, ws, out_dtype=np.float16 if dtype == torch.float16 else np.float32)
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], want)
    assert (gu.host(out)[rows] == 91).all() and (gu.host(out)[:, n:] == 91).all()


def in_panels(a_q):
    rows, k = a_q.shape
    padded = np.zeros(((rows + 15) // 16 * 16, k), np.int8)
    padded[:rows] = a_q
    return np.ascontiguousarray(padded.reshape(-1, 16, k // 128, 4, 2, 16).transpose(0, 2, 4, 3, 1, 5))


def project_over_panels(a_q, a_s, packed, ws, packed_k, out, **variant):
    rows, k = a_q.shape
    panels = in_panels(a_q)
    stored = packed if packed_k == 0 else orc.q4_pack_k(packed, packed_k)
    gu.kernel("e8p_q4_projection", M=rows, N=len(ws), K=k, packed_k=packed_k, panels=True, workspace=False, **variant)(
        A=gu.dev(panels), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(ws), Sums=gu.dev(a_q.astype(np.int32).sum(1).astype(np.int32)), W=gu.dev(stored))


@pytest.mark.parametrize("dtype,pad", [(torch.float16, 1), (torch.float16, 4), (torch.float32, 3)], ids=["fp16-odd", "fp16-8-bytes", "fp32"])
def test_q4_over_panels_strides(dtype, pad):
    rows, n, k = 150, 9005, 512
    a_q, a_s, packed, ws = q4_case(np.random.default_rng(orc.SEED), rows, n, k)
    out = torch.full((rows + 1, n + pad), 91, dtype=dtype, device=gu.DEV)
    project_over_panels(a_q, a_s, packed, ws, 0, out, output_stride=n + pad, output_dtype="float16" if dtype == torch.float16 else "float32")
    want = orc.project(a_q, a_s, orc.q4_integers(packed, TABLE), ws, out_dtype=np.float16 if dtype == torch.float16 else np.float32)
    np.testing.assert_array_equal(gu.host(out)[:rows, :n], want)
    assert (gu.host(out)[rows] == 91).all() and (gu.host(out)[:, n:] == 91).all()


@pytest.mark.parametrize("codec", ["q4", "w8"])
def test_a_linear_over_panels_gives_the_bits_of_the_row_major_one(codec):
    """Rows either side of the lines, one state; the codes and scales that `run` leaves are the quantiser's; and from a graph."""
    rng = np.random.default_rng(orc.SEED)
    n, k = 9728, 512
    weight = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32) if codec == "q4" else rng.integers(-127, 128, (n, k), dtype=np.int8)
    linear = programs.QuantizedLinear(codec, weight, rng.uniform(0.005, 0.02, n).astype(np.float16), 1300, packed_k=128 if codec == "q4" else 0)
    taken = [r for r, over in enumerate(linear.over_panels) if over]
    assert taken and taken[0] > 64 and len(linear.over_panels) == programs.PANEL_ROWS + 1
    for rows in (taken[0] - 1, taken[0], 512, 700, 768, 1025):
        x = gu.dev(rng.normal(0, 1, (rows, k)).astype(np.float16))
        got = linear.run(x).clone()
        codes, scales = linear.a_q[:rows].clone(), linear.a_s[:rows].clone()
        want = linear.project(linear.quantize(x))
        assert torch.equal(got, want) and torch.equal(codes, linear.a_q[:rows]) and torch.equal(scales, linear.a_s[:rows]), rows
    x = gu.dev(rng.normal(0, 1, (512, k)).astype(np.float16))
    want, stream = linear.run(x).clone(), torch.cuda.Stream()
    gu.sync()
    with torch.cuda.stream(stream):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = linear.run(x)
    for _ in range(3):
        linear.out.zero_()
        gu.sync()
        graph.replay()
        gu.sync()
        assert torch.equal(got, want)


# Every form of the panel kernel (blocks of channels to a workgroup, of rows to a wave, rows that leave waves a block short) through its steady state: four phases,
# the last one short, so that codes requested inside the loop are multiplied and both weight buffers are written again after they were.  Sums by 64-bit products, exact.
@pytest.mark.parametrize("codec", ["q4", "w8"])
@pytest.mark.parametrize("blocks,n,k", [(1, 1000, 3456), (2, 5000, 3456), (3, 8200, 1920), (4, 12290, 1920), (5, 16400, 1920)])
def test_panel_forms_through_many_phases(blocks, n, k, codec):
    rng = np.random.default_rng(orc.SEED + n)
    a_q = rng.integers(-127, 128, (512, k), dtype=np.int8)
    a_s, ws = rng.uniform(0.005, 0.02, 512).astype(np.float16), rng.uniform(0.005, 0.02, n).astype(np.float16)
    weight = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32) if codec == "q4" else rng.integers(-128, 128, (n, k), dtype=np.int8)
    integers = orc.q4_integers(weight, TABLE) if codec == "q4" else weight
    acc = gu.host(gu.dev(a_q).double() @ gu.dev(integers).double().T).astype(np.int32)
    symbol, stored = ("e8p_q4_projection", gu.dev(weight)) if codec == "q4" else ("int8_projection", gu.dev(weight))
    for rows in (200, 256, 300, 384, 450, 512):
        kernel = gu.kernel(symbol, M=rows, N=n, K=k, panels=True, workspace=False)
        units = kernel.geometry(rows)[0][0]
        assert -(-(-(-n // 16)) // units) == blocks or torch.cuda.get_device_properties(0).multi_processor_count != 256
        out = torch.full((rows + 1, n), 91, dtype=torch.float16, device=gu.DEV)
        if codec == "q4":
            kernel(A=gu.dev(in_panels(a_q[:rows])), AS=gu.dev(a_s), Book=gu.book(), Out=out, S=gu.dev(ws),
                   Sums=gu.dev(a_q[:rows].astype(np.int32).sum(1).astype(np.int32)), W=stored)
        else:
            kernel(A=gu.dev(in_panels(a_q[:rows])), Output=out, TokenScale=gu.dev(a_s), Weight=stored, WeightScale=gu.dev(ws))
        np.testing.assert_array_equal(gu.host(out)[:rows], orc.rescale(acc[:rows], ws, a_s[:rows], np.float16), err_msg=f"{rows} rows")
        assert (gu.host(out)[rows] == 91).all()


@pytest.mark.parametrize("codec, packed_k", [("q4", 0), ("q4", 128), ("w8", 0)])
def test_a_linear_over_panels_of_a_long_k(codec, packed_k):
    rng = np.random.default_rng(orc.SEED + 1)
    n, k = 7168, 5120
    weight = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32) if codec == "q4" else rng.integers(-127, 128, (n, k), dtype=np.int8)
    linear = programs.QuantizedLinear(codec, weight, rng.uniform(0.005, 0.02, n).astype(np.float16), 512, packed_k=packed_k)
    for rows in (200, 256, 333, 512):
        assert linear.over_panels[rows] or torch.cuda.get_device_properties(0).multi_processor_count != 256
        x = gu.dev(rng.normal(0, 1, (rows, k)).astype(np.float16))
        got = linear.run(x).clone()
        assert torch.equal(got, linear.project(linear.quantize(x))), rows


def test_panels_are_refused_where_no_kernel_serves_them():
    for symbol, variant in (("activation_quantization", dict(K=1000, panels=True)), ("activation_quantization", dict(K=256, group_size=128, panels=True)),
                            ("activation_quantization", dict(K=256, fused=True, panels=True)), ("activation_quantization", dict(K=32896, panels=True)),
                            ("e8p_q4_projection", dict(M=512, N=256, K=128, panels=True)), ("e8p_q4_projection", dict(M=2049, N=256, K=256, panels=True)),
                            ("e8p_q4_projection", dict(M=64, N=256, K=256, panels=True, algorithm="runs")),
                            ("e8p_q4_projection", dict(M=64, N=256, K=256, panels=True, workspace=True)),
                            ("int8_projection", dict(M=64, N=256, K=320, panels=True)), ("int8_projection", dict(M=64, N=256, K=256, panels=True, block_m=64))):
        with pytest.raises(gu.lib.OrxError):
            gu.lib.Kernel(symbol, **variant)
