"""Projections of 2 and more rows on split activations (linear_mm_*): every kernel
of them (128-token tiles of 256 and 128 rows, 64-token ones of 128, 32-token k-split
blocks of 64 and 32 rows, 16-token blocks of 32 and 16; every weight format and
epilogue) at ragged edges of its tiles and steps (EVERY_KERNEL, whose routes
tests/test_linear_routes_host.py asserts without a GPU), the int8 kernel over pairs
of rows of a large weight, against the CPU oracle within the bound of another f32
summation order (2e-6 * sum |x w| + 1e-7 per output, as tests/test_linear_gpu.py
derives it); activations far apart in scale within a row, whose segments scale apart,
and beside outliers; rows holding an inf or NaN; and a capture on a context whose
workspace is too small for the split, which runs the kernel that needs none."""
import numpy as np
import pytest

import g4a
import g4a.synth as synth
import oracle
from test_linear_gpu import Dev, _bound, _check_fused, _check_sum, _qw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op,N,K,M,bits,signed", [
    ("linear", 33, 320, 16, 4, False),       # k-split, fewer steps than waves, a ragged 32-row block
    ("linear", 2050, 576, 33, 2, False),     # a segment of one step, N not a multiple of 4
    ("linear", 700, 1536, 97, 8, True),
    ("linear", 700, 1536, 97, 8, False),
    ("gelu_cols", 95, 1600, 40, 4, False),
    ("geglu", 100, 448, 65, 4, False),
    ("geglu", 130, 1536, 31, 2, False),
    ("linear", 4100, 320, 1030, 4, False),   # tiles, the last of each ragged
    ("geglu", 3100, 320, 700, 2, False),
    ("geglu", 1050, 320, 900, 8, True),
    ("gelu_cols", 4099, 320, 600, 4, False),
    ("linear", 2050, 1024, 990, 4, False),   # 64-token tiles
    ("geglu", 3000, 832, 300, 8, True),
    ("linear", 33, 64, 2, 4, False),         # 2 .. 16 rows: x split in registers, fewer steps than waves
    ("linear", 2050, 1600, 16, 2, False),
    ("linear", 100, 1536, 7, 8, True),       # 16 waves, some with one step more; at 1024 and 2048 one and two each
    ("linear", 33, 1024, 16, 4, False),
    ("linear", 4090, 2048, 2, 2, False),
    ("linear", 50, 960, 5, 4, False),        # below and above their range
    ("linear", 50, 2112, 5, 4, False),
    ("linear", 17, 6144, 15, 8, False),
    ("geglu", 100, 448, 3, 4, False),
    ("geglu", 8200, 576, 13, 2, False),
    ("geglu", 45, 1600, 5, 8, True),
    ("gelu_cols", 95, 1600, 12, 4, False),
    ("linear", 16400, 320, 9, 4, False),
    ("linear", 16400, 320, 3, 2, False),
])
def test_forms_match_the_oracle(ctx, op, N, K, M, bits, signed):
    name = f"{op} N={N} K={K} M={M} b{bits}{'s' if signed else ''}"
    print(f"[gpu] {name}", flush=True)
    w, x = _qw(1, N, K, bits, signed, None), synth.normal_f32(2, 1, M * K).reshape(M, K)
    with Dev(ctx) as d:
        dw, dx, y = d.w(w), d.arr(x), d.empty((M, N))
        if op == "linear":
            ctx.linear_q(dw, dx.ptr, y.ptr, M)
            _check_sum(y.to_host(), oracle.linear_q(x, w), _bound(x, w), name)
        elif op == "geglu":
            w2 = _qw(3, N, K, bits, signed, None)
            ctx.linear_q_geglu(dw, d.w(w2), dx.ptr, y.ptr, M)
            _check_fused(y.to_host(), x, w, w2, None, 0, name)
        else:
            b = synth.normal_f32(4, 2, M * (N + 5)).reshape(M, N + 5)
            ctx.linear_q_gelu_mul_cols(dw, dx.ptr, d.arr(b).ptr, N + 5, 3, y.ptr, M)
            _check_fused(y.to_host(), x, w, None, b, 3, name)


# kernel, entry point, N, K, M, bits: no multiple of a tile or of a scale's segment
EVERY_KERNEL = [
    ("0_b2_mode0", "linear", 2946, 1728, 1392, 2),
    ("0_b2_mode1", "geglu", 1635, 320, 1933, 2),
    ("0_b2_mode2", "gelu_cols", 2575, 320, 2382, 2),
    ("0_b4_mode0", "linear", 1175, 384, 4918, 4),
    ("0_b4_mode1", "geglu", 1594, 320, 2087, 4),
    ("0_b4_mode2", "gelu_cols", 3545, 320, 1752, 4),
    ("0_b8_mode0", "linear", 2598, 832, 1752, 8),
    ("0_b8_mode1", "geglu", 1261, 832, 1610, 8),
    ("0_b8_mode2", "gelu_cols", 3207, 1088, 1228, 8),
    ("1_b2_mode0", "linear", 2931, 1152, 2727, 2),
    ("1_b2_mode1", "geglu", 2461, 896, 1544, 2),
    ("1_b2_mode2", "gelu_cols", 1915, 640, 4207, 2),
    ("1_b4_mode0", "linear", 1822, 640, 4178, 4),
    ("1_b4_mode1", "geglu", 1251, 640, 4347, 4),
    ("1_b4_mode2", "gelu_cols", 3103, 704, 3542, 4),
    ("2_b2_mode0", "linear", 607, 1088, 453, 2),
    ("2_b2_mode1", "geglu", 519, 320, 1456, 2),
    ("2_b2_mode2", "gelu_cols", 357, 1088, 712, 2),
    ("2_b4_mode0", "linear", 391, 1152, 617, 4),
    ("2_b4_mode1", "geglu", 555, 320, 1384, 4),
    ("2_b4_mode2", "gelu_cols", 302, 1088, 870, 4),
    ("2_b8_mode0", "linear", 547, 640, 1377, 8),
    ("2_b8_mode2", "gelu_cols", 939, 640, 903, 8),
    ("3_b2_mode0", "linear", 27, 384, 17, 2),
    ("3_b2_mode1", "geglu", 22, 320, 24, 2),
    ("3_b2_mode2", "gelu_cols", 27, 320, 17, 2),
    ("3_b4_mode0", "linear", 25, 320, 17, 4),
    ("3_b4_mode1", "geglu", 23, 320, 18, 4),
    ("3_b4_mode2", "gelu_cols", 22, 448, 17, 4),
    ("3_b8_mode0", "linear", 26, 320, 18, 8),
    ("3_b8_mode1", "geglu", 25, 320, 21, 8),
    ("3_b8_mode2", "gelu_cols", 23, 320, 18, 8),
    ("4_b2_mode0", "linear", 839, 320, 1862, 2),
    ("4_b2_mode1", "geglu", 525, 320, 2089, 2),
    ("4_b2_mode2", "gelu_cols", 2386, 320, 645, 2),
    ("4_b4_mode0", "linear", 1237, 320, 1328, 4),
    ("4_b4_mode1", "geglu", 551, 320, 1963, 4),
    ("4_b4_mode2", "gelu_cols", 1477, 320, 1196, 4),
    ("4_b8_mode0", "linear", 1011, 320, 1079, 8),
    ("4_b8_mode1", "geglu", 389, 320, 2014, 8),
    ("4_b8_mode2", "gelu_cols", 2246, 320, 466, 8),
    ("few_r1_b2_mode0", "linear", 21, 64, 2, 2),
    ("few_r1_b2_mode1", "geglu", 8585, 64, 2, 2),
    ("few_r1_b2_mode2", "gelu_cols", 22, 64, 4, 2),
    ("few_r1_b4_mode0", "linear", 21, 64, 3, 4),
    ("few_r1_b4_mode1", "geglu", 8302, 64, 2, 4),
    ("few_r1_b4_mode2", "gelu_cols", 25, 64, 2, 4),
    ("few_r1_b8_mode0", "linear", 22, 64, 2, 8),
    ("few_r1_b8_mode1", "geglu", 8810, 64, 3, 8),
    ("few_r1_b8_mode2", "gelu_cols", 21, 64, 2, 8),
    ("few_r2_b2_mode0", "linear", 16861, 64, 5, 2),
    ("few_r2_b2_mode1", "geglu", 23, 64, 4, 2),
    ("few_r2_b2_mode2", "gelu_cols", 17467, 64, 5, 2),
    ("few_r2_b4_mode0", "linear", 16514, 64, 7, 4),
    ("few_r2_b4_mode1", "geglu", 21, 64, 2, 4),
    ("few_r2_b4_mode2", "gelu_cols", 16431, 64, 6, 4),
    ("few_r2_b8_mode0", "linear", 17027, 64, 5, 8),
    ("few_r2_b8_mode1", "geglu", 21, 64, 3, 8),
    ("few_r2_b8_mode2", "gelu_cols", 19687, 64, 5, 8),
    ("few_w16_b2_mode0", "linear", 21, 1088, 3, 2),
    ("few_w16_b4_mode0", "linear", 21, 1152, 2, 4),
    ("few_w16_b8_mode0", "linear", 21, 1088, 2, 8),
]


def _ends(n, count, seed):
    """Indices at both ends of n and some between."""
    if n <= 3 * count:
        return np.arange(n)
    mid = np.random.default_rng(seed).choice(np.arange(count, n - count), count, replace=False)
    return np.sort(np.r_[0:count, n - count:n, mid])


@pytest.mark.parametrize("kernel,op,N,K,M,bits", EVERY_KERNEL)
def test_every_kernel_matches_the_oracle(ctx, kernel, op, N, K, M, bits):
    print(f"[gpu] {kernel} {op} N={N} K={K} M={M}", flush=True)
    signed = bits == 8 and N % 2 == 1  # 8-bit rows of both kinds
    rows, toks = _ends(N, 150, 1), _ends(M, 70, 2)
    w, x = _qw(1, N, K, bits, signed, None), synth.normal_f32(2, 1, M * K).reshape(M, K)
    xt = np.ascontiguousarray(x[toks])

    def part(w):
        qb = np.ascontiguousarray(np.asarray(w.qbytes, np.uint8).reshape(N, -1)[rows])
        return oracle.QWeight(qb, w.scales.reshape(N, -1)[rows], rows.size, K, bits, signed, K)

    with Dev(ctx) as d:
        dw, dx, y = d.w(w), d.arr(x), d.empty((M, N))
        if op == "linear":
            ctx.linear_q(dw, dx.ptr, y.ptr, M)
            _check_sum(y.to_host()[np.ix_(toks, rows)], oracle.linear_q(xt, part(w)), _bound(xt, part(w)), kernel)
        elif op == "geglu":
            w2 = _qw(3, N, K, bits, signed, None)
            ctx.linear_q_geglu(dw, d.w(w2), dx.ptr, y.ptr, M)
            _check_fused(y.to_host()[np.ix_(toks, rows)], xt, part(w), part(w2), None, 0, kernel)
        else:
            b = synth.normal_f32(4, 2, M * (N + 5)).reshape(M, N + 5)
            ctx.linear_q_gelu_mul_cols(dw, dx.ptr, d.arr(b).ptr, N + 5, 3, y.ptr, M)
            _check_fused(y.to_host()[np.ix_(toks, rows)], xt, part(w), None, np.ascontiguousarray(b[np.ix_(toks, rows + 3)]),
                         0, kernel)


@pytest.mark.parametrize("bits,signed", [(4, False), (8, True), (2, False)])
def test_weights_at_eight_byte_alignment(ctx, bits, signed):
    # 8 bytes past a 16-byte boundary: the tiles' 16-byte weight copies do not run
    N, K, M = 4096, 320, 700
    w, x = _qw(9, N, K, bits, signed, None), synth.normal_f32(10, 1, M * K).reshape(M, K)
    print(f"[gpu] b{bits}", flush=True)
    raw = ctx.upload(np.concatenate([np.zeros(8, np.uint8), np.ascontiguousarray(w.qbytes, np.uint8).ravel()]))
    with Dev(ctx) as d:
        dw, y = d.w(w), d.empty((M, N))
        args = g4a.QWeightArgs(raw.ptr + 8, dw.args.scales, N, K, bits, int(signed), K)
        ctx.linear_q(g4a.DeviceQWeight(args, None, None), d.arr(x).ptr, y.ptr, M)
        _check_sum(y.to_host(), oracle.linear_q(x, w), _bound(x, w), f"b{bits}")
    raw.free()


@pytest.mark.parametrize("M", [9, 20, 400])
def test_scales_apart_and_non_finite_rows(ctx, M):
    N, K = 2048, 1024
    w, x = _qw(5, N, K, 4, False, None), synth.normal_f32(6, 1, M * K).reshape(M, K).copy()
    x[0, :256] *= np.float32(1e30)
    x[1, 256:512] *= np.float32(1e-30)
    x[2] *= np.float32(1e-38)
    x[3, ::2] *= np.float32(2.0 ** -20)
    x[4] = 0.0
    x[5, 700] = np.inf
    x[6, 3] = np.nan
    print(f"[gpu] M={M}", flush=True)
    fine = [m for m in range(M) if m not in (5, 6)]
    with Dev(ctx) as d:
        y = d.empty((M, N))
        ctx.linear_q(d.w(w), d.arr(x).ptr, y.ptr, M)
        got = y.to_host()
    # the bound's absolute part is for rows of about unit values: compare per row in units of its largest
    unit = np.maximum(np.abs(x[fine]).max(1, keepdims=True), np.float32(1e-45)).astype(np.float64)
    want = oracle.linear_q(x[fine], w)
    assert np.all(np.abs(got[fine].astype(np.float64) - want) <= 2e-6 * _bound(x[fine], w) + 1e-7 * unit)
    assert not got[4].any()
    assert not np.isfinite(got[5]).any() and np.isnan(got[6]).all()
    # the infinity of its weight's sign (NaN at a weight of 0), as f32 products give it
    assert np.array_equal(got[5], oracle.linear_q(x[5:6], w)[0], equal_nan=True)


def _beside_outliers(power, N, K, M, bits, signed):
    """Normal activations, one of 2^power in every 64, and weights that are 0 there."""
    qb, sc, g = synth.quant_weight(13, N, K, bits, signed_i8=signed, group_size=None)
    qb = np.array(qb, np.uint8).reshape(N, -1)
    x = synth.normal_f32(14, 1, M * K).reshape(M, K).copy()
    per = 8 // bits
    for k in range(5, K, 64):
        shift = bits * (k % per)
        zero = 0 if signed else (1 << (bits - 1)) << shift
        qb[:, k // per] = (qb[:, k // per] & (0xFF ^ (((1 << bits) - 1) << shift))) | zero
        x[:, k] = np.float32(2.0 ** power)
    return oracle.QWeight(qb, sc, N, K, bits, signed, g), x


@pytest.mark.parametrize("bits,signed", [(4, False), (2, False), (8, True)])
@pytest.mark.parametrize("M", [9, 20, 400])
def test_activations_beside_outliers_keep_their_bits(ctx, M, bits, signed):
    # one |x| of 2^26 times the others in every 64 k, where every weight is 0: the outputs are
    # sums of the others, held to the bound of f32 sums of those alone
    w, x = _beside_outliers(26, 2048, 1024, M, bits, signed)
    print(f"[gpu] M={M} b{bits}", flush=True)
    with Dev(ctx) as d:
        y = d.empty((M, 2048))
        ctx.linear_q(d.w(w), d.arr(x).ptr, y.ptr, M)
        _check_sum(y.to_host(), oracle.linear_q(x, w), _bound(x, w), f"M={M} b{bits}")


@pytest.mark.parametrize("M", [9, 20, 400])
def test_activations_far_below_an_outlier_keep_2_to_the_minus_50_of_it(ctx, M):
    # 2^36 times the others: each is held to 2^-50 of that, 2^-14, so an output misses the f32
    # bound by at most 2^-14 * sum |w|
    w, x = _beside_outliers(36, 2048, 1024, M, 4, False)
    print(f"[gpu] M={M}", flush=True)
    with Dev(ctx) as d:
        y = d.empty((M, 2048))
        ctx.linear_q(d.w(w), d.arr(x).ptr, y.ptr, M)
        got = y.to_host().astype(np.float64)
    rounding = 2.0 ** -14 * _bound(np.ones((1, 1024), np.float32), w)
    err = np.abs(got - oracle.linear_q(x, w))
    print(f"  worst err / bound {(err / (2e-6 * _bound(x, w) + 1e-7 + rounding)).max():.3f}", flush=True)
    assert np.all(err <= 2e-6 * _bound(x, w) + 1e-7 + rounding)


@pytest.mark.parametrize("M", [3, 8, 9])
def test_rows_of_a_large_weight(ctx, M):
    # 64 MiB and more of packed weights: pairs of rows on the int8 matrix cores up to 8 rows
    N, K = 131077, 2048
    w, x = _qw(11, N, K, 2, False, None), synth.normal_f32(12, 1, M * K).reshape(M, K)
    print(f"[gpu] M={M}", flush=True)
    rows = np.r_[0:40, 70000:70040, N - 40:N]
    part = oracle.QWeight(np.ascontiguousarray(w.qbytes.reshape(N, -1)[rows]), w.scales.reshape(N, -1)[rows], rows.size, K,
                          2)
    with Dev(ctx) as d:
        y = d.empty((M, N))
        ctx.linear_q(d.w(w), d.arr(x).ptr, y.ptr, M)
        _check_sum(y.to_host()[:, rows], oracle.linear_q(x, part), _bound(x, part), f"M={M}")


def test_capture_without_room_for_the_split(ctx):
    N, K, M = 256, 1536, 3000  # the split takes 19 MB; a context starts with no workspace
    w, x = _qw(7, N, K, 4, False, None), synth.normal_f32(8, 1, M * K).reshape(M, K)
    with g4a.Context(0) as own, Dev(own) as d:
        dw, dx, y = d.w(w), d.arr(x), d.empty((M, N))
        print("[gpu] capture", flush=True)
        own.capture_begin()
        own.linear_q(dw, dx.ptr, y.ptr, M)
        graph = own.capture_end()
        want, bound = oracle.linear_q(x[:100], w), _bound(x[:100], w)
        for _ in range(2):
            graph.launch()
            _check_sum(y.to_host()[:100], want, bound, "replay")
            own.linear_q(dw, dx.ptr, y.ptr, M)  # the workspace grows between the replays
            _check_sum(y.to_host()[:100], want, bound, "eager")
        graph.free()
