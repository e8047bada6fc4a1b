"""OperationType::FP32 on the GPU: the float kernels one by one against float64
NumPy statements of the same arithmetic, then the whole layer (C++ API through
bt_encoder_layer_forward, the PyTorch operator, the whole-encoder entry) against the
CPU oracle.

Tolerances (float): kernels carry a bound derived from fp32 rounding written in each
test; the whole layer must agree with the fp32 oracle within max-abs 2e-4 and mean-abs
2e-5 over the valid rows (outputs are O(1) after the last LayerNorm; both sides round
in fp32, in different orders)."""
import math
import os

import numpy as np
import pytest
import torch

import bytetransformer_amd as bt
from bytetransformer_amd import ops, workload
from oracle import bert_oracle as O

pytestmark = pytest.mark.gpu

F32_MAX_ABS, F32_MEAN_ABS = 2e-4, 2e-5
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def _say(*a):
    print(*a, flush=True)


def _dev(a, device):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


@pytest.fixture(params=[2, 3], ids=["default-order", "balanced-order"])
def att_order(request):
    """Runs a test under the default workgroup order and with the balanced work list
    forced on (small launches would not use it by themselves)."""
    ops.set_option("attention_xcd_map", request.param)
    yield request.param
    ops.set_option("attention_xcd_map", 2)


# ---- GEMM ------------------------------------------------------------------------
@pytest.mark.parametrize("rows,M,N,K", [(300, 300, 768, 768), (1000, 777, 2304, 768),
                                        (4920, 4920, 3072, 768), (640, 513, 768, 3072),
                                        (70, 70, 136, 200), (5, 3, 8, 4), (129, 129, 132, 20)])
def test_gemm_f32_plain_and_bias(device, rows, M, N, K):
    _say("gemm_f32", rows, M, N, K)
    rs = np.random.RandomState(rows + N)
    a = rs.standard_normal((rows, K)).astype(np.float32)
    a[M:] = np.nan                                   # rows past the live count are never read
    w = (rs.standard_normal((K, N)) * 0.05).astype(np.float32)
    bias = rs.standard_normal(N).astype(np.float32)
    vr = torch.tensor([M], dtype=torch.int32, device=device)
    # |error| <= K * 2^-24 * sum|a||w| is the textbook bound; sqrt(K) of it is generous
    bound = 4 * math.sqrt(K) * 2.0 ** -24 * (np.abs(a[:M]).astype(np.float64) @ np.abs(w)) + 1e-7
    for b in (None, bias):
        exp = O.gemm(a[:M], w, b)
        sentinel = torch.full((rows, N), 7.0, dtype=torch.float32, device=device)
        g = ops.gemm_f32(_dev(a, device), _dev(w, device), None if b is None else _dev(b, device),
                         valid_rows=vr, out=sentinel).cpu().numpy()
        assert np.all(np.abs(g[:M] - exp) <= bound), np.abs(g[:M] - exp).max()
        assert np.all(g[M:] == 7.0)


def test_gemm_f32_detects_transposed_or_shifted_operands(device):
    """Identity-like weights pin the operand orientation: A . P with P a cyclic column
    shift must shift the columns of A, exactly."""
    rs = np.random.RandomState(3)
    a = rs.standard_normal((200, 64)).astype(np.float32)
    p = np.roll(np.eye(64, dtype=np.float32), 5, axis=1)      # column j of A lands in j + 5
    g = ops.gemm_f32(_dev(a, device), _dev(p, device)).cpu().numpy()
    assert np.array_equal(g, np.roll(a, 5, axis=1))


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("rows,M,N,K", [(1, 1, 4, 4), (65, 33, 68, 20), (64, 64, 64, 64), (130, 97, 100, 1036),
                                        (33, 32, 32, 16)])
def test_gemm_f32_every_tile_at_its_edges(device, tile, rows, M, N, K):
    """Each tile with remainders in rows, columns and k (fewer k than waves, a cut last slice),
    gathered rows and the epilogue: as close to the exact product as a float accumulator gets."""
    rs = np.random.RandomState(rows * 7 + K)
    a = rs.standard_normal((rows, K)).astype(np.float32)
    w = (rs.standard_normal((K, N)) * 0.2).astype(np.float32)
    bias = rs.standard_normal(N).astype(np.float32)
    index = np.concatenate([rs.permutation(rows)[:M], np.full(rows - M, 1 << 30)]).astype(np.int32)
    exp = O.gemm(a[index[:M]].astype(np.float64), w.astype(np.float64), bias.astype(np.float64))
    bound = 2.0 ** -24 * (2 + math.sqrt(K)) * (np.abs(a[index[:M]]).astype(np.float64) @ np.abs(w) + np.abs(bias))
    ops.set_option("f32_gemm_tile", tile)
    try:
        out = torch.full((rows, N), 7.0, dtype=torch.float32, device=device)
        g = ops.gemm_f32(_dev(a, device), _dev(w, device), _dev(bias, device),
                         valid_rows=torch.tensor([M], dtype=torch.int32, device=device),
                         a_row_index=_dev(index, device), rows_cap=rows, out=out).cpu().numpy()
    finally:
        ops.set_option("f32_gemm_tile", -1)
    assert np.all(np.abs(g[:M] - exp) <= bound), (np.abs(g[:M] - exp) / bound).max()
    assert np.all(g[M:] == 7.0)


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("rows,M,K", [(100, 20, 36), (5000, 70, 64), (1200000, 40, 1024)])
def test_gemm_f32_gathers_any_row_of_a(device, tile, rows, M, K):
    """rows_cap bounds the output and not the operand that the rows are gathered from: rows past it, and (the last
    shape) rows of one tile more than 4 GiB apart."""
    _say("gemm_f32 gather", tile, rows, M, K)
    rs = np.random.RandomState(M + tile)
    N = 72
    index = np.concatenate([[rows - 1, 0, rows // 2], rs.permutation(rows)[:M - 3]]).astype(np.int32)
    if K == 1024:                                       # (only the rows that are read are filled)
        index[:] = np.where(np.arange(M) % 2, np.arange(M), rows - 1 - np.arange(M))
    live = rs.standard_normal((M, K)).astype(np.float32)
    a = torch.empty(rows, K, dtype=torch.float32, device=device)
    a[torch.from_numpy(index.astype(np.int64)).to(device)] = _dev(live, device)
    live = a[torch.from_numpy(index.astype(np.int64)).to(device)].cpu().numpy()   # (an index may come twice)
    w = (rs.standard_normal((K, N)) * 0.1).astype(np.float32)
    exp = O.gemm(live.astype(np.float64), w.astype(np.float64))
    bound = 2.0 ** -24 * (2 + math.sqrt(K)) * (np.abs(live).astype(np.float64) @ np.abs(w))
    ops.set_option("f32_gemm_tile", tile)
    try:
        g = ops.gemm_f32(a, _dev(w, device), valid_rows=torch.tensor([M], dtype=torch.int32, device=device),
                         a_row_index=_dev(index, device), rows_cap=M).cpu().numpy()
    finally:
        ops.set_option("f32_gemm_tile", -1)
    assert g.shape == (M, N)
    assert np.all(np.abs(g - exp) <= bound), (np.abs(g - exp) / bound).max()


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_gemm_f32_at_the_ends_of_the_float_range(device, tile):
    """The bfloat16 triples hold a float between 2^-110 and the largest bfloat16: infinities, NaN, floats past that
    and sums of tiny operands must come out as float arithmetic has them, and rows without any as before."""
    rs = np.random.RandomState(tile)
    rows, N, K = 70, 68, 52
    a = rs.standard_normal((rows, K)).astype(np.float32)
    w = (rs.standard_normal((K, N)) * 0.1 + 0.01).astype(np.float32)
    top = np.float32(3.4e38)               # a float, but rounds to an infinite bfloat16
    a[3, 5], a[4, 0], a[5, 51] = np.inf, -np.inf, np.nan
    a[6, :] = 0
    a[6, 7] = top
    a[7, 2], a[7, 9] = np.inf, -np.inf     # NaN wherever both weights have one sign
    a[8, :], a[9, :] = a[8, :] * np.float32(1e-35), a[9, :] * np.float32(1e-38)
    a[10, :] = a[10, :] * np.float32(2.0 ** -60)
    a[65, :] = a[65, :] * np.float32(1e-30)
    a[66, :] = 0
    w[7, 64] = 0                           # 0 * inf
    w[:, 65] = w[:, 65] * np.float32(2.0 ** -60)
    w[11, 66] = np.inf
    w[11, 67] = -top
    with np.errstate(invalid="ignore", over="ignore"):
        a64, w64 = a.astype(np.float64), w.astype(np.float64)
        exp = a64 @ w64
        exp[np.abs(exp) > np.finfo(np.float32).max] *= np.inf
        # a float accumulator, and denormal products and sums: half of float's smallest step each
        bound = 2.0 ** -24 * (2 + math.sqrt(K)) * (np.abs(a64) @ np.abs(w64)) + 2 * K * 2.0 ** -150
    ops.set_option("f32_gemm_tile", tile)
    try:
        g = ops.gemm_f32(_dev(a, device), _dev(w, device)).cpu().numpy().astype(np.float64)
    finally:
        ops.set_option("f32_gemm_tile", -1)
    # (a product of more than 3.4e38 on the way to a smaller sum may or may not overflow: leave such sums out)
    with np.errstate(invalid="ignore", over="ignore"):
        near = np.nan_to_num(np.abs(a64) @ np.abs(w64), nan=0.0, posinf=0.0) > 3e38
    special = ~np.isfinite(exp)
    assert special[3:6].all() and special[7].all() and special[:, 66].all() and np.isfinite(exp[6, :66]).all()
    assert np.array_equal(g[special & ~near], exp[special & ~near], equal_nan=True)
    usual = ~special & ~near
    assert usual[8:11].sum() > 100 and usual[6, :66].all()
    err = np.abs(g[usual] - exp[usual])
    assert np.all(err <= bound[usual]), (err / bound[usual]).max()
    assert np.all(g[66, :66] == 0)


def test_gemm_f32_bias_gelu_and_gather(device):
    _say("gemm_f32 gelu + gather")
    rs = np.random.RandomState(11)
    B, S, H, F = 4, 50, 128, 512
    lens = np.array([50, 0, 17, 33])
    x = rs.standard_normal((B, S, H)).astype(np.float32)
    mask = workload.make_mask(lens, S, np.float32)
    w = (rs.standard_normal((H, F)) * 0.2).astype(np.float32)
    bias = rs.standard_normal(F).astype(np.float32)
    g_bi, g_wi, M = ops.build_offsets(_dev(mask, device), want_count=True)
    packed = O.compress(x, g_wi.cpu().numpy()[:M])
    exp = O.gemm(packed, w, bias, "gelu_tanh")
    # the product's fp32 rounding (as in the plain test) passes through a slope <= 1.13,
    # then the activation adds a few ulp of its own
    bound = 1.13 * 4 * math.sqrt(H) * 2.0 ** -24 * (np.abs(packed).astype(np.float64) @ np.abs(w)) \
        + 4e-6 * np.abs(exp) + 2e-6
    g = ops.gemm_f32(_dev(x, device).view(B * S, H), _dev(w, device), _dev(bias, device),
                     gelu=True, valid_rows=g_bi[B:], a_row_index=g_wi).cpu().numpy()
    assert np.all(np.abs(g[:M] - exp) <= bound), np.abs(g[:M] - exp).max()
    assert np.all(g[M:] == 0)
    # special values of the activation: 0 -> 0, large |x| -> x or 0
    z = np.zeros((4, 4), np.float32)
    for v, want in ((0.0, 0.0), (30.0, 30.0), (-30.0, 0.0), (1e4, 1e4), (-1e4, 0.0)):
        b4 = np.full(4, v, np.float32)
        got = ops.gemm_f32(_dev(z, device), _dev(z, device), _dev(b4, device), gelu=True)
        assert np.all(got.cpu().numpy() == want), (v, got)


# ---- LayerNorm -------------------------------------------------------------------
# ---- split operands ----------------------------------------------------------------
def _joined(pairs, exps):
    """What pairs [rows, K / 32, 64] and an exponent per row (or per 256 of a row: [ceil(K / 256), rows]) stand for."""
    p = pairs.cpu().numpy().astype(np.float64)
    x = (p[:, :, :32] + p[:, :, 32:] / 2048).reshape(p.shape[0], -1)
    e = exps.cpu().numpy()
    e = e[:, None] if e.ndim == 1 else np.repeat(e.T, 256, axis=1)[:, :x.shape[1]]
    with np.errstate(invalid="ignore"):
        return x * 2.0 ** -e.astype(np.float64)


def _pair_bound(x, groups=None):
    """2^-23 of a value, 2^-50 of the largest that shares its scale (2^-25, half the spacing of
    subnormal fp16, in l, worth 2^-11, of a value scaled to at least 2^14)."""
    with np.errstate(invalid="ignore"):
        fin = np.where(np.isfinite(x), np.abs(x), 0).astype(np.float64)
    top = fin.max(1, keepdims=True)
    if groups:
        top = np.concatenate([np.repeat(fin[:, k:k + 256].max(1, keepdims=True), fin[:, k:k + 256].shape[1], 1)
                              for k in range(0, x.shape[1], 256)], 1)
    return fin * 2.0 ** -23 + top * 2.0 ** -50 + 2.0 ** -149


@pytest.mark.parametrize("K,N", [(64, 32), (256, 96), (320, 64), (768, 160)])
def test_split_f32_holds_what_it_was_given(device, K, N):
    """Weights and gathered rows over the whole range of floats, zeros, infinities and NaN among them."""
    _say("split_f32", K, N)
    rs = np.random.RandomState(K)
    w = (rs.standard_normal((K, N)) * 2.0 ** rs.randint(-20, 20, (K, N))).astype(np.float32)
    w[:, 1] = 0
    w[:, 2] *= np.float32(1e-30)
    w[:, 3] = np.finfo(np.float32).max * rs.choice([-1, 1], K)
    w[:, 4] = 2.0 ** -140
    w[3, 5], w[K - 1, 6], w[K // 2, 7] = np.inf, -np.inf, np.nan
    x = (rs.standard_normal((40, K)) * 2.0 ** rs.randint(-60, 60, (40, 1))).astype(np.float32)
    x[11, 5], x[12, 6], x[13] = np.inf, np.nan, 0
    idx = rs.permutation(40)[:33].astype(np.int32)
    bias = rs.standard_normal(N).astype(np.float32)
    vr = torch.tensor([31], dtype=torch.int32, device=device)
    (wp,), rows, bounds = ops.split_f32([_dev(w, device)], _dev(x, device), 0, _dev(bias, device), _dev(idx, device), vr, 33)
    for got, exp, groups in ((_joined(*wp), w.T, True), (_joined(*rows)[:31], x[idx[:31]], False)):
        fin = np.isfinite(exp)
        assert np.array_equal(np.isnan(got), np.isnan(exp)) and np.array_equal(got[np.isinf(exp)], exp[np.isinf(exp)])
        off = np.abs(np.where(fin, got, 0) - np.where(fin, exp, 0).astype(np.float64))
        assert np.all(off <= _pair_bound(exp, groups)), (off / _pair_bound(exp, groups)).max()
    assert not rows[0][31:].any() and not rows[1][31:].any()       # rows past the live count untouched
    top = np.where(np.isfinite(w), np.abs(w), 0)
    assert bounds[:, 0].max().item() == top.max() and bounds[:, 1].max().item() == np.abs(bias).max()


@pytest.mark.parametrize("lens,S", [([5], 5), ([0, 17, 0], 17), ([64, 1, 33], 64), ([200, 0, 131, 65, 200, 7, 1, 90, 199], 200), ([3] * 64, 8), ([100] * 33, 129)])
def test_split_f32_counts_the_mask_rows(device, lens, S):
    """The launch that counts its rows leaves the offsets of bt_build_offsets, and the same pairs of the same rows and weights."""
    _say("split_f32 mask rows", len(lens), S)
    rs = np.random.RandomState(S)
    B, K = len(lens), 128
    mask = np.zeros((B, S, S), np.float32)
    for b, n in enumerate(lens):
        mask[b, :, :n] = 1
    x, w = _dev(rs.standard_normal((B * S, K)).astype(np.float32), device), _dev(rs.standard_normal((K, 64)).astype(np.float32), device)
    m = _dev(mask, device)
    (wp,), got, _, (batch_idx, word_idx, seq_order) = ops.split_f32([w], x, mask=m, layer=True)
    exp_word = np.concatenate([b * S + np.arange(n) for b, n in enumerate(lens)] + [b * S + np.arange(n, S) for b, n in enumerate(lens)])
    M = sum(lens)
    assert np.array_equal(batch_idx.cpu().numpy(), np.concatenate([[0], np.cumsum(lens)]))
    assert np.array_equal(word_idx.cpu().numpy(), exp_word)
    assert np.array_equal(seq_order.cpu().numpy(), sorted(range(B), key=lambda b: (-lens[b], b)))
    vr = torch.tensor([M], dtype=torch.int32, device=device)
    (vp,), ref, _ = ops.split_f32([w], x, row_index=word_idx, valid_rows=vr, layer=True)
    assert all(torch.equal(one, other) for one, other in zip(wp + got, vp + ref))


@pytest.mark.parametrize("tile", [-1, 0, 1, 2])
@pytest.mark.parametrize("rows,M,N,K", [(300, 300, 768, 768), (200, 131, 160, 64), (97, 96, 32, 320), (64, 1, 2304, 768), (140, 140, 192, 512),
                                        (130, 129, 96, 3072), (193, 193, 416, 832)])
def test_gemm_f32_split_against_float64(device, tile, rows, M, N, K):
    _say("gemm_f32_split", tile, rows, M, N, K)
    rs = np.random.RandomState(rows + N + K)
    x = (rs.standard_normal((rows, K)) * 2.0 ** rs.randint(-30, 30, (rows, 1))).astype(np.float32)
    w = (rs.standard_normal((K, N)) * 2.0 ** rs.randint(-30, 30, (1, N)) * 2.0 ** rs.randint(-9, 9, (K // 64, 1)).repeat(64, 0))
    w = w.astype(np.float32)
    bias = np.zeros(N, np.float32)
    vr = torch.tensor([M], dtype=torch.int32, device=device)
    (wp,), a, _ = ops.split_f32([_dev(w, device)], _dev(x, device))
    ops.set_option("f32_gemm_tile", tile)
    try:
        out = torch.full((rows, N), 7.0, dtype=torch.float32, device=device)
        g = ops.gemm_f32_split(a, wp, None, None, vr, out).cpu().numpy()
        gb = ops.gemm_f32_split(a, wp, _dev(bias, device), None, vr).cpu().numpy()
    finally:
        ops.set_option("f32_gemm_tile", -1)
    exp = x[:M].astype(np.float64) @ w.astype(np.float64)
    # each operand to 2^-23, the second numbers' product 2^-22 left out, K / 16 float roundings at most, which do not add up
    # in one direction: (4 + sqrt(K) / 2) 2^-23 of sum |a||w|
    bound = (4 + math.sqrt(K) / 2) * 2.0 ** -23 * (np.abs(x[:M]).astype(np.float64) @ np.abs(w).astype(np.float64))
    assert np.all(np.abs(g[:M] - exp) <= bound), (np.abs(g[:M] - exp) / bound).max()
    assert np.all(g[M:] == 7.0) and np.array_equal(gb[:M], g[:M])
    if K >= 512 and M * N > 10000:
        # from there on no further from float64 than the products of whole floats, on operands of one scale
        y, v = rs.standard_normal((M, K)).astype(np.float32), (rs.standard_normal((K, N)) * 0.02).astype(np.float32)
        (vp,), b, _ = ops.split_f32([_dev(v, device)], _dev(y, device))
        ref = y.astype(np.float64) @ v.astype(np.float64)
        mine = np.linalg.norm(ops.gemm_f32_split(b, vp).cpu().numpy() - ref)
        whole = np.linalg.norm(ops.gemm_f32(_dev(y, device), _dev(v, device)).cpu().numpy() - ref)
        _say("from float64: pairs %.2e whole %.2e" % (mine / np.linalg.norm(ref), whole / np.linalg.norm(ref)))
        assert mine <= whole


# hint None: the count itself; 0: padded rows, all of them live; else one that is out of date, and more rows than one round has
@pytest.mark.parametrize("rows,M,N,K,hint", [(2561, 2560, 3072, 64, None), (3000, 2049, 3072, 768, None),
                                             (2560, 2305, 3070 // 32 * 32, 320, None), (2100, 2048, 4096, 128, None),
                                             (2300, 2300, 3072, 128, 0), (6000, 5801, 3072, 192, 2200), (5000, 30, 3072, 64, 2560)])
def test_gemm_f32_split_known_rows_change_no_bit(device, rows, M, N, K, hint):
    """The tile that a known row count may choose gives the bits of the other, among rows and columns out of proportion too."""
    _say("gemm_f32_split rows_hint", rows, M, N, K, hint)
    known, cus = hint or M, torch.cuda.get_device_properties(device).multi_processor_count
    assert -(-known // 256) * -(-N // 128) <= cus and -(-known // 96) * -(-N // 128) > 2 * cus, "one round of the large tile for more"
    rs = np.random.RandomState(rows + K)
    x, w = rs.standard_normal((rows, K)).astype(np.float32), (rs.standard_normal((K, N)) * 0.02).astype(np.float32)
    x[5, 1], x[M - 1, 2], x[min(300, M - 2), 3] = 1e20, 1e20, np.inf
    w[7, 40], w[9, N - 1] = 1e12, 1e-30
    bias = _dev((rs.standard_normal(N) * 0.1).astype(np.float32), device)
    vr = None if hint == 0 else torch.tensor([M], dtype=torch.int32, device=device)
    wd, xd = _dev(w, device), _dev(x, device)
    (wp,), a, _ = ops.split_f32([wd], xd, layer=True)
    ge = torch.full((rows,), 9, dtype=torch.int32, device=device)
    got = []
    for tile, given in ((2, 0), (-1, known)):
        ops.set_option("f32_gemm_tile", tile)
        try:
            raw = torch.zeros(rows, 1 + (N + 1023) // 1024, dtype=torch.int32, device=device)
            got.append((ops.gemm_f32_split(a, wp, bias, None, vr, weight=wd, rows=xd, rows_hint=given),
                        ops.gemm_f32_split(a, wp, bias, ge, vr, raw=raw, weight=wd, rows=xd, rows_hint=given), raw))
        finally:
            ops.set_option("f32_gemm_tile", -1)
    for one, other in zip(*got):
        assert torch.equal(one.view(torch.int32), other.view(torch.int32))
    assert not got[1][0][M:].any() and got[1][0][:M].isfinite().float().mean() > 0.9


@pytest.mark.parametrize("tile", [0, 1, 2])
def test_gemm_f32_split_passes_infinities_and_nan_on(device, tile):
    _say("gemm_f32_split inf nan", tile)
    rs = np.random.RandomState(3)
    x, w = rs.standard_normal((70, 128)).astype(np.float32), rs.standard_normal((128, 64)).astype(np.float32)
    x[3, 7], x[40, 100], x[41, 3], w[9, 5] = np.inf, -np.inf, np.nan, np.inf
    x[50, 9] = 0                                      # 0 . inf
    bias = rs.standard_normal(64).astype(np.float32)
    with np.errstate(invalid="ignore", over="ignore"):
        exp = x.astype(np.float64) @ w.astype(np.float64) + bias
    (wp,), a, _ = ops.split_f32([_dev(w, device)], _dev(x, device))
    ops.set_option("f32_gemm_tile", tile)
    try:
        g = ops.gemm_f32_split(a, wp, _dev(bias, device)).cpu().numpy()
        ge = torch.full((70,), 6, dtype=torch.int32, device=device)
        h = _joined(ops.gemm_f32_split(a, wp, _dev(bias, device), ge), ge)
    finally:
        ops.set_option("f32_gemm_tile", -1)
    fin = np.isfinite(exp)
    assert fin.mean() > 0.9
    assert np.array_equal(np.isnan(g), np.isnan(exp)) and np.array_equal(g[np.isinf(exp)], exp[np.isinf(exp)])
    assert np.abs(g[fin] - exp[fin]).max() <= 1e-4
    gelu = exp[fin] / (1 + np.exp(-2 * 0.7978845608028654 * (exp[fin] + 0.044715 * exp[fin] ** 3)))
    assert np.isfinite(h[fin]).all() and np.abs(h[fin] - gelu).max() <= 1e-4
    assert np.all(np.isnan(h[~fin]) | np.isinf(h[~fin]) | (h[~fin] == 0))       # GELU(-inf) is -0 or NaN in float arithmetic


@pytest.mark.parametrize("tile", [0, 1, 2])
def test_gemm_f32_split_leaves_dead_rows_alone(device, tile):
    """What lies in the pairs of rows past the live count, infinities and NaN here, changes no bit of the others."""
    _say("gemm_f32_split dead rows", tile)
    rs = np.random.RandomState(tile)
    rows, M, N, K = 150, 101, 160, 192
    x, w = rs.standard_normal((rows, K)).astype(np.float32), rs.standard_normal((K, N)).astype(np.float32)
    bias, vr = _dev(rs.standard_normal(N).astype(np.float32), device), torch.tensor([M], dtype=torch.int32, device=device)
    ge = torch.full((rows,), 6, dtype=torch.int32, device=device)
    (wp,), (pairs, exps), _ = ops.split_f32([_dev(w, device)], _dev(x, device))
    dead = pairs.clone()
    dead[M:] = float("nan")
    dead[M:, ::2, ::3] = float("inf")
    ops.set_option("f32_gemm_tile", tile)
    try:
        for g in (None, ge):
            out = [torch.full((rows, N) if g is None else (rows, N // 32, 64), 7.0, device=device,
                              dtype=torch.float32 if g is None else torch.float16) for _ in range(2)]
            for p, o in zip((pairs, dead), out):
                ops.gemm_f32_split((p, exps), wp, bias, g, vr, o)
            assert torch.equal(*out) and bool((out[0][M:] == 7).all())
    finally:
        ops.set_option("f32_gemm_tile", -1)


@pytest.mark.parametrize("H", [64, 768, 1024])
def test_layernorm_f32_split_keeps_the_gelu_in_range(device, H):
    """The LayerNorm's rows are those of the plain one, its pairs stand for them, and the exponents it gives to FFN1 leave
    every result of it finite and where it belongs, large weights and biases included."""
    _say("layernorm_f32_split", H)
    rs = np.random.RandomState(H)
    rows, M, F = 45, 40, 96
    out, res = rs.standard_normal((rows, H)).astype(np.float32), rs.standard_normal((50, H)).astype(np.float32)
    ridx = rs.permutation(50)[:rows].astype(np.int32)
    bias, beta = (rs.standard_normal(H).astype(np.float32) for _ in range(2))
    gamma = (1 + rs.standard_normal(H)).astype(np.float32) * 30
    w, b1 = (rs.standard_normal((H, F)) * 50).astype(np.float32), (rs.standard_normal(F) * 1e4).astype(np.float32)
    vr = torch.tensor([M], dtype=torch.int32, device=device)
    (wp,), _, bounds = ops.split_f32([_dev(w, device)], None, 0, _dev(b1, device))
    args = [_dev(a, device) for a in (res, bias, gamma, beta)]
    mine, plain = _dev(out, device), _dev(out, device)
    pairs, exps, ge = ops.add_bias_residual_layernorm_f32_split(mine, *args, bounds, 1e-6, vr, _dev(ridx, device))
    ops.add_bias_residual_layernorm_f32(plain, *args, 1e-6, valid_rows=vr, residual_row_index=_dev(ridx, device))
    assert torch.equal(mine, plain)
    ln = plain.cpu().numpy()[:M]
    assert np.all(np.abs(_joined(pairs, exps)[:M] - ln) <= _pair_bound(ln))
    got = _joined(ops.gemm_f32_split((pairs, exps), wp, _dev(b1, device), ge, vr), ge)[:M]
    u = ln.astype(np.float64) @ w.astype(np.float64) + b1
    with np.errstate(over="ignore"):
        exp = u / (1 + np.exp(-2 * 0.7978845608028654 * (u + 0.044715 * u ** 3)))
    assert np.isfinite(got).all()
    # the product to 2^-20 of sum |a||w|, GELU in float, pairs to 2^-23
    bound = 2.0 ** -20 * (np.abs(ln).astype(np.float64) @ np.abs(w).astype(np.float64) + np.abs(b1)) + 1e-6
    assert np.all(np.abs(got - exp) <= bound), (np.abs(got - exp) / bound).max()


@pytest.mark.parametrize("size", [1e14, 1e19, 1e30])
def test_layernorm_f32_split_bounds_rows_whose_squares_are_no_floats(device, size):
    """Rows whose sum of squares leaves the float range, a product beyond fp16 that does not, and a bias with an infinity:
    every finite result of FFN1 stays finite and where it belongs."""
    _say("layernorm_f32_split large", size)
    rs = np.random.RandomState(5)
    rows, H, F = 33, 768, 64
    zero = np.zeros(H, np.float32)
    out, res = (rs.standard_normal((rows, H)).astype(np.float32) for _ in range(2))
    gamma = (rs.standard_normal(H) * size).astype(np.float32)
    w, b1 = (rs.standard_normal((H, F)) * (1e8 / size)).astype(np.float32), np.zeros(F, np.float32)
    b1[5] = np.inf
    (wp,), _, bounds = ops.split_f32([_dev(w, device)], None, 0, _dev(b1, device))
    mine = _dev(out, device)
    pairs, exps, ge = ops.add_bias_residual_layernorm_f32_split(mine, *[_dev(a, device) for a in (res, zero, gamma, zero)],
                                                                bounds, 1e-6)
    got = _joined(ops.gemm_f32_split((pairs, exps), wp, _dev(b1, device), ge), ge)
    ln = mine.cpu().numpy()
    assert np.isfinite(ln).all()
    u = ln.astype(np.float64) @ w.astype(np.float64) + b1
    fin = np.isfinite(u)
    assert np.array_equal(fin, np.repeat([np.arange(F) != 5], rows, 0)) and np.abs(u[fin]).max() > 65504
    exp = np.maximum(u, 0)                                          # GELU at 1e9: one side or the other
    # the product to 2^-20 of sum |a||w|; GELU of what lies about zero differs from this by less than 1
    bound = 2.0 ** -20 * (np.abs(ln).astype(np.float64) @ np.abs(w).astype(np.float64)) + 1
    assert np.isfinite(got[fin]).all() and np.all(np.abs(got - exp)[fin] <= bound[fin])
    assert np.all(np.isinf(got[:, 5]))


def _with_raw(pairs, exps, raw):
    """What pairs stand for where some blocks of 32 are floats."""
    words = raw.cpu().numpy().view(np.uint32)
    bits = words[:, 1:]
    assert np.array_equal(words[:, 0] != 0, bits.any(1))
    bits = (bits[:, :, None] >> np.arange(32, dtype=np.uint32) & 1).reshape(len(bits), -1)[:, :pairs.shape[1]]
    got = _joined(pairs, exps)
    floats = pairs.cpu().numpy().view(np.float32).reshape(got.shape)
    return np.where(np.repeat(bits, 32, axis=1) == 1, floats.astype(np.float64), got), bits


def _gelu64(u):
    with np.errstate(over="ignore", invalid="ignore"):
        return np.where(np.isneginf(u), -0.0, u / (1 + np.exp(-2 * 0.7978845608028654 * (u + 0.044715 * u ** 3))))


@pytest.mark.parametrize("tile", [-1, 0, 1, 2])
@pytest.mark.parametrize("what", ["ordinary", "bias -1e12", "bias -1e30", "bias 1e12", "bias 1e30", "weight 1e9", "weight 1e20", "gamma 1e20"])
def test_one_large_column_of_ffn1_leaves_the_others_alone(device, tile, what):
    """FFN1 and FFN2 as a layer runs them, with one column of FFN1 that is out of all proportion and that FFN2 gives no
    weight (or one of the LayerNorm, that FFN1 gives none): every other result of FFN1, and every result of FFN2, is what it would be without that column."""
    _say("one large column", tile, what)
    rs = np.random.RandomState(11)
    M, rows, H, F = 69, 75, 768, 1088
    col, zero = 77, np.zeros(H, np.float32)
    out, res = (rs.standard_normal((rows, H)).astype(np.float32) for _ in range(2))
    gamma = (1 + 0.05 * rs.standard_normal(H)).astype(np.float32)
    w1, b1 = (rs.standard_normal((H, F)) * 0.05).astype(np.float32), (rs.standard_normal(F) * 0.1).astype(np.float32)
    w2 = (rs.standard_normal((F, H)) * 0.05).astype(np.float32)
    if what.startswith("bias"):
        b1[col] = float(what[5:])
    elif what.startswith("weight"):
        w1[33, col] = float(what[7:])
    elif what.startswith("gamma"):
        gamma[9], w1[9] = float(what[6:]), 0
    w2[col] = 0
    vr = torch.tensor([M], dtype=torch.int32, device=device)
    w1d, w2d, b1d = _dev(w1, device), _dev(w2, device), _dev(b1, device)
    wp, _, bounds = ops.split_f32([w1d, w2d], None, 0, b1d, layer=True)
    mine = _dev(out, device)
    raw = torch.full((rows, 1 + (F + 1023) // 1024), -1, dtype=torch.int32, device=device)
    ops.set_option("f32_gemm_tile", tile)
    try:
        pairs, exps, ge = ops.add_bias_residual_layernorm_f32_split(mine, *[_dev(a, device) for a in (res, zero, gamma, zero)],
                                                                    bounds, 1e-6, vr, raw=raw)
        mid = ops.gemm_f32_split((pairs, exps), wp[0], b1d, ge, vr, raw=raw, weight=w1d, rows=mine)
        got2 = ops.gemm_f32_split((mid, ge), wp[1], None, None, vr, torch.full((rows, H), 7.0, device=device), a_raw=raw,
                                  weight=w2d).cpu().numpy()
    finally:
        ops.set_option("f32_gemm_tile", -1)
    got, bits = _with_raw(mid, ge, raw)
    assert np.all(raw.cpu().numpy()[M:] == -1) and bool(bits[:M].any()) == (what not in ("ordinary", "bias -1e12", "bias -1e30"))
    ln = mine.cpu().numpy()[:M].astype(np.float64)
    u = ln @ w1.astype(np.float64) + b1
    exp = _gelu64(u)
    others = np.arange(F) != col
    # the product to 2^-20 of sum |a||w|, GELU in float, pairs to 2^-22
    bound = 2.0 ** -20 * (np.abs(ln) @ np.abs(w1).astype(np.float64) + np.abs(b1)) + 1e-6
    off = np.abs(got[:M] - exp)
    assert np.all(off[:, others] <= bound[:, others]), (off / bound)[:, others].max()
    assert np.all(off[:, col] <= bound[:, col])
    exp2 = got[:M][:, others] @ w2[others].astype(np.float64)
    bound2 = (4 + math.sqrt(F) / 2) * 2.0 ** -23 * (np.abs(got[:M][:, others]) @ np.abs(w2[others]).astype(np.float64))
    assert np.all(np.abs(got2[:M] - exp2) <= bound2), (np.abs(got2[:M] - exp2) / bound2).max()
    assert np.all(got2[M:] == 7.0)


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("kind", ["ordinary", "scales", "small ones", "feature 1e16", "feature 1e30", "two values", "weight row 1e20",
                                  "weight 1e25", "both"])
def test_operands_out_of_proportion_are_summed_from_the_floats(device, tile, kind):
    """Values that leave their row, or their chunk of a column, no bits, and that meet a zero: the other products are summed
    as floats.  Scales that differ by a factor of a thousand are none of that."""
    _say("out of proportion", tile, kind)
    rs = np.random.RandomState(6)
    rows, M, N, K = 77, 70, 160, 320
    x, w = rs.standard_normal((90, K)).astype(np.float32), (rs.standard_normal((K, N)) * 0.05).astype(np.float32)
    bias = rs.standard_normal(N).astype(np.float32)
    idx = rs.permutation(90)[:rows].astype(np.int32)
    marked_rows, marked_columns = np.zeros(90, bool), np.zeros((2, N), bool)
    if kind == "scales":
        by = (2.0 ** rs.uniform(-5, 5, K)).astype(np.float32)
        x, w = x * by, (w.T / by).T.copy()
    if kind == "small ones":
        x[:, ::10] *= np.float32(1e-15)
        w[::10] *= np.float32(1e15)
        marked_rows[:], marked_columns[:] = True, True
    if kind.startswith("feature") or kind == "both":
        at = rs.permutation(90)[:40]
        x[at, 7] = 1e30 if kind == "both" else float(kind[8:])
        w[7] = 0
        marked_rows[at] = True
    if kind == "two values":
        x[:20] = 0
        x[:20, 3], x[:20, 9], w[3] = 1e30, rs.standard_normal(20), 0
        marked_rows[:20] = True
    if kind in ("weight row 1e20", "both"):
        w[5], x[:, 5] = 1e20, 0
        marked_columns[0] = True
    if kind == "weight 1e25":
        w[300, 33], x[:, 300] = -1e25, 0
        marked_columns[1, 33] = True
    xd, wd, vr = _dev(x, device), _dev(w, device), torch.tensor([M], dtype=torch.int32, device=device)
    (wp,), a, _ = ops.split_f32([wd], xd, row_index=_dev(idx, device), valid_rows=vr, rows_cap=rows, layer=True)
    assert np.array_equal(a[1].cpu().numpy()[:M] >= 2048, marked_rows[idx[:M]])
    assert np.array_equal(wp[1].cpu().numpy() >= 2048, marked_columns)
    live = x[idx[:M]].astype(np.float64)
    exp, size = live @ w.astype(np.float64) + bias, np.abs(live) @ np.abs(w).astype(np.float64) + np.abs(bias)
    bound = (4 + math.sqrt(K) / 2) * 2.0 ** -23 * size
    ge = torch.full((rows,), 7, dtype=torch.int32, device=device)
    more = dict(weight=wd, rows=xd, row_index=_dev(idx, device))
    ops.set_option("f32_gemm_tile", tile)
    try:
        got = ops.gemm_f32_split(a, wp, _dev(bias, device), None, vr, torch.full((rows, N), 7.0, device=device), **more).cpu().numpy()
        raw = torch.zeros(rows, 2, dtype=torch.int32, device=device)
        gelu, _ = _with_raw(ops.gemm_f32_split(a, wp, _dev(bias, device), ge, vr, raw=raw, **more), ge, raw)
    finally:
        ops.set_option("f32_gemm_tile", -1)
    assert np.all(np.abs(got[:M] - exp) <= bound), (np.abs(got[:M] - exp) / bound).max()
    assert np.all(got[M:] == 7.0)
    # GELU's slope is below 1.13, its float arithmetic good to 2^-20 of the argument
    assert np.all(np.abs(gelu[:M] - _gelu64(exp)) <= 2 * bound + 2.0 ** -20 * np.abs(exp)), "gelu"


@pytest.mark.parametrize("K", [768, 3072])
@pytest.mark.parametrize("where", ["rows", "weight", "both"])
def test_split_operands_of_any_scales_are_as_near_as_whole_floats(device, K, where):
    """Features whose scales differ by up to 2^76 (16 standard deviations of 2^12), with weights of one scale, the other way
    about, and inversely, so that every product counts: no further from float64 than the products of whole floats, or than
    operands off by 2^-22.5 each, from where on they are marked."""
    rs = np.random.RandomState(K)
    rows, N = 200, 256
    for bits in (0, 1, 2, 3, 4, 6, 8, 12):
        by, by2 = 2.0 ** (bits * rs.standard_normal(K)), 2.0 ** (bits * rs.standard_normal(K))
        x, w = rs.standard_normal((rows, K)), rs.standard_normal((K, N)) * 0.02
        if where != "weight":
            x *= by
        if where != "rows":
            w *= (1 / by if where == "both" else by2)[:, None]
        xd, wd = _dev(x.astype(np.float32), device), _dev(w.astype(np.float32), device)
        (wp,), a, _ = ops.split_f32([wd], xd, layer=True)
        ref = xd.double() @ wd.double()
        far = lambda got: ((got.double() - ref).norm() / ref.norm()).item()   # noqa: E731
        mine, whole = far(ops.gemm_f32_split(a, wp, weight=wd, rows=xd)), far(ops.gemm_f32(xd, wd))
        marked = [int((e >= 2048).sum()) for e in (a[1], wp[1])]
        _say("scales", where, K, bits, "pairs %.2e whole %.2e" % (mine, whole), "marked", marked)
        assert mine <= max(whole, 2.0 ** -22)
        assert bits > 2 or not any(marked)


@pytest.mark.parametrize("path", ["th_op", "encoder"])
@pytest.mark.parametrize("rm", [True, False])
def test_fp32_layers_with_weights_that_nothing_meets(device, path, rm):
    """A model whose last features are padding: zero wherever they are computed, so that what lies in the rows of the weights
    that read them, 1e20 here, counts for nothing."""
    _say("fp32 layers, weights that nothing meets", path, rm)
    cfg = workload.EncoderConfig("f32pad", 17, 120, 8, layers=2, dtype="fp32", lens=(120, 3, 41, 0, 64, 119) + (90,) * 11)
    wl = workload.make_workload(cfg, bias_std=0.05, random_affine=True)
    H, at = cfg.hidden, cfg.hidden - 3
    wl.x[..., at:] = 0
    readers = ("qkv_kernel", "attr_output_kernel", "inter_kernel", "output_kernel")
    for w in wl.layers:
        w["qkv_kernel"][:, 2 * H + at:], w["qkv_bias"][2 * H + at:] = 0, 0          # V
        w["inter_kernel"][:, at:H], w["inter_bias"][at:H] = 0, 0
        for n in ("attr_output", "output"):
            w[n + "_kernel"][:, at:], w[n + "_bias"][at:] = 0, 0
            w[n + "_layernorm_gamma"][at:], w[n + "_layernorm_beta"][at:] = 0, 0
        for n in readers:
            w[n][at:H] = 0
    exp = _oracle32(wl)
    for w in wl.layers:
        w["qkv_kernel"][at:, :2 * H + at] = 1e20
        w["attr_output_kernel"][at:, :at] = -1e20
        w["inter_kernel"][at:, :at], w["inter_kernel"][at:, H:] = 1e20, -1e20
        w["output_kernel"][at:H, :at] = 1e20
    x, m = _dev(wl.x, device), _dev(wl.mask, device)
    if path == "th_op":
        bt.load_th_op()
        got = x
        for w in wl.layers:
            got = torch.ops.ByteTransformer.BertTransformer(
                cfg.head_num, cfg.head_size, *[_dev(w[n], device) for n in workload.WEIGHT_NAMES], got, m, rm, True)
    else:
        got = bt.BertEncoder(cfg.head_num, cfg.head_size, [{k: _dev(v, device) for k, v in w.items()} for w in wl.layers],
                             is_remove_padding=rm)(x, m)
    got = got.cpu().numpy()
    _f32_check(got if rm else O.masked_output(got, wl.lens), exp, wl.lens, "f32 padding/%s" % path, rm)


@pytest.mark.parametrize("path", ["th_op", "encoder"])
@pytest.mark.parametrize("rm", [True, False])
@pytest.mark.parametrize("value", [-1e12, -1e30, 1e12])
def test_fp32_layers_with_one_large_ffn1_bias(device, path, rm, value):
    """Layers that split their operands, against the oracle without the column, whose GELU is zero or has no weight behind it."""
    _say("fp32 layers, large bias", path, rm, value)
    cfg = workload.EncoderConfig("f32big", 17, 120, 8, layers=2, dtype="fp32", lens=(120, 3, 41, 0, 64, 119) + (90,) * 11)
    wl = workload.make_workload(cfg, bias_std=0.05, random_affine=True)
    for w in wl.layers:
        w["inter_kernel"][:, 5], w["inter_bias"][5], w["output_kernel"][5] = 0, 0, 0
    exp = _oracle32(wl)
    for w in wl.layers:
        w["inter_bias"][5] = value
    x, m = _dev(wl.x, device), _dev(wl.mask, device)
    if path == "th_op":
        bt.load_th_op()
        got = x
        for w in wl.layers:
            got = torch.ops.ByteTransformer.BertTransformer(
                cfg.head_num, cfg.head_size, *[_dev(w[n], device) for n in workload.WEIGHT_NAMES], got, m, rm, True)
    else:
        got = bt.BertEncoder(cfg.head_num, cfg.head_size, [{k: _dev(v, device) for k, v in w.items()} for w in wl.layers],
                             is_remove_padding=rm)(x, m)
    got = got.cpu().numpy()
    _f32_check(got if rm else O.masked_output(got, wl.lens), exp, wl.lens, "f32 large bias/%s" % path, rm)


@pytest.mark.parametrize("path", ["c_api", "th_op", "encoder"])
@pytest.mark.parametrize("rm", [True, False])
def test_fp32_layers_on_split_operands(device, path, rm):
    """Sizes from which on a float layer splits its operands, against the oracle."""
    _say("fp32 split layers", path, rm)
    cfg = workload.EncoderConfig("f32s", 17, 120, 8, layers=2, dtype="fp32", lens=(120, 3, 41, 0, 64, 119) + (90,) * 11)
    wl = workload.make_workload(cfg, bias_std=0.05, random_affine=True)
    x, m = _dev(wl.x, device), _dev(wl.mask, device)
    if path == "c_api":
        got = bt.encoder_forward(_layers(wl, device, is_remove_padding=rm), x, m)
    elif path == "th_op":
        bt.load_th_op()
        got = x
        for w in wl.layers:
            got = torch.ops.ByteTransformer.BertTransformer(
                cfg.head_num, cfg.head_size, *[_dev(w[n], device) for n in workload.WEIGHT_NAMES], got, m, rm, True)
    else:
        got = bt.BertEncoder(cfg.head_num, cfg.head_size, [{k: _dev(v, device) for k, v in w.items()} for w in wl.layers],
                             is_remove_padding=rm)(x, m)
    got = got.cpu().numpy()
    _f32_check(got if rm else O.masked_output(got, wl.lens), _oracle32(wl), wl.lens, "f32 split/%s" % path, rm)


@pytest.mark.parametrize("lens,S", [((512, 0, 300, 37), 512), (None, 40), (None, 205), (None, 1024), (None, 20)])
def test_fp32_layers_rows_from_the_mask_never_change_the_result(device, lens, S):
    """Float layers that split their operands: rows counted by the launch that splits them, or by a prologue.  An empty
    sequence, 64 sequences of a few dozen tokens, odd lengths, the most mask rows the launch takes, more sequences than it takes."""
    _say("fp32 qkv_mask_rows", lens, S)
    bt.load_th_op()
    batch = len(lens) if lens else {40: 64, 205: 20, 1024: 16, 20: 128}[S]
    assert batch * S * 3 // 5 >= 1220 and ops.get_option("qkv_mask_rows") == -1
    cfg = workload.EncoderConfig("f32 mr", batch, S, 8, layers=1, dtype="fp32", lens=lens or (), seed=S)
    wl = workload.make_workload(cfg, bias_std=0.05, random_affine=True)
    w = [_dev(wl.layers[0][n], device) for n in workload.WEIGHT_NAMES]
    x, m = _dev(wl.x, device), _dev(wl.mask, device)
    got = {}
    try:
        for choice in (0, 1, -1):
            ops.set_option("qkv_mask_rows", choice)
            got[choice] = torch.ops.ByteTransformer.BertTransformer(8, 64, *w, x, m, True, True)
    finally:
        ops.set_option("qkv_mask_rows", -1)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[-1])
    live = torch.arange(S, device=device)[None, :] < torch.as_tensor(np.asarray(wl.lens), device=device)[:, None]
    assert got[-1][live].isfinite().all() and got[-1][live].any(-1).all() and not got[-1][~live].any()


@pytest.mark.parametrize("H", [768, 1024, 64, 4096, 260])
def test_layernorm_f32(device, H):
    _say("layernorm_f32", H)
    rs = np.random.RandomState(H)
    rows, M = 37, 30
    out = rs.standard_normal((rows, H)).astype(np.float32)
    res = (rs.standard_normal((rows, H)) + 3.0).astype(np.float32)
    bias = rs.standard_normal(H).astype(np.float32)
    gamma = (1 + 0.2 * rs.standard_normal(H)).astype(np.float32)
    beta = (0.3 * rs.standard_normal(H)).astype(np.float32)
    exp = O.add_bias_residual_layernorm(out[:M], res[:M], bias, gamma, beta, 1e-6, fp16_adds=False)
    vr = torch.tensor([M], dtype=torch.int32, device=device)
    g = ops.add_bias_residual_layernorm_f32(_dev(out, device), _dev(res, device), _dev(bias, device),
                                            _dev(gamma, device), _dev(beta, device), 1e-6,
                                            valid_rows=vr).cpu().numpy()
    assert np.all(np.abs(g[:M] - exp) <= 4e-6 * np.abs(exp) + 4e-6), np.abs(g[:M] - exp).max()
    assert np.array_equal(g[M:], out[M:])            # rows past M untouched
    # gamma = 1, beta = 0: every row has mean 0 and variance 1 / (1 + eps / var)
    one, zero = np.ones(H, np.float32), np.zeros(H, np.float32)
    g = ops.add_bias_residual_layernorm_f32(_dev(out, device), _dev(res, device), _dev(zero, device),
                                            _dev(one, device), _dev(zero, device), 1e-6).cpu().numpy()
    assert np.all(np.abs(g.mean(-1)) < 1e-5) and np.all(np.abs(g.var(-1) - 1) < 1e-4)


def test_layernorm_restore_f32_zero_fills(device):
    rs = np.random.RandomState(5)
    B, S, H = 5, 33, 768
    lens = np.array([33, 0, 20, 1, 32])
    mask = workload.make_mask(lens, S, np.float32)
    bi, wi, M = O.build_offsets(mask)
    out = rs.standard_normal((B * S, H)).astype(np.float32)
    res = rs.standard_normal((B * S, H)).astype(np.float32)
    bias = rs.standard_normal(H).astype(np.float32)
    gamma = (1 + 0.2 * rs.standard_normal(H)).astype(np.float32)
    beta = (0.3 * rs.standard_normal(H)).astype(np.float32)
    exp = O.restore(O.add_bias_residual_layernorm(out[:M], res[:M], bias, gamma, beta, 1e-6,
                                                  fp16_adds=False), bi, B, S)
    g_bi, _, _ = ops.build_offsets(_dev(mask, device))
    target = torch.full((B, S, H), float("nan"), dtype=torch.float32, device=device)
    g = ops.add_bias_residual_layernorm_restore_f32(
        _dev(out, device), _dev(res, device), _dev(bias, device), _dev(gamma, device),
        _dev(beta, device), g_bi, B, S, 1e-6, out_padded=target).cpu().numpy()
    for b in range(B):
        assert np.all(g[b, lens[b]:].view(np.uint32) == 0)
    assert np.all(np.abs(g - exp) <= 4e-6 * np.abs(exp) + 4e-6)


# ---- attention -------------------------------------------------------------------
def _naive_attention(qkv, lens, S, heads, d, scale, padded, mask=None, bias=None):
    """float64, one (sequence, head) at a time, logits + bias + (mask - 1) * 10000."""
    H = heads * d
    out = np.zeros((qkv.shape[0], H))
    start = 0
    for b, n in enumerate(lens):
        r0 = b * S if padded else start
        nq = S if padded else n
        nk = S if (padded and mask is not None) else n
        start += n
        if nk == 0:
            continue
        rows = qkv[r0:r0 + max(nq, nk)].astype(np.float64)
        for g in range(heads):
            q = rows[:nq, g * d:(g + 1) * d]
            k = rows[:nk, H + g * d:H + (g + 1) * d]
            v = rows[:nk, 2 * H + g * d:2 * H + (g + 1) * d]
            s = q @ k.T * scale
            if bias is not None:
                s = s + bias[g, :nq, :nk]
            if mask is not None:
                s = s + (mask[b, :nq, :nk].astype(np.float64) - 1.0) * 10000.0
            e = np.exp(s - s.max(-1, keepdims=True))
            p = e / (e.sum(-1, keepdims=True) + 1e-6)
            out[r0:r0 + nq, g * d:(g + 1) * d] = p @ v
    return out


F32_ATT_CASES = [
    ([64, 38], 64, 12, 64), ([154], 256, 12, 64), ([1, 16, 17, 0, 100, 128, 129], 160, 3, 64),
    ([300, 77, 5], 320, 2, 64), ([40, 33], 40, 4, 32), ([70, 9], 72, 2, 128),
    ([50, 31], 50, 2, 48), ([50, 31], 50, 3, 104),
]


@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("lens,S,heads,d", F32_ATT_CASES)
def test_attention_f32(device, lens, S, heads, d, padded, att_order):
    _say("attention_f32", lens, S, heads, d, padded)
    rs = np.random.RandomState(S + heads + d)
    B, H = len(lens), heads * d
    rows_cap = B * S
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = np.full((rows_cap, 3 * H), np.nan, np.float32)
    if padded:
        qkv[:] = rs.standard_normal(qkv.shape).astype(np.float32)   # padded rows hold finite junk
    else:
        qkv[:bi[-1]] = rs.standard_normal((bi[-1], 3 * H)).astype(np.float32)
    qkv[:, :H] *= 2.0
    scale = 1 / math.sqrt(d)
    exp = _naive_attention(qkv, lens, S, heads, d, scale, padded)
    # the issue order (longest first) must not change anything
    order = np.argsort(-np.asarray(lens), kind="stable").astype(np.int32)
    g = ops.attention_f32(_dev(qkv, device), _dev(bi, device), B, S, heads, scale,
                          padded_rows=padded, seq_order=_dev(order, device)).cpu().numpy()
    g0 = ops.attention_f32(_dev(qkv, device), _dev(bi, device), B, S, heads, scale,
                           padded_rows=padded).cpu().numpy()
    live = ~np.isnan(g0)
    assert np.array_equal(np.isnan(g), ~live) and np.array_equal(g[live], g0[live])
    for b, n in enumerate(lens):
        r0 = b * S if padded else bi[b]
        # padded rows: queries past the length attend the valid keys too (defined output)
        nq = S if padded else n
        if n == 0:
            continue
        err = np.abs(g[r0:r0 + nq] - exp[r0:r0 + nq])
        assert err.max() <= 2e-5, (b, err.max())


@pytest.mark.parametrize("padded", [False, True])
def test_attention_f32_mask_and_bias(device, padded, att_order):
    """An arbitrary 0/1 mask (every query keeps at least one key) and a bias: the kernel
    must apply both per (query, key), on both row layouts."""
    _say("attention_f32 mask+bias", padded)
    rs = np.random.RandomState(9)
    lens, S, heads, d = [72, 30, 50], 72, 3, 64
    B, H = len(lens), heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((B * S, 3 * H)).astype(np.float32)
    mask = (rs.rand(B, S, S) < 0.6).astype(np.float32)
    mask[:, :, 0] = 1
    if not padded:
        for b, n in enumerate(lens):
            mask[b, :, n:] = 0
    bias = rs.standard_normal((heads, S, S)).astype(np.float32)
    scale = 0.125
    exp = _naive_attention(qkv, lens, S, heads, d, scale, padded, mask, bias)
    g = ops.attention_f32(_dev(qkv, device), _dev(bi, device), B, S, heads, scale,
                          padded_rows=padded, mask=_dev(mask, device),
                          bias=_dev(bias, device)).cpu().numpy()
    for b, n in enumerate(lens):
        r0, nq = (b * S, S) if padded else (bi[b], n)
        err = np.abs(g[r0:r0 + nq] - exp[r0:r0 + nq])
        assert err.max() <= 2e-5, (b, err.max())


@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("lens,S,heads,d", [([65, 1, 0, 33], 65, 3, 64), ([128, 96, 64, 32], 128, 2, 64), ([97, 31], 97, 5, 40),
                                            ([129, 63, 95], 131, 3, 32), ([16, 5], 16, 2, 8), ([400], 400, 1, 56)])
def test_attention_f32_on_shared_keys(device, lens, S, heads, d, padded, add, att_order):
    """64 queries whose keys two groups of waves share, and 128: lengths about a group's tile (32) and a turn (64), a group
    without a key, a sequence without any. Sums of n keys in two orders, each of them off by at most a few n 2^-24 of values
    of O(1): 2e-5, as in the tests above."""
    rs = np.random.RandomState(S + heads + d)
    B, H = len(lens), heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((B * S, 3 * H)).astype(np.float32)
    if not padded:
        qkv[bi[-1]:] = np.nan
    mask = bias = None
    if add:
        bias = rs.standard_normal((heads, S, S)).astype(np.float32)
        mask = (rs.rand(B, S, S) < 0.6).astype(np.float32)
        mask[:, :, 0] = 1
        if not padded:
            for b, n in enumerate(lens):
                mask[b, :, n:] = 0
    scale = 1 / math.sqrt(d)
    exp = _naive_attention(qkv, lens, S, heads, d, scale, padded, mask, bias)
    on = [None if t is None else _dev(t, device) for t in (mask, bias)]
    for qb in (1, 2):
        ops.set_option("attention_qb", qb)
        try:
            g = ops.attention_f32(_dev(qkv, device), _dev(bi, device), B, S, heads, scale, padded_rows=padded, mask=on[0],
                                  bias=on[1]).cpu().numpy()
        finally:
            ops.set_option("attention_qb", -1)
        for b, n in enumerate(lens):
            r0, nq = (b * S, S) if padded else (bi[b], n)
            if n == 0:
                continue
            err = np.abs(g[r0:r0 + nq] - exp[r0:r0 + nq])
            assert err.max() <= 2e-5, (qb, b, err.max())


@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("lens,S,heads,d", [([70, 9, 33], 72, 2, 128), ([40, 33], 40, 4, 32),
                                            ([150, 64, 1], 160, 2, 96), ([64, 38], 64, 3, 64),
                                            ([33, 70], 70, 4, 16), ([100, 5], 100, 2, 80),
                                            ([64, 64], 64, 3, 8)])
def test_attention_generic_f16(device, lens, S, heads, d, padded, att_order):
    """The same kernel on fp16 tensors (head sizes the fp16 attention kernels do not take):
    inputs rounded to fp16, arithmetic in float, one fp16 rounding of the output."""
    _say("attention_generic_f16", lens, S, heads, d, padded)
    rs = np.random.RandomState(S + heads + d)
    B, H = len(lens), heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((B * S, 3 * H)).astype(np.float16)
    if not padded:
        qkv[bi[-1]:] = np.float16("nan")
    mask = None
    bias = (0.5 * rs.standard_normal((heads, S, S))).astype(np.float16)
    if padded:
        mask = (rs.rand(B, S, S) < 0.7).astype(np.float16)
        mask[:, :, 0] = 1
    scale = 1 / math.sqrt(d)
    exp = _naive_attention(qkv.astype(np.float32), lens, S, heads, d, scale, padded,
                           None if mask is None else mask.astype(np.float32),
                           bias.astype(np.float32))
    g = ops.attention_generic_f16(_dev(qkv, device), _dev(bi, device), B, S, heads, scale,
                                  padded_rows=padded,
                                  mask=None if mask is None else _dev(mask, device),
                                  bias=_dev(bias, device)).cpu().numpy()
    assert g.dtype == np.float16
    for b, n in enumerate(lens):
        r0, nq = (b * S, S) if padded else (bi[b], n)
        err = np.abs(g[r0:r0 + nq].astype(np.float64) - exp[r0:r0 + nq])
        assert np.all(err <= 2.0 ** -10 * np.abs(exp[r0:r0 + nq]) + 1e-4), (b, err.max())


@pytest.mark.parametrize("bits", [3, 10, 14, 20, 24])
@pytest.mark.parametrize("d", [32, 96, 128])
def test_attention_generic_f16_keeps_small_probabilities(device, d, bits):
    """One key takes nearly all of the probability and has V = 0; the rest share 1.3 * 2^-bits of it each, and are
    all that is in the result. Their probabilities are good to 2^-23 of themselves or 2^-38 of the largest one."""
    S, heads = 70, 2
    H = heads * d
    qkv = np.zeros((S, 3 * H), np.float16)
    qkv[:, 0:H:d] = 1                                        # Q: (1, 0, ...) in every head
    top = np.float16(bits * math.log(2) - math.log(1.3))     # ln of (largest / another)
    qkv[40, H:2 * H:d] = top                                 # K of the favoured key, in the first tile
    rs = np.random.RandomState(bits)
    qkv[:, 2 * H:] = (30000 + 20000 * rs.rand(S, H)).astype(np.float16)
    qkv[40, 2 * H:] = 0
    bi = np.array([0, S], np.int32)
    exp = _naive_attention(qkv.astype(np.float32), [S], S, heads, d, 1.0, False)
    g = ops.attention_generic_f16(_dev(qkv, device), _dev(bi, device), 1, S, heads, 1.0).cpu().numpy()
    # one fp16 rounding (normal or denormal), the probabilities, and the exponential's 2^-22
    bound = 2.0 ** -11 * np.abs(exp) + 2.0 ** -25 + np.abs(exp) * 2.0 ** -20 + S * 50000 * 2.0 ** -38
    assert exp.min() > 1e-3 and np.all(np.abs(g.astype(np.float64) - exp) <= bound), np.abs(g / exp - 1).max()


@pytest.mark.parametrize("d,S,lens", [(32, 300, [300, 77, 130]), (96, 128, [128, 65]), (128, 300, [300, 200]),
                                      (128, 1024, [1024])])
@pytest.mark.parametrize("sharp", [1.0, 4.0])
def test_attention_generic_f16_is_as_exact_as_float_arithmetic(device, d, S, lens, sharp):
    """Its distance from float64 is that of the float kernel on the same numbers with one rounding to fp16."""
    rs = np.random.RandomState(S + d)
    heads, B = 3, len(lens)
    H = heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((bi[-1], 3 * H)).astype(np.float16)
    qkv[:, :H] *= np.float16(sharp)
    args = _dev(bi, device), B, S, heads, 1 / math.sqrt(d)
    exp = _naive_attention(qkv.astype(np.float32), lens, S, heads, d, 1 / math.sqrt(d), False)
    got = ops.attention_generic_f16(_dev(qkv, device), *args).cpu().numpy().astype(np.float64) - exp
    wide = ops.attention_f32(_dev(qkv.astype(np.float32), device), *args).cpu().numpy()
    wide = wide.astype(np.float16).astype(np.float64) - exp
    rms = [float(np.sqrt((e ** 2).mean())) for e in (got, wide)]
    _say("generic attention: rms error %.4e, float kernel rounded to fp16 %.4e" % tuple(rms))
    assert rms[0] <= 1.002 * rms[1] and np.abs(got).max() <= 1.01 * np.abs(wide).max(), rms


@pytest.mark.parametrize("d", [48, 128])
def test_attention_generic_f16_passes_nan_on(device, d):
    """A NaN in Q, K or V reaches the outputs that depend on it and no others."""
    rs = np.random.RandomState(d)
    S, heads, lens = 150, 2, [150, 70, 130]
    H = heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((bi[-1], 3 * H)).astype(np.float16)
    want = np.zeros((bi[-1], H), bool)
    qkv[5, 3] = np.nan                              # Q of one query, head 0
    want[5, :d] = True
    qkv[150 + 69, H + d + 1] = np.nan               # K of the second sequence's last key, head 1
    want[150:220, d:] = True
    qkv[220 + 64, 2 * H + 7] = np.nan               # V of one key of the third sequence, column 7 of head 0
    want[220:, 7] = True
    g = ops.attention_generic_f16(_dev(qkv, device), _dev(bi, device), 3, S, heads, 1 / math.sqrt(d)).cpu().numpy()
    assert np.array_equal(np.isnan(g), want) and np.isfinite(g[~want]).all()


@pytest.mark.parametrize("scale", [-0.125, 0.0, -0.0, 1e-30, -3.0, 40.0])
@pytest.mark.parametrize("d", [32, 48, 96, 128])
@pytest.mark.parametrize("S,heads,lens", [(150, 2, [150, 64, 7, 130]), (70, 12, [70, 33, 64, 1, 66] * 22)])
def test_attention_generic_f16_takes_any_scale(device, scale, d, S, heads, lens):
    """Sequences that end inside a tile, scales that are negative, zero or next to it, and large; few
    workgroups and enough of them for 128-query tiles."""
    rs = np.random.RandomState(d)
    B, H = len(lens), heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((B * S, 3 * H)).astype(np.float16)
    bias = (0.5 * rs.standard_normal((heads, S, S))).astype(np.float16)
    for b in (None, bias):
        exp = _naive_attention(qkv.astype(np.float32), lens, S, heads, d, scale, False, None,
                               None if b is None else b.astype(np.float32))
        g = ops.attention_generic_f16(_dev(qkv, device), _dev(bi, device), B, S, heads, scale,
                                      bias=None if b is None else _dev(b, device)).cpu().numpy()
        # logits reach |scale| |q . k|, rounded to 2^-24 of themselves (and once more in the exponent)
        top = abs(scale) * 8 * d
        bound = 2.0 ** -10 * np.abs(exp[:bi[-1]]) + 1e-4 + 4 * 2.0 ** -24 * top
        err = np.abs(g[:bi[-1]].astype(np.float64) - exp[:bi[-1]])
        assert np.all(err <= bound), (scale, d, err.max())


@pytest.mark.parametrize("kind", ["mask", "bias", "both"])
@pytest.mark.parametrize("S,d", [(1, 64), (2, 64), (3, 128), (63, 64), (65, 64), (129, 64), (130, 32), (67, 128)])
def test_additive_terms_at_odd_lengths(device, S, d, kind):
    """Rows of the mask and of the bias start anywhere and end inside a tile: the 64-wide streaming
    kernel (with one and with two query blocks, and its key-split form) and the generic one."""
    rs = np.random.RandomState(S + d)
    heads, lens = 3, [S, max(1, S // 2)]
    B, H = len(lens), heads * d
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((B * S, 3 * H)).astype(np.float16)
    mask = bias = None
    if kind != "bias":
        mask = (rs.rand(B, S, S) < 0.6).astype(np.float16)
        mask[:, :, S // 2] = 1
    if kind != "mask":
        bias = rs.standard_normal((heads, S, S)).astype(np.float16)
    padded = mask is not None
    exp = _naive_attention(qkv.astype(np.float32), lens, S, heads, d, 0.125, padded,
                           None if mask is None else mask.astype(np.float32),
                           None if bias is None else bias.astype(np.float32))
    args = dict(padded_rows=padded, mask=None if mask is None else _dev(mask, device),
                bias=None if bias is None else _dev(bias, device))
    got = [ops.attention_generic_f16(_dev(qkv, device), _dev(bi, device), B, S, heads, 0.125, **args)]
    if d == 64:
        by_head = _dev(np.ascontiguousarray(qkv.reshape(B * S, 3, heads, d).transpose(1, 2, 0, 3)), device)
        for option, value in (("attention_qb", 1), ("attention_qb", 2), ("attention_key_split", 1)):
            ops.set_option(option, value)
            try:
                got.append(ops.attention_grouped(by_head, _dev(bi, device), B, S, 0.125, **args))
            finally:
                ops.set_option(option, -1)
    for i, g in enumerate(got):
        for b, n in enumerate(lens):
            r0, nq = (b * S, S) if padded else (bi[b], n)
            err = np.abs(g.cpu().numpy()[r0:r0 + nq].astype(np.float64) - exp[r0:r0 + nq])
            bound = 1e-4 if i == 0 else 2e-3   # (the 64-wide kernel rounds its probabilities to fp16)
            assert np.all(err <= 2.0 ** -10 * np.abs(exp[r0:r0 + nq]) + bound), (i, b, err.max())


@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("lens", [[32], [64], [128, 65], [127, 160], [256], [1024]])
def test_attention_f32_last_columns(device, d, lens):
    """Sequences whose last keys count in the last tile, so that the last product of a query's row changes every
    column: all columns are there, and the same in every run."""
    rs = np.random.RandomState(d)
    heads, S = 3, max(lens)
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((bi[-1], 3 * heads * d)).astype(np.float32)
    exp = _naive_attention(qkv, lens, S, heads, d, 1 / math.sqrt(d), False)
    runs = [ops.attention_f32(_dev(qkv, device), _dev(bi, device), len(lens), S, heads, 1 / math.sqrt(d))
            for _ in range(4)]
    assert all(torch.equal(r, runs[0]) for r in runs)
    err = np.abs(runs[0].cpu().numpy() - exp)
    assert err.max() <= 2e-5, (err.max(), np.unique(np.nonzero(err > 2e-5)[1]))


def test_attention_f32_rows_sum_and_uniform_keys(device):
    """V = const per column: the output is that constant times sum(P) = 1 / (1 + 1e-6 / sum e),
    whatever Q and K are; identical keys give a uniform P."""
    rs = np.random.RandomState(2)
    S, heads, d = 96, 2, 64
    H = heads * d
    lens = [96, 41]
    bi = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = rs.standard_normal((2 * S, 3 * H)).astype(np.float32)
    qkv[:, 2 * H:] = np.arange(H, dtype=np.float32)[None, :]
    g = ops.attention_f32(_dev(qkv, device), _dev(bi, device), 2, S, heads, 0.125).cpu().numpy()
    M = bi[-1]
    assert np.all(np.abs(g[:M] - np.arange(H)[None, :]) <= 2e-5 * (1 + np.arange(H))[None, :])


# ---- the whole layer -------------------------------------------------------------
def _f32_check(got, exp, lens, tag, pads_zero_required):
    mx, mean, pads_zero = O.parity_metrics(got, exp, lens)
    _say("parity %s: max-abs %.3e mean-abs %.3e pads_zero %s" % (tag, mx, mean, pads_zero))
    assert np.isfinite(got).all()
    assert mx <= F32_MAX_ABS and mean <= F32_MEAN_ABS, (mx, mean)
    if pads_zero_required:
        assert pads_zero


def _oracle32(wl, **kw):
    out = O.encoder(wl.x, wl.mask, wl.layers, wl.cfg.head_num, **kw)
    return O.masked_output(out.numpy(), wl.lens)


def _layers(wl, device, **kw):
    return [bt.BertEncoderLayer(wl.cfg.head_num, wl.cfg.head_size,
                                {k: _dev(v, device) for k, v in w.items()}, **kw)
            for w in wl.layers]


def test_cfg0_fp32_matches_the_committed_golden_output(device):
    """The stated fp32 configuration: B = 2 (padded path as in the reference), lengths
    [64, 38], against the oracle and the committed golden output of the same seed."""
    wl = workload.make_workload("cfg0")
    assert wl.x.dtype == np.float32
    got = bt.encoder_forward(_layers(wl, device), _dev(wl.x, device), _dev(wl.mask, device))
    got = O.masked_output(got.cpu().numpy(), wl.lens)
    _f32_check(got, _oracle32(wl), wl.lens, "cfg0/fp32/oracle", False)
    _f32_check(got, np.load(os.path.join(GOLDEN, "cfg0_out.npy")), wl.lens, "cfg0/fp32/golden", False)


@pytest.mark.parametrize("path", ["c_api", "th_op", "whole"])
@pytest.mark.parametrize("rm", [True, False])
def test_fp32_layers_all_paths(device, path, rm):
    _say("fp32 layers", path, rm)
    cfg = workload.EncoderConfig("f32", 5, 80, 4, layers=2, dtype="fp32", lens=(80, 3, 41, 0, 64))
    wl = workload.make_workload(cfg, bias_std=0.1, random_affine=True)
    exp = _oracle32(wl)
    x, m = _dev(wl.x, device), _dev(wl.mask, device)
    if path == "c_api":
        got = bt.encoder_forward(_layers(wl, device, is_remove_padding=rm), x, m)
    elif path == "th_op":
        bt.load_th_op()
        got = x
        for w in wl.layers:
            got = torch.ops.ByteTransformer.BertTransformer(
                cfg.head_num, cfg.head_size, *[_dev(w[n], device) for n in workload.WEIGHT_NAMES],
                got, m, rm, True)
    else:
        enc = bt.BertEncoder(cfg.head_num, cfg.head_size,
                             [{k: _dev(v, device) for k, v in w.items()} for w in wl.layers],
                             is_remove_padding=rm)
        got = enc(x, m)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    assert got.dtype == np.float32
    if rm:
        _f32_check(got, exp, wl.lens, "f32/%s/rm" % path, True)
    else:
        # an empty sequence has no defined rows on the padded path; compare the rest
        _f32_check(O.masked_output(got, wl.lens), exp, wl.lens, "f32/%s/padded" % path, False)


def test_fp32_attention_bias_tao_and_ffn_width(device):
    """attention_bias, a softmax temperature and intermediate_size = 2 through the float layer."""
    cfg = workload.EncoderConfig("f32b", 3, 48, 2, layers=1, ffn_mult=2, dtype="fp32",
                                 lens=(48, 20, 33))
    wl = workload.make_workload(cfg, bias_std=0.1, random_affine=True)
    bias = np.random.RandomState(4).standard_normal((2, 48, 48)).astype(np.float32)
    exp = O.masked_output(O.encoder_layer(wl.x, wl.mask, wl.layers[0], 2, tao=1.7,
                                          attention_bias=bias).numpy(), wl.lens)
    layer = bt.BertEncoderLayer(2, 64, {k: _dev(v, device) for k, v in wl.layers[0].items()},
                                tao=1.7)
    got = layer(_dev(wl.x, device), _dev(wl.mask, device), attention_bias=_dev(bias, device))
    _f32_check(got.cpu().numpy(), exp, wl.lens, "f32/bias+tao+ffn2", True)


def test_fp32_bert_base_shape_one_layer(device):
    """A BERT-base layer at batch 8 x 256 in float: big enough for the 128x128 GEMM tiles and
    several key tiles, small enough for the CPU oracle."""
    cfg = workload.EncoderConfig("f32base", 8, 256, 12, layers=1, dtype="fp32")
    wl = workload.make_workload(cfg)
    got = bt.encoder_forward(_layers(wl, device), _dev(wl.x, device), _dev(wl.mask, device))
    _f32_check(got.cpu().numpy(), _oracle32(wl), wl.lens, "f32/bert-base", True)


def test_fp32_dtype_mismatches_are_rejected(device):
    cfg = workload.EncoderConfig("e32", 3, 16, 2, layers=1, dtype="fp32", lens=(16, 3, 9))
    wl = workload.make_workload(cfg)
    layer = bt.BertEncoderLayer(2, 64, {k: _dev(v, device) for k, v in wl.layers[0].items()})
    with pytest.raises(RuntimeError, match="weights' dtype"):
        layer(_dev(wl.x, device).half(), _dev(wl.mask, device).half())
    mixed = {k: _dev(v, device) for k, v in wl.layers[0].items()}
    mixed["inter_bias"] = mixed["inter_bias"].half()
    with pytest.raises(ValueError, match="has dtype"):
        bt.BertEncoderLayer(2, 64, mixed)
