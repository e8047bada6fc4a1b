"""The first LayerNorm in FFN1's launch: against float64, and where its rows and tiles can go wrong."""
import pytest
import torch

import bytetransformer_amd as bt
from bytetransformer_amd import ops

pytestmark = pytest.mark.gpu

EPS = 1e-6


def _exact(src, residual, bias, gamma, beta, w, ffn_bias):
    """The layer's steps: two adds rounded to half, statistics and results in float64, the rows rounded to half once."""
    x = ((src + residual) + bias).double()
    rows = (x - x.mean(1, keepdim=True)) / (x.var(1, unbiased=False, keepdim=True) + EPS).sqrt() * gamma.double() + beta.double()
    return rows, torch.nn.functional.gelu(rows.half().double() @ w.double() + ffn_bias.double(), approximate="tanh")


def _run(rows, hidden, n, kn, live=None, gather=False, all_live=None):
    gen = torch.Generator(device="cuda").manual_seed(rows * 7 + hidden + n)

    def normal(*shape, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=gen)

    src, residual, bias = normal(rows, hidden), normal(rows, hidden), normal(hidden, std=0.1)
    gamma, beta, w, ffn_bias = normal(hidden, std=0.1, mean=1.0), normal(hidden, std=0.1), normal(hidden, n, std=0.02), normal(n, std=0.1)
    m = rows if live is None else live
    count = None if live is None else torch.tensor([live], dtype=torch.int32, device="cuda")
    index = torch.randperm(rows, generator=gen, device="cuda").int() if gather else None
    before = torch.full((rows, hidden), 7.0, dtype=torch.float16, device="cuda"), torch.full((rows, n), 7.0, dtype=torch.float16, device="cuda")
    got, out = ops.layernorm_gemm_bias_gelu(
        src, residual, bias, gamma, beta, w if kn else w.t().contiguous(), ffn_bias, eps=EPS, valid_rows=count,
        residual_row_index=index, all_live=live is None if all_live is None else all_live, w_kn=kn, dst=before[0], out=before[1])
    if m:
        want = _exact(src[:m], residual[index[:m].long()] if gather else residual[:m], bias, gamma, beta, w, ffn_bias)
        # half's rounding, 2^-11 of a value, and 2^-20 for the float sums behind it (values up to about 6)
        assert ((got[:m].double() - want[0]).abs() <= want[0].abs() * 2 ** -11 + 2 ** -18).all()
        # a row that rounds the other way moves a product of 1024 terms of 0.02 by less than 2^-11 * 6 * 0.02 * sqrt(1024) * 5
        assert (out[:m].double() - want[1]).abs().max().item() <= 2e-2
        err = (out[:m].double() - want[1]).norm() / want[1].norm()
        assert err.item() <= 2 ** -11
    assert (got[m:] == 7).all() and (out[m:] == 7).all(), "rows past the live ones are not written"
    return got, out


@pytest.mark.parametrize("hidden,rows,kn", [(768, r, True) for r in (1, 15, 16, 17, 32, 33, 64, 79, 80)] +
                         [(768, r, False) for r in (1, 16, 17, 32)] + [(1024, r, True) for r in (1, 32, 33, 64)] +
                         [(1024, r, False) for r in (15, 32)])
def test_rows(hidden, rows, kn):
    """Both widths of tile at both ends of their rows, remainders of 16."""
    assert ops.layernorm_gemm_bias_gelu_pays(rows, True, 4 * hidden, hidden, w_kn=kn)
    _run(rows, hidden, 4 * hidden, kn)


@pytest.mark.parametrize("kn,rows", [(True, 111), (False, 44)])
@pytest.mark.parametrize("share", [0.0, 0.01, 0.6, 1.0])
def test_live_rows_on_the_device(rows, kn, share):
    """A padded batch, its residual gathered, up to more live rows than one round of the chip has."""
    assert ops.layernorm_gemm_bias_gelu_pays(rows, False, 3072, 768, w_kn=kn)
    _run(rows, 768, 3072, kn, live=int(-(-rows * share // 1)), gather=True)


@pytest.mark.parametrize("kn,rows", [(True, 80), (True, 64), (False, 32)])
@pytest.mark.parametrize("live", [0, 1, 31])
def test_fewer_live_rows_than_vouched_for(rows, kn, live):
    """A caller's count decides the tile, the device's what is computed."""
    assert ops.layernorm_gemm_bias_gelu_pays(rows, True, 3072, 768, w_kn=kn)
    _run(rows, 768, 3072, kn, live=live, gather=True, all_live=True)


@pytest.mark.parametrize("n", [768, 1536])
def test_narrow_products(n):
    for kn in (True, False):
        _run(30, 768, n, kn)


def test_both_layouts_give_the_same_bits():
    a, b = _run(30, 768, 3072, True), _run(30, 768, 3072, False)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def _two_launches(rows, hidden, n, kn, live=None, gather=False):
    """The inputs of _run through the LayerNorm's launch and FFN1's."""
    gen = torch.Generator(device="cuda").manual_seed(rows * 7 + hidden + n)

    def normal(*shape, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=gen)

    src, residual, bias = normal(rows, hidden), normal(rows, hidden), normal(hidden, std=0.1)
    gamma, beta, w, ffn_bias = normal(hidden, std=0.1, mean=1.0), normal(hidden, std=0.1), normal(hidden, n, std=0.02), normal(n, std=0.1)
    count = None if live is None else torch.tensor([live], dtype=torch.int32, device="cuda")
    index = torch.randperm(rows, generator=gen, device="cuda").int() if gather else None
    ops.add_bias_residual_layernorm(src, residual, bias, gamma, beta, eps=EPS, valid_rows=count, residual_row_index=index)
    return src, ops.gemm_bias_gelu(src, w if kn else w.t().contiguous(), ffn_bias, valid_rows=count, w_kn=kn)


@pytest.mark.parametrize("rows,live", [(1, None), (16, None), (31, None), (32, None), (33, None), (64, None), (65, None), (80, None),
                                       (44, 17), (64, 40), (88, 50), (111, 67), (111, 111)])
@pytest.mark.parametrize("hidden,n", [(768, 3072), (768, 1024), (1024, 4096), (1024, 1024)])
@pytest.mark.parametrize("kn", [True, False])
def test_bits_of_the_two_launches(hidden, n, kn, rows, live):
    """Sums in the order of the product that these sizes would get: four slices of k where that is tile 14 (at 3072 columns up
    to 64 rows of capacity), one chain beyond."""
    if not ops.layernorm_gemm_bias_gelu_pays(rows, live is None, n, hidden, w_kn=kn):
        pytest.skip("two launches at these sizes")
    gather = live is not None
    got, want = _run(rows, hidden, n, kn, live, gather), _two_launches(rows, hidden, n, kn, live, gather)
    m = rows if live is None else live
    assert torch.equal(got[0][:m], want[0][:m]) and torch.equal(got[1][:m], want[1][:m])


def test_sizes_that_keep_two_launches():
    for rows, n, k, kn in ((81, 3072, 768, True), (33, 3072, 768, False), (65, 4096, 1024, True), (33, 4096, 1024, False),
                           (32, 2048, 512, True), (32, 800, 768, True), (32, 3072, 640, True)):
        assert not ops.layernorm_gemm_bias_gelu_pays(rows, True, n, k, w_kn=kn)
    x = torch.zeros(8, 640, dtype=torch.float16, device="cuda")
    v = torch.zeros(640, dtype=torch.float16, device="cuda")
    with pytest.raises(ops.BtError):
        ops.layernorm_gemm_bias_gelu(x, x, v, v, v, torch.zeros(640, 2560, dtype=torch.float16, device="cuda"),
                                     torch.zeros(2560, dtype=torch.float16, device="cuda"), w_kn=True)


@pytest.mark.parametrize("batch,seq_len", [(1, 32), (1, 72), (3, 14), (4, 25)])
def test_weight_copies_change_no_bit(batch, seq_len):
    """Never, always and the table's choice of copies, on padded and on packed rows."""
    bt.load_th_op()
    gen = torch.Generator(device="cuda").manual_seed(seq_len)

    def normal(*shape, std=0.02, mean=0.0):
        return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=gen)

    H = 768
    w = [normal(H, 3 * H), normal(3 * H), normal(H, H), normal(H), normal(H, std=0.05, mean=1.0), normal(H), normal(H, 4 * H), normal(4 * H),
         normal(4 * H, H), normal(H), normal(H, std=0.05, mean=1.0), normal(H)]
    x = normal(batch, seq_len, H, std=1.0)
    lens = torch.arange(seq_len, 0, -(seq_len // batch), device="cuda")[:batch]
    mask = (torch.arange(seq_len, device="cuda")[None, None, :] < lens[:, None, None]).half().expand(batch, seq_len, seq_len).contiguous()
    got = []
    try:
        for choice in (0, 1, -1):
            ops.set_option("layer_prepack", choice)
            got.append(torch.ops.ByteTransformer.BertTransformer(12, 64, *w, x, mask, True, True))
    finally:
        ops.set_option("layer_prepack", -1)
    assert got[0].isfinite().all() and torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


def _layer_inputs(batch, seq_len, H=768):
    gen = torch.Generator(device="cuda").manual_seed(seq_len)

    def normal(*shape, std=0.02, mean=0.0):
        return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=gen)

    w = [normal(H, 3 * H), normal(3 * H), normal(H, H), normal(H), normal(H, std=0.05, mean=1.0), normal(H), normal(H, 4 * H), normal(4 * H),
         normal(4 * H, H), normal(H), normal(H, std=0.05, mean=1.0), normal(H)]
    x = normal(batch, seq_len, H, std=1.0)
    lens = torch.arange(seq_len, 0, -(seq_len // batch), device="cuda")[:batch]
    mask = (torch.arange(seq_len, device="cuda")[None, None, :] < lens[:, None, None]).half().expand(batch, seq_len, seq_len).contiguous()
    return w, x, mask


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("batch,seq_len", [(1, 32), (1, 72), (1, 200)])
def test_ffn1_bias_inside_a_buffer(batch, seq_len, packed):
    """A bias that starts 8 bytes into a flat parameter buffer, on both sides of the rows that this launch takes."""
    bt.load_th_op()
    w, x, mask = _layer_inputs(batch, seq_len)
    want = torch.ops.ByteTransformer.BertTransformer(12, 64, *w, x, mask, packed, True)
    flat = torch.zeros(w[7].numel() + 4, dtype=torch.float16, device="cuda")
    flat[4:] = w[7]
    w[7] = flat[4:]
    assert w[7].data_ptr() % 16 == 8
    assert torch.equal(torch.ops.ByteTransformer.BertTransformer(12, 64, *w, x, mask, packed, True), want)
