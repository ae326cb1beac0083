"""GPU parity of what an attention layer's training pass has beside its attention kernels, against float64 on the same stored
operands (models/aff_transformer.py:103-155 under autograd).

Bars, relative 2-norm: a result stored in 16 bits one rounding of it, 4e-4 fp16 and 3e-3 bf16; fp32 arithmetic on sums of up to 64
terms and an exponential 1e-6; position gradients, summed in double, 1e-6 of the sum of the terms' magnitudes.
"""
import pytest
import torch

from clusten import _native

pytestmark = pytest.mark.gpu

BAR = {torch.float16: 4e-4, torch.bfloat16: 3e-3, torch.float32: 1e-6}
DTYPES = list(BAR)


def near(got, ref, bar):
    assert got.shape == ref.shape and (got.double() - ref.double()).norm() <= bar * ref.double().norm()


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("b,h,n,m,rows,k", [(1, 1, 1, 4, 1, 1), (2, 3, 37, 48, 225, 5), (3, 16, 100, 48, 12321, 5), (1, 5, 1030, 12, 961, 3)])
def test_position_bias(device, dt, b, h, n, m, rows, k):
    gen = torch.Generator(device).manual_seed(n)
    table, w, bias = (torch.randn(*s, generator=gen, device=device) for s in ((rows, k), (h, k), (h,)))
    t64, w64 = table.to(dt).double(), w.to(dt).double()
    got, padded = _native.position_bias(table, w, bias, dt)
    near(got, (t64 @ w64.t() + bias.to(dt).double()).t(), BAR[dt])
    assert torch.equal(padded[:, :k], table.to(dt)) and not padded[:, k:].any()
    near(_native.position_bias(table, w, None, dt)[0], (t64 @ w64.t()).t(), BAR[dt])
    d = torch.randn(b, h, n, m, generator=gen, device=device).to(dt)
    pe = torch.randint(rows, (b, n, m), generator=gen, device=device)
    d_w, d_b = _native.position_grad(d, pe, padded, k)
    terms = d.double().unsqueeze(-1) * t64[pe].unsqueeze(1)
    assert ((d_w.double() - terms.sum((0, 2, 3))).abs() <= 1e-6 * terms.abs().sum((0, 2, 3)) / (b * n * m) ** 0.5).all()
    assert ((d_b.double() - d.double().sum((0, 2, 3))).abs() <= 1e-6 * d.double().abs().sum((0, 2, 3)) / (b * n * m) ** 0.5).all()


# one workgroup, two, the most and the most with values to spare; whole and partial groups of four heads
@pytest.mark.parametrize("b,h,n,m", [(1, 1, 128, 16), (1, 4, 129, 16), (2, 7, 21845, 48), (2, 5, 21900, 48)])
def test_position_gradient_workgroups(device, b, h, n, m):
    gen = torch.Generator(device).manual_seed(n)
    table = torch.randn(225, 5, generator=gen, device=device)
    _, padded = _native.position_bias(table, torch.randn(h, 5, device=device), None, torch.float16)
    d = torch.randn(b, h, n, m, generator=gen, device=device).half()
    pe = torch.randint(225, (b, n, m), generator=gen, device=device)
    d_w, d_b = _native.position_grad(d, pe, padded, 5)
    for head in range(h):
        terms = d[:, head].double().unsqueeze(-1) * padded.double()[pe][..., :5]
        assert ((d_w[head].double() - terms.sum((0, 1, 2))).abs() <= 1e-6 * terms.abs().sum((0, 1, 2)) / (b * n * m) ** 0.5).all()
        assert (d_b[head].double() - d[:, head].double().sum()).abs() <= 1e-6 * d[:, head].double().abs().sum() / (b * n * m) ** 0.5


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("b,h,n", [(1, 1, 1), (3, 2, 7), (2, 16, 49), (5, 3, 64), (1, 4, 63)])
def test_dense_attention(device, dt, b, h, n):
    gen = torch.Generator(device).manual_seed(n)
    c, rows, scale = 32 * h, 169, 32 ** -0.5

    def draw(*shape):
        return torch.randn(*shape, generator=gen, device=device)

    qkv, d_out = draw(b, n, 3 * c).to(dt), draw(b, n, c).to(dt)
    table, w, pe_b, bk, bv = draw(rows, 5), 0.3 * draw(h, 5), draw(h), draw(c), draw(c)
    pe = torch.randint(rows, (b, n, n), generator=gen, device=device)
    bias, padded = _native.position_bias(table, w, pe_b, dt)

    rows64, bias64, bk64, bv64 = (t.double().requires_grad_(True) for t in (qkv, bias, bk, bv))
    q = rows64[..., :c].view(b, n, h, 32).permute(0, 2, 1, 3)
    kv = rows64[..., c:].view(b, n, h, 2, 32).permute(3, 0, 2, 1, 4)
    logits = q @ kv[0].transpose(-1, -2) * scale + bias64.t()[pe].permute(0, 3, 1, 2)
    blank = (q * bk64.view(1, h, 1, 32)).sum(-1, keepdim=True) * scale
    p = torch.softmax(torch.cat([logits, blank], -1), -1)
    ref = (p[..., :-1] @ kv[1] + p[..., -1:] * bv64.view(1, h, 1, 32)).permute(0, 2, 1, 3).reshape(b, n, c)
    d_ref = torch.autograd.grad(ref, (rows64, bk64, bv64, bias64), d_out.double())

    near(_native.dense_attention_train(qkv, bias, pe, bk, bv, h, scale), ref.detach(), BAR[dt])
    got = _native.dense_attention_train_backward(qkv, bias, padded, pe, bk, bv, d_out, 5, h, scale)
    near(got[0], d_ref[0], BAR[dt])
    # of the keys' part too, which is the smallest
    near(got[0][..., c:], d_ref[0][..., c:], 2 * BAR[dt])
    if n > 1:                                                # with one token d_logit of a row is minus that of its blank token
        near(got[1], d_ref[1], 3e-6)
    near(got[2], d_ref[2], 3e-6)
    d_w, d_b = d_ref[3] @ padded[:, :5].double(), d_ref[3].sum(1)
    size = d_ref[3].abs().sum(1)
    assert ((got[3].double() - d_w).abs() <= 2e-6 * d_ref[3].abs() @ padded[:, :5].double().abs()).all()
    assert ((got[4].double() - d_b).abs() <= 2e-6 * size).all()


def test_exponential_of_fp32_global_attention(device):
    """Scores far below a row's maximum.  With q = 0 they are the table's values; token i sees the blank token (score 0, value 0) and one
    other at -40 - 0.789 i, so that its result is that exponential: one of 1 ulp (2^-23), a sum, a reciprocal and two products rounded
    once each, 2^-23 + 4 * 2^-24.  An exponential whose argument times log2 e is rounded is off by 3.4e-6."""
    n, h = 48, 2
    scores = torch.cat([torch.tensor([-1000.0]), -40 - 0.789 * torch.arange(n)]).to(device)
    pe, at = torch.zeros(1, n, n, dtype=torch.int64, device=device), torch.arange(n, device=device)
    pe[0, at, at] = at + 1
    qkv = torch.zeros(1, n, 96 * h, device=device)
    qkv[..., 32 * h:].view(1, n, h, 2, 32)[..., 1, :] = 1.0
    blank = torch.zeros(32 * h, device=device)
    out = _native.dense_attention_train(qkv, scores.expand(h, n + 1).contiguous(), pe, blank, blank, h, 1.0)
    ref = (scores[1:].double().exp() / (1 + scores[1:].double().exp())).view(1, n, 1)
    assert ((out.double() - ref).abs() <= 3 * 2 ** -23 * ref).all()


def test_position_gradient_of_global_attention_cancels(device):
    """Terms that cancel but for 2^-26 of them: uniform probabilities of 1/64 and powers of two, so that every product is exact and a sum in
    double is too.  Two images of 63 tokens; the large terms stand in rows that different waves add up."""
    n, table = 63, torch.zeros(64, 5)
    table[1, :2] = torch.tensor([1.0, 0.5])
    pe, qkv, d_out = torch.zeros(2, n, n, dtype=torch.int64), torch.zeros(2, n, 96), torch.zeros(2, n, 32)
    pe[:, :, 0] = 1
    qkv[:, 0, 64], qkv[:, 1, 64] = 1.0, -1.0
    d_out[:, 0, 0], d_out[:, 1, 0], d_out[:, 16, 0] = 2.0 ** 26, 1.0, -2.0 ** 26
    table, pe, qkv, d_out, blank = (t.to(device) for t in (table, pe, qkv, d_out, torch.zeros(32)))
    bias, padded = _native.position_bias(table, torch.zeros(1, 5, device=device), None, torch.float32)
    got = _native.dense_attention_train_backward(qkv, bias, padded, pe, blank, blank, d_out, 5, 1, 1.0)
    assert got[3].tolist() == [[2 / 64, 1 / 64, 0, 0, 0]] and got[4].tolist() == [0]


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("b,h,n,ch", [(1, 1, 8, 32), (2, 4, 100, 32), (3, 2, 203, 16), (1, 8, 777, 32), (2, 2, 64, 64)])
def test_rows_of_an_attention_layer(device, dt, b, h, n, ch):
    """Both scatters in one launch into the columns of d_qkv, against the scatters one by one."""
    gen = torch.Generator(device).manual_seed(n)
    c, m = h * ch, 8 * min(6, n // 8)
    qkv = torch.randn(b, n, 3 * c, generator=gen, device=device).to(dt)
    d_out = torch.randn(b, n, c, generator=gen, device=device).to(dt)
    probs, d_logit = (torch.randn(b, h, n, m, generator=gen, device=device).to(dt) for _ in range(2))
    d_blank, blank = torch.randn(b, h, n, generator=gen, device=device), torch.rand(b, h, n, generator=gen, device=device)
    numbers = torch.rand(b, n, (n + 7) // 8, generator=gen, device=device).argsort(-1)[..., :m // 8].int().contiguous()
    pairs = _native.cluster_pairs_from_numbers(numbers)
    d_qkv = torch.full_like(qkv, 7.0)
    d_bk, d_bv = _native.attention_rows_backward(qkv, d_qkv, probs, d_logit, d_out, d_blank, blank, pairs, 0.3)
    assert (d_qkv[..., :c] == 7.0).all()
    q, g = qkv[..., :c].view(b, n, h, ch).permute(0, 2, 1, 3), d_out.view(b, n, h, ch).permute(0, 2, 1, 3)
    d_k, d_v = _native.scatter_rows_by_cluster(d_logit, q, pairs), _native.scatter_rows_by_cluster(probs, g, pairs)
    kv = d_qkv[..., c:].view(b, n, h, 2, ch).permute(3, 0, 2, 1, 4)
    near(kv[0], 0.3 * d_k.double(), 2 * BAR[dt])
    assert torch.equal(kv[1], d_v)
    near(d_bk, 0.3 * (d_blank.double().unsqueeze(-1) * q.double()).sum((0, 2)).reshape(-1), 5e-6)
    near(d_bv, (blank.double().unsqueeze(-1) * g.double()).sum((0, 2)).reshape(-1), 5e-6)


# head shares of a cluster: all heads to one workgroup, and one each
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("b,h,n,ch", [(2, 2, 101, 32), (1, 8, 8, 16), (40, 2, 3999, 32)])
def test_rows_of_lists_that_are_not_whole_clusters(device, dt, b, h, n, ch):
    """A cluster number outside the sequence, and lists of any rows: NaN in every key and value column, nothing left as it was."""
    gen = torch.Generator(device).manual_seed(1)
    c, m = h * ch, 8
    qkv, d_out = torch.randn(b, n, 3 * c, generator=gen, device=device).to(dt), torch.randn(b, n, c, generator=gen, device=device).to(dt)
    probs, d_logit = (torch.randn(b, h, n, m, generator=gen, device=device).to(dt) for _ in range(2))
    blank = torch.rand(b, h, n, generator=gen, device=device)
    numbers = torch.randint((n + 7) // 8, (b, n, 1), generator=gen, device=device).int()
    numbers[-1, n // 2, 0] = (n + 7) // 8
    lists = torch.randint(n, (b, n, m), generator=gen, device=device)
    for pairs in (_native.cluster_pairs_from_numbers(numbers), _native.cluster_pairs(lists)):
        d_qkv = torch.full_like(qkv, 7.0)
        _native.attention_rows_backward(qkv, d_qkv, probs, d_logit, d_out, blank, blank, pairs, 0.3)
        assert (d_qkv[..., :c] == 7.0).all() and d_qkv[..., c:].isnan().all()


@pytest.mark.parametrize("b,n,n_out,m,rows,masked", [(1, 1, 1, 1, 1, False), (2, 50, 12, 48, 225, True), (3, 777, 194, 49, 12321, False)])
def test_merge_weights(device, b, n, n_out, m, rows, masked):
    gen = torch.Generator(device).manual_seed(n)
    table, prob = torch.randn(rows, 4, generator=gen, device=device), torch.rand(b, n, generator=gen, device=device)
    pe, idx = (torch.randint(k, (b, n_out, m), generator=gen, device=device) for k in (rows, n))
    mask = torch.randint(2, (b, n_out, m), generator=gen, device=device) if masked else None
    d = torch.randn(b, n_out, m, 4, generator=gen, device=device)
    d_table, d_prob = _native.merge_weights_backward(d, table, pe, idx, prob, mask)
    t64, p64 = table.double().requires_grad_(True), prob.double().requires_grad_(True)
    w = t64[pe] * p64.gather(1, idx.reshape(b, -1)).reshape(b, n_out, m, 1)
    w = w if mask is None else w * mask.unsqueeze(3)
    ref = torch.autograd.grad(w, (t64, p64), d.double())
    near(d_table, ref[0], 5e-7)
    near(d_prob, ref[1], 5e-7)


@pytest.mark.parametrize("dt,stream", [(torch.float16, torch.float16), (torch.float16, torch.float32), (torch.bfloat16, torch.float32),
                                       (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
@pytest.mark.parametrize("c,b,n", [(32, 1, 1), (64, 2, 16 * 1024 + 1), (128, 3, 99), (256, 1, 7), (512, 2, 2049)])
def test_row_score(device, dt, stream, c, b, n):
    gen = torch.Generator(device).manual_seed(n)
    x, w = torch.randn(b, n, c, generator=gen, device=device).to(stream), torch.randn(1, c, generator=gen, device=device) * c ** -0.5
    bias, d = torch.randn(1, generator=gen, device=device), torch.randn(b, n, 1, generator=gen, device=device).to(dt)
    score = _native.row_score(x, w, bias, dt)
    x64, w64 = x.to(dt).double(), w.to(dt).double()
    near(score, torch.sigmoid((x64 @ w64.t() + bias.to(dt).double()).to(dt).double()), 2 * BAR[dt])
    d_x, d_w, d_b = _native.row_score_backward(x, w, score, d)
    d_z = d.double() * score.double() * (1 - score.double())
    near(d_x, d_z * w64, BAR[stream])
    near(d_w, (d_z * x64).sum((0, 1)), 2e-6)
    assert (d_b.double() - d_z.sum()).abs() <= 2e-6 * d_z.norm()           # what a sum of such terms comes to, not this one


@pytest.mark.parametrize("columns", [True, False])
@pytest.mark.parametrize("b,n", [(1, 1), (3, 49), (2, 63), (2, 64), (2, 65)])
def test_global_attention_of_an_fp32_forward(device, b, n, columns):
    """q and kv as columns of one matrix, as the block kernels leave them, and as tensors of their own; up to 64 tokens are one kernel."""
    import copy
    from aff.model import ClusterAttention
    torch.manual_seed(n)
    attn = ClusterAttention(64, 2).to(device)
    with torch.no_grad():
        for p in attn.parameters():
            p.copy_(torch.randn_like(p) * 0.5)
    table, pe = torch.randn(169, 5, device=device), torch.randint(169, (b, n, n), device=device)
    qkv = torch.randn(b, n, 192, device=device)
    q, kv = (qkv[..., :64], qkv[..., 64:]) if columns else (qkv[..., :64].contiguous(), qkv[..., 64:].contiguous())
    everyone = torch.arange(n, device=device).expand(b, n, n)
    with torch.no_grad():
        got = attn.attend(q, kv, everyone, None, pe, True, table)
        ref = copy.deepcopy(attn).double().attend(q.double(), kv.double(), everyone, None, pe, True, table.double())
    near(got, ref, BAR[torch.float32])


# one row, a workgroup's, one more, several rows a thread
@pytest.mark.parametrize("rows", [1, 256, 1025, 12321])
@pytest.mark.parametrize("dt", DTYPES)
def test_merge_table(device, dt, rows):
    """Against float64 from the same rounded Linear layer: where a rounding falls the other way a value moves by one of dt, which the norm
    of four values can blow up, so that 16-bit bars are those of a rounding times ten.  Through the module besides, and differentiated twice."""
    from aff.model import _weight_table, default_ops
    gen = torch.Generator(device).manual_seed(rows)
    net = torch.nn.Sequential(torch.nn.Linear(5, 4), torch.nn.LayerNorm(4), torch.nn.GELU()).to(device)
    with torch.no_grad():
        for p in net.parameters():
            p.copy_(torch.randn(p.shape, generator=gen, device=device))
    table, d = torch.randn(rows, 5, generator=gen, device=device), torch.randn(rows, 4, generator=gen, device=device)
    params = (net[0].weight, net[0].bias, net[1].weight, net[1].bias)
    ref = [p.detach().to(dt if i < 2 else torch.float32).double().requires_grad_() for i, p in enumerate(params)]
    y = table.to(dt).double() @ ref[0].t() + ref[1]
    y = y + (y.to(dt).double() - y).detach()
    y = torch.nn.functional.gelu(torch.nn.functional.layer_norm(y, (4,), ref[2], ref[3], 1e-5))
    want = torch.autograd.grad(y, ref, d.double())
    bar = {torch.float32: 1e-5, torch.float16: 4e-3, torch.bfloat16: 3e-2}[dt]
    for create in (False, True):
        with torch.autocast("cuda", dtype=torch.float16 if dt == torch.float32 else dt, enabled=dt != torch.float32):
            out = _weight_table(net, table, default_ops())
        assert type(out.grad_fn).__name__ == "_MergeTableBackward"
        near(out, y.detach(), bar)
        for got, g in zip(torch.autograd.grad(out, params, d, create_graph=create), want):
            assert got.shape == g.shape and (got - g).norm() <= bar * max(g.norm(), (d.double().norm() ** 2 / 4) ** 0.5)


def test_merge_weights_of_neighbours_outside(device):
    """Neighbours that are no token: NaN where they stand, nothing read or written there, every other value as without them."""
    gen = torch.Generator(device).manual_seed(2)
    b, n, n_out, m, rows = 2, 50, 12, 48, 225
    table, prob = torch.randn(rows, 4, generator=gen, device=device), torch.rand(b, n, generator=gen, device=device)
    pe, idx = (torch.randint(k, (b, n_out, m), generator=gen, device=device) for k in (rows - 1, n))
    d = torch.randn(b, n_out, m, 4, generator=gen, device=device)
    bad = idx.clone()
    bad[0, 3, 5], bad[1, 11, 47], bad[1, 0, 0] = n, -1, 1 << 40
    out, pe_bad = bad != idx, pe.clone()
    pe_bad[out] = rows - 1                                       # a row of the table of their own
    got, want = _native.merge_weights(table, pe_bad, bad, prob, None), _native.merge_weights(table, pe_bad, idx, prob, None)
    assert got[out].isnan().all() and torch.equal(got[~out], want[~out])
    d_table, d_prob = _native.merge_weights_backward(d, table, pe_bad, bad, prob, None)
    masked = _native.merge_weights_backward(d, table, pe_bad, idx, prob, (~out).long())
    assert d_table[-1].isnan().all()
    near(d_table[:-1], masked[0][:-1], 5e-7)
    near(d_prob, masked[1], 5e-7)


def test_merge_weights_of_positions_outside(device):
    """Positions that are no row of the table: NaN where they stand and in their neighbour's gradient, nothing read there, every other
    value as without them."""
    gen = torch.Generator(device).manual_seed(3)
    b, n, n_out, m, rows = 2, 50, 12, 48, 225
    table, prob = torch.randn(rows, 4, generator=gen, device=device), torch.rand(b, n, generator=gen, device=device)
    pe, idx = (torch.randint(k, (b, n_out, m), generator=gen, device=device) for k in (rows, n - 1))
    d = torch.randn(b, n_out, m, 4, generator=gen, device=device)
    bad = pe.clone()
    bad[0, 3, 5], bad[1, 11, 47], bad[1, 0, 0] = rows, -1, 1 << 40
    out = bad != pe
    idx[out] = n - 1                                             # a neighbour of their own
    got, want = _native.merge_weights(table, bad, idx, prob, None), _native.merge_weights(table, pe, idx, prob, None)
    assert got[out].isnan().all() and torch.equal(got[~out], want[~out])
    d_table, d_prob = _native.merge_weights_backward(d, table, bad, idx, prob, None)
    masked = _native.merge_weights_backward(d, table, pe, idx, prob, (~out).long())
    assert d_prob[:, -1].isnan().all()
    near(d_prob[:, :-1], masked[1][:, :-1], 5e-7)
    near(d_table, masked[0], 5e-7)


def merging(device, n=48, c=32):
    """A merge of n tokens that all see each other: the module, scores, and its forward on given scores and mask."""
    from aff.model import ClusterMerging, default_ops, relative_position_table
    gen = torch.Generator(device).manual_seed(n)
    torch.manual_seed(n)
    merge = ClusterMerging(c, 2 * c, ops=default_ops()).to(device)
    table = relative_position_table(64)[0].to(device)
    at = torch.arange(n, device=device)
    pos = torch.stack([at % 7, at // 7], 1).float().expand(2, n, 2).contiguous()
    everyone = at.expand(2, n, n).contiguous()
    pe = torch.randint(table.shape[0], (2, n, n), generator=gen, device=device)
    feat, score = torch.randn(2, n, c, generator=gen, device=device), torch.rand(2, n, 1, generator=gen, device=device)

    def call(score, mask=None, module=merge, positions=torch.int64):
        return module(pos, feat, everyone, mask, score, 4, pe.to(positions), 0, table)[1]
    return merge, score, call


def test_merge_of_strided_scores(device):
    """Scores that are a column of wider rows, in training: the gradients of the same scores in rows of their own, but for the order of
    the atomic additions (48 terms a score, 1e-6 of them)."""
    merge, score, call = merging(device)
    results = []
    for s in (score, torch.cat([score, score + 1, score], 2)[..., :1]):
        s = s.detach().requires_grad_()
        results.append(torch.autograd.grad(call(s).square().sum(), [s, *merge.parameters()]))
    for a, b in zip(*results):
        near(a, b, 1e-5)


def test_merge_of_narrow_positions(device):
    """Positions in 32 bits, which the recorded lookup takes and the kernel does not, in training."""
    merge, score, call = merging(device)
    results = []
    for dt in (torch.int64, torch.int32):
        s = score.clone().requires_grad_()
        results.append(torch.autograd.grad(call(s, positions=dt).square().sum(), [s, *merge.parameters()]))
    for a, b in zip(*results):
        near(a, b, 1e-5)


def layered(merge):
    """The same merge, its weights by recorded operations."""
    import copy
    other = copy.deepcopy(merge)
    other.ops = type(other.ops)(**{**vars(other.ops), "merge_weights": None})
    return other


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.float64])
def test_merge_with_a_mask_of_fractions(device, dt):
    """A mask that is no table of 0 and 1, in inference and in training, as a constant and as what takes a gradient itself."""
    merge, score, call = merging(device)
    mask = torch.rand(2, 48, 48, generator=torch.Generator(device).manual_seed(1), device=device).to(dt)
    with torch.no_grad():
        near(call(score, mask), call(score, mask.float(), layered(merge)), 1e-5)
    results = []
    for module in (merge, layered(merge)):
        s, m = score.clone().requires_grad_(), mask.float().requires_grad_()
        constant = mask if module is merge else mask.float()
        results.append(torch.autograd.grad(call(s, constant, module).square().sum(), [s, *module.parameters()])
                       + torch.autograd.grad(call(s, m, module).square().sum(), [m, s]))
    for a, b in zip(*results):
        near(a, b, 1e-5)


def test_merge_under_deterministic_algorithms(device):
    """The scores' gradient is made of atomic additions: not where the caller asked for the same bits every time."""
    merge, score, call = merging(device)
    s, routes, grads = score.clone().requires_grad_(), [], []
    for _ in range(2):
        torch.use_deterministic_algorithms(True, warn_only=True)
        try:
            out = call(s)
            grads.append(torch.autograd.grad(out.square().sum(), s, retain_graph=True)[0])
        finally:
            torch.use_deterministic_algorithms(False)
        routes.append([f for f in walk(out.grad_fn) if type(f).__name__ == "_MergeWeightsBackward"])
    assert not any(routes) and torch.equal(*grads)
    out = call(s)
    assert any(type(f).__name__ == "_MergeWeightsBackward" for f in walk(out.grad_fn))


def walk(node):
    seen, todo = set(), [node]
    while todo:
        f = todo.pop()
        if f is not None and f not in seen:
            seen.add(f)
            todo += [g for g, _ in f.next_functions]
    return seen
