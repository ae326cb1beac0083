"""GPU parity of a block's backward: the kernels between its products (`clusten_gelu_backward`, `clusten_norm_backward`,
`clusten_kv_columns`, `clusten_blank_grad`, `clusten_table_linear_grad`) against float64, and training passes of whole models
through the block kernels against the same models layer by layer (models/aff_transformer.py:181-232).

Bars of the kernels, max|got - ref| / max|ref|: results stored in 16 bits half a unit in the last place and a little for the
fp32 arithmetic ahead of it, 6e-4 fp16 and 5e-3 bf16; fp32 results 2e-6, sums over the rows 1e-5 (fp32 sums of up to 2e4 terms in
some hundred partial sums).
"""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from aff.model import AutoFocusFormer, BasicLayer, ClusterTransformerBlock, default_ops, relative_position_table
from clusten import _native

pytestmark = pytest.mark.gpu

BAR = {torch.float16: 6e-4, torch.bfloat16: 5e-3, torch.float32: 2e-6}
DTYPES = list(BAR)


def close(got, ref, bar):
    ref = ref.double()
    assert got.shape == ref.shape
    assert (got.double() - ref).abs().max() <= bar * ref.abs().max().clamp(min=1e-30)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("count", [8, 2040, 2056, 100_000])
def test_gelu_backward(device, dt, count):
    gen = torch.Generator(device).manual_seed(count)
    h = (3 * torch.randn(count, generator=gen, device=device)).to(dt)
    d = torch.randn(count, generator=gen, device=device).to(dt)
    x = h.double().requires_grad_(True)
    ref = F.gelu(x)
    ref_d, = torch.autograd.grad(ref, x, d.double())
    g, d_h = _native.gelu_backward(h, d.clone())
    close(g, ref.detach(), BAR[dt])
    close(d_h, ref_d, BAR[dt])


def test_gelu_backward_in_the_tail(device):
    """Where the derivative is small its relative error is that of rounding it to bf16, 2^-8, and a little: fp32 arithmetic with an
    exponent of up to 72 leaves 1e-5."""
    h = torch.linspace(-12, -1.5, 4096, device=device).to(torch.bfloat16)
    x = h.double()
    cdf = 0.5 * torch.erfc(-x * 0.5 ** 0.5)
    ref = cdf + x * torch.exp(-0.5 * x * x) / (2 * torch.pi) ** 0.5
    g, d_h = _native.gelu_backward(h, torch.ones_like(h))
    assert ((d_h.double() - ref).abs() <= (2 ** -8 + 2e-5) * ref.abs()).all()
    ref = x * cdf
    assert ((g.double() - ref).abs() <= (2 ** -8 + 2e-5) * ref.abs()).all()


@pytest.mark.parametrize("dt,stream", [(torch.float16, torch.float16), (torch.float16, torch.float32),
                                       (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("c,b,n", [(32, 1, 1), (32, 3, 1021), (64, 2, 16 * 1024 + 3), (128, 3, 333), (256, 1, 7), (512, 2, 2051)])
def test_norm_backward(device, dt, stream, c, b, n):
    gen = torch.Generator(device).manual_seed(c + n)

    def draw(*shape):
        return torch.randn(*shape, generator=gen, device=device)

    x, d_y, d_res = (1 + 2 * draw(b, n, c)).to(stream), draw(b, n, c).to(dt), draw(b, n, c).to(stream)
    w, scale = 1 + 0.2 * draw(c), torch.tensor([1.25, 0.0, 2.0][:b], device=device)
    x64 = x.double().requires_grad_(True)
    w64, b64 = w.double().requires_grad_(True), torch.zeros(c, device=device, dtype=torch.float64, requires_grad=True)
    ref = torch.autograd.grad(F.layer_norm(x64, (c,), w64, b64), (x64, w64, b64), d_y.double())
    mean = x.double().mean(-1)
    stats = torch.stack([mean, (x.double().var(-1, unbiased=False) + 1e-5).rsqrt()], -1).float().reshape(-1, 2).contiguous()
    d_x, branch, d_w, d_b = _native.norm_backward(d_y, x, stats, w, d_res, True, scale)
    close(d_x, ref[0] + d_res.double(), BAR[stream])
    close(branch, d_x.double() * scale.double().view(b, 1, 1), BAR[dt])
    close(d_w, ref[1], 1e-5)
    close(d_b, ref[2], 1e-5)
    d_x, branch, _, _ = _native.norm_backward(d_y, x, stats, w)
    close(d_x, ref[0], BAR[stream])
    assert branch is None


# a row tile, two of them, more tiles than workgroups (1024), last ones partly filled
ROWS = [(32, 64, 1, 1), (32, 96, 3, 11), (64, 192, 2, 16 * 1024 + 5), (128, 384, 1, 4097), (128, 256, 3, 33), (256, 768, 1, 49),
        (256, 512, 2, 2100), (512, 1536, 1, 15), (512, 512, 3, 1400)]
# relative 2-norm: one rounding of a result (a third of the bar in the mean) and what d_h rounded on its way does to a sum
NORM_BAR = {torch.float16: 5e-4, torch.bfloat16: 4e-3, torch.float32: 6e-7}


@pytest.mark.parametrize("dt,stream", [(torch.float16, torch.float16), (torch.float16, torch.float32),
                                       (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
@pytest.mark.parametrize("c,hidden,b,n", ROWS)
@pytest.mark.parametrize("scaled", [False, True])
def test_block_backward_over_rows(device, dt, stream, c, hidden, b, n, scaled):
    """The two kernels of a block's backward against float64 on the same stored operands."""
    gen = torch.Generator(device).manual_seed(c + n)

    def draw(*shape, scale=1.0):
        return torch.randn(*shape, generator=gen, device=device) * scale

    w_p, w_1, w_2 = draw(c, c, scale=c ** -0.5), draw(hidden, c, scale=c ** -0.5), draw(c, hidden, scale=hidden ** -0.5)
    w_q, w_kv = draw(c, c, scale=c ** -0.5), draw(2 * c, c, scale=c ** -0.5)
    packed, at = _native.block_pack(c, dt, [(w, True) for w in (w_p, w_1, w_2, w_q, w_kv)])
    x, d_out, d_y = (draw(b, n, c) + 0.5).to(stream), draw(b, n, c).to(stream), draw(b, n, 3 * c).to(dt)
    h, norm_w = draw(b, n, hidden).to(dt), 1 + 0.2 * draw(c)
    scale = draw(2, b).abs().to(dt).float() if scaled else None
    x64, w64, zero = x.double().requires_grad_(True), norm_w.double().requires_grad_(True), torch.zeros(c, device=device).double()
    b64 = zero.clone().requires_grad_(True)
    norm = F.layer_norm(x64, (c,), w64, b64)
    mean = x.double().mean(-1)
    stats = torch.stack([mean, (x.double().var(-1, unbiased=False) + 1e-5).rsqrt()], -1).float().reshape(-1, 2).contiguous()

    def as_stored(t):
        return t.to(dt).double()

    def near(got, ref, bar=NORM_BAR[dt]):
        assert got.shape == ref.shape and (got.double() - ref).norm() <= bar * ref.norm()

    got = _native.block_tail_backward(d_out, x, stats, norm_w, h, packed, at[:3], scale)
    d_f = as_stored(as_stored(d_out) * (1.0 if scale is None else scale[1].double().view(b, 1, 1)))
    h64 = h.double().requires_grad_(True)
    g = F.gelu(h64)
    d_h = as_stored(torch.autograd.grad(g, h64, d_f @ as_stored(w_2))[0])
    grads = torch.autograd.grad(norm, (x64, w64, b64), d_h @ as_stored(w_1), retain_graph=True)
    d_x = (d_out.double() + grads[0]).to(stream).double()
    branch = as_stored(d_x * (1.0 if scale is None else scale[0].double().view(b, 1, 1)))
    for t, ref in zip(got, (d_x, branch, d_f, g.detach(), d_h, branch @ as_stored(w_p))):
        near(t, ref)
    for t, ref in zip(got[6:], grads[1:]):
        near(t, ref, max(NORM_BAR[dt], 2e-6))

    for d_res in (None, d_out):
        got = _native.norm_linear_backward(d_y, x, stats, norm_w, packed, at[3:], d_res)
        grads = torch.autograd.grad(norm, (x64, w64, b64), d_y.double() @ as_stored(torch.cat([w_q, w_kv])), retain_graph=True)
        near(got[0], grads[0] if d_res is None else grads[0] + d_res.double(), NORM_BAR[stream])
        for t, ref in zip(got[1:], grads[1:]):
            near(t, ref, 2e-6)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("b,h,n,ch", [(1, 1, 1, 32), (2, 2, 777, 32), (3, 4, 100, 8), (2, 16, 259, 32)])
def test_attention_columns(device, dt, b, h, n, ch):
    gen = torch.Generator(device).manual_seed(n)
    c = h * ch

    def draw(*shape):
        return torch.randn(*shape, generator=gen, device=device)

    qkv, d_out, d_k, d_v = draw(b, n, 3 * c).to(dt), draw(b, n, c).to(dt), draw(b, h, n, ch).to(dt), draw(b, h, n, ch).to(dt)
    d_blank, prob = draw(b, h, n), draw(b, h, n)
    d_qkv = torch.full((b, n, 3 * c), 7.0, device=device, dtype=dt)
    d_bk, d_bv = _native.attention_columns_backward(qkv, d_qkv, d_k, d_v, d_out, d_blank, prob, 0.3)
    kv = torch.stack([0.3 * d_k.double(), d_v.double()], 3).permute(0, 2, 1, 3, 4).reshape(b, n, 2 * c)
    assert (d_qkv[..., :c] == 7.0).all()
    close(d_qkv[..., c:], kv, BAR[dt])
    q = qkv[..., :c].double().view(b, n, h, ch)
    close(d_bk, 0.3 * (d_blank.double().permute(0, 2, 1)[..., None] * q).sum((0, 1)).reshape(-1), 1e-5)
    close(d_bv, (prob.double().permute(0, 2, 1)[..., None] * d_out.double().view(b, n, h, ch)).sum((0, 1)).reshape(-1), 1e-5)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("rows,n,k", [(1, 1, 1), (1023, 3, 5), (12321, 16, 5), (1025, 2, 8)])
def test_table_linear_grad(device, dt, rows, n, k):
    gen = torch.Generator(device).manual_seed(rows)
    d, x = torch.randn(rows, n, generator=gen, device=device), torch.randn(rows, k, generator=gen, device=device).to(dt)
    d_w, d_b = _native.table_linear_grad(d, x)
    close(d_w, d.double().t() @ x.double(), 1e-5)
    close(d_b, d.double().sum(0), 1e-5)


def build(ops, device, drop_path=0.0, nbhd_size=(48, 48, 48, 48)):
    """A model of as many stages as `nbhd_size` has, on 576, 144, 36 and 9 tokens."""
    torch.manual_seed(5)
    k = len(nbhd_size)
    kw = dict(img_size=96, embed_dim=(32, 64, 128, 256)[:k], num_heads=(1, 2, 4, 8)[:k], depths=(1, 2, 2, 1)[:k], mlp_ratio=2.0,
              cluster_size=8, nbhd_size=nbhd_size, num_classes=40, drop_path_rate=drop_path)
    return AutoFocusFormer(ops=ops, **kw).to(device)


def step(net, dt, device, seed=3):
    gen = torch.Generator(device).manual_seed(seed)
    images = torch.randn(3, 3, 96, 96, generator=gen, device=device)
    labels = torch.randint(40, (3,), generator=gen, device=device)
    torch.manual_seed(9)
    with torch.autocast("cuda", dtype=torch.float16 if dt == torch.float32 else dt, enabled=dt != torch.float32):
        logits = net(images)
        loss = F.cross_entropy(logits.float(), labels)
    net.zero_grad(set_to_none=True)
    (loss * (1.0 if dt == torch.float32 else 1024.0)).backward()
    return logits.detach(), {name: p.grad for name, p in net.named_parameters()}


def norm_error(got, ref):
    got, ref = got.detach(), ref.detach()
    return float((got.double() - ref.double()).norm() / ref.double().norm().clamp(min=1e-30))


# Two orders of the same sums and roundings: about four times the largest relative difference seen, of the logits and of all
# gradients together (2.5e-7, 5.4e-4, 3.5e-3) and of a single parameter's (3.8e-6, 1.8e-3, 2.7e-2).
BARS = {torch.float32: (1e-6, 1.5e-5), torch.float16: (2e-3, 8e-3), torch.bfloat16: (1.5e-2, 0.1)}
# Gradients that are nearly nothing are measured by that of their layer's weight: a bias ahead of a BatchNorm (exactly 0), and
# of the score that only weighs a token against its neighbours.
CANCELS = ("patch_embed.proj1.bias", "prob_net.bias")


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("drop_path", [0.0, 0.4])
def test_training_step_layer_by_layer(device, dt, drop_path):
    ops = default_ops()
    layered = SimpleNamespace(**{**vars(ops), "block_tail": None})
    # in bf16 with local lists in every stage (the third: 24 of 36 tokens): the attention of a global one is the framework's batched
    # products, which are not to be given transposed operands of that type
    nbhd_size = (48, 48, 24) if dt == torch.bfloat16 else (48, 48, 48, 48)
    got, got_grads = step(build(ops, device, drop_path, nbhd_size).train(), dt, device)
    ref, ref_grads = step(build(layered, device, drop_path, nbhd_size).train(), dt, device)
    together, single = BARS[dt]
    assert norm_error(got, ref) < together
    everything = torch.cat([g.reshape(-1) for g in got_grads.values()])
    assert norm_error(everything, torch.cat([g.reshape(-1) for g in ref_grads.values()])) < together
    for name, g in ref_grads.items():
        assert got_grads[name].dtype == g.dtype
        by = ref_grads[name[:-4] + "weight"] if name.endswith(CANCELS) else g
        assert (got_grads[name].double() - g.double()).norm() <= single * by.double().norm(), name


def dense_block(device, ops=None, c=64, h=2):
    torch.manual_seed(2)
    blk = ClusterTransformerBlock(c, h, ops=ops or default_ops()).to(device)
    feat = torch.randn(2, 36, c, device=device)
    table = torch.randn(121, 5, device=device)
    pe_idx = torch.randint(121, (2, 36, 36), device=device)
    return blk, feat, lambda x: blk(x, None, None, pe_idx, True, table)


def test_second_derivatives_and_frozen_parameters(device):
    blk, feat, call = dense_block(device)
    ref_blk, _, ref_call = dense_block(device, SimpleNamespace(**{**vars(default_ops()), "block_tail": None}))

    def penalty(call, blk):
        x = feat.clone().requires_grad_(True)
        out, branch = call(x)
        out = out if branch is None else out + branch
        g, = torch.autograd.grad(out.square().sum(), x, create_graph=True)
        return torch.autograd.grad(g.square().sum(), [x, blk.mlp.fc1.weight, blk.attn.q.weight])

    for got, ref in zip(penalty(call, blk), penalty(ref_call, ref_blk)):
        assert norm_error(got, ref) < 1e-4
    for p in blk.parameters():
        p.requires_grad_(False)
    blk.norm2.weight.requires_grad_(True)
    blk.mlp.fc2.bias.requires_grad_(True)
    out, _ = call(feat)
    out.square().sum().backward()
    assert blk.norm2.weight.grad is not None and blk.mlp.fc2.bias.grad is not None and blk.attn.q.weight.grad is None


def test_hooks_and_replaced_layers_are_called(device):
    """Modules with hooks or of other types run as modules, with gradients and without."""
    for grad in (True, False):
        blk, feat, call = dense_block(device)
        with torch.set_grad_enabled(grad):
            plain, branch = call(feat)
            assert branch is None                                   # the block kernels ran
            seen = []
            handle = blk.mlp.register_forward_hook(lambda *a: seen.append(1))
            out, branch = call(feat)
            assert seen and norm_error(out + branch, plain) < 1e-5
            handle.remove()

            for name in ("mlp", "attn", "attn.proj", "mlp.drop") + (("norm1",) if grad else ()):    # a norm is a kernel in inference
                mod = blk.get_submodule(name)                       # a forward of the module's own, as wrapping libraries set
                mod.forward = lambda *a, f=mod.forward: 2 * f(*a)
                out, branch = call(feat)
                assert norm_error(out if branch is None else out + branch, plain) > 1e-2, name
                del mod.forward

            class Doubled(torch.nn.Linear):
                def forward(self, x):
                    return 2 * super().forward(x)

            twice = Doubled(64, 64).to(device)
            twice.load_state_dict(blk.attn.proj.state_dict())
            blk.attn.proj = twice
            out, branch = call(feat)
            assert branch is not None and norm_error(out + branch, plain) > 1e-2


def test_forward_mode(device):
    blk, feat, call = dense_block(device)
    with torch.autograd.forward_ad.dual_level():
        out, branch = call(torch.autograd.forward_ad.make_dual(feat, torch.ones_like(feat)))
        assert torch.autograd.forward_ad.unpack_dual(out + branch).tangent is not None


@pytest.mark.parametrize("grad", [True, False])
def test_dropout_follows_its_own_mode(device, grad):
    """Dropout of a block in eval mode that is itself in training mode drops (Monte-Carlo dropout), and stochastic depth of a
    training block that is itself in eval mode does not."""
    torch.manual_seed(0)
    blk = ClusterTransformerBlock(64, 2, drop=0.5, attn_drop=0.5, drop_path=0.9, ops=default_ops()).to(device).eval()
    feat, table = torch.randn(8, 36, 64, device=device), torch.randn(121, 5, device=device)
    pe_idx = torch.randint(121, (8, 36, 36), device=device)

    def call():
        with torch.set_grad_enabled(grad):
            out, branch = blk(feat, None, None, pe_idx, True, table)
            return (out if branch is None else out + branch).detach()

    plain = call()
    for name in ("mlp.drop", "attn.proj_drop", "attn.attn_drop"):
        blk.get_submodule(name).train()
        assert norm_error(call(), plain) > 1e-2, name
        blk.eval()
    blk.train()
    for name in ("mlp.drop", "attn.proj_drop", "attn.attn_drop", "drop_path"):
        blk.get_submodule(name).eval()
    assert norm_error(call(), plain) < 1e-5
    blk.drop_path.train()
    assert norm_error(call(), plain) > 1e-2


@pytest.mark.parametrize("grad", [True, False])
def test_parameters_that_are_plain_attributes(device, grad):
    """A replica, as `nn.DataParallel` makes them: no entries in the modules' tables of parameters."""
    blk, feat, call = dense_block(device)
    replica, = torch.nn.parallel.replicate(blk, [device])
    args = (None, None, torch.randint(121, (2, 36, 36), device=device), True, torch.randn(121, 5, device=device))
    assert not replica.norm1._parameters
    with torch.set_grad_enabled(grad):
        (want, _), (got, branch) = blk(feat, *args), replica(feat, *args)
        assert branch is None and torch.equal(got, want)                # the block kernels, for the replica too
        if grad:
            got.square().sum().backward()
            assert blk.mlp.fc1.weight.grad.norm() > 0 and blk.attn.blank_k.grad.norm() > 0


@pytest.mark.parametrize("layered", [False, True])
@pytest.mark.parametrize("forward,backward", [(None, torch.float16), (torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16),
                                              (torch.float16, None)])
def test_backward_under_another_autocast(device, forward, backward, layered):
    """The backward of a block computes in the types of its forward, wherever it is called: the gradients are the same numbers."""
    ops = SimpleNamespace(**{**vars(default_ops()), **({"block_tail": None} if layered else {})})
    results = []
    for amp in (forward, backward):
        stage, feat, call = local_stage(device, ops)
        with torch.autocast("cuda", dtype=forward or torch.float16, enabled=forward is not None):
            out = call(feat)
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            out.square().sum().backward()
        results.append([p.grad for p in stage.parameters()])
    for got, ref in zip(*results):
        assert norm_error(got, ref) < (5e-2 if layered else 1e-6)    # layer by layer the products follow the region


def test_gradients_that_are_parts_of_a_buffer(device):
    """Incoming gradients off 16-byte boundaries, and expanded ones."""
    blk, feat, call = dense_block(device)
    _, stage_feat, stage = local_stage(device, default_ops())
    for feat, f in ((feat, lambda x: call(x)[0]), (stage_feat, stage)):
        x = feat.clone().requires_grad_(True)
        out = f(x)
        buffer = torch.randn(out.numel() + 1, generator=torch.Generator(device).manual_seed(1), device=device)
        part = buffer[1:].view(out.shape)
        got, = torch.autograd.grad(out, x, part, retain_graph=True)
        want, = torch.autograd.grad(out, x, part.clone(), retain_graph=True)
        assert torch.equal(got, want)
        part = buffer[1].expand(out.shape)
        got, = torch.autograd.grad(out, x, part, retain_graph=True)
        want, = torch.autograd.grad(out, x, part.contiguous())
        assert torch.equal(got, want)


def test_batched_gradients(device):
    """`is_grads_batched` through a training block: each row as by itself."""
    blk, feat, call = dense_block(device)
    x = feat.clone().requires_grad_(True)
    wanted = [x] + list(blk.parameters())
    batch = torch.randn(3, *feat.shape, generator=torch.Generator(device).manual_seed(1), device=device)
    out, branch = call(x)
    assert branch is None                                            # the block kernels ran
    got = torch.autograd.grad(out, wanted, batch, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for g, ref in zip(got, torch.autograd.grad(out, wanted, batch[i], retain_graph=True)):
            assert norm_error(g[i], ref) < 1e-5


def gathered(t, idx):
    b, h, n, c = t.shape
    m = idx.shape[-1]
    return t.gather(2, idx.reshape(b, 1, n * m, 1).expand(-1, h, -1, c)).view(b, h, n, m, c)


RECORDED = SimpleNamespace(qk=lambda q, k, idx: (q.unsqueeze(3) * gathered(k, idx)).sum(-1),
                           av=lambda a, v, idx: (a.unsqueeze(-1) * gathered(v, idx)).sum(3), wf=None)


def local_stage(device, ops):
    """Two blocks on 100 tokens: a short last cluster, pad slots and a mask."""
    torch.manual_seed(3)
    stage = BasicLayer(64, None, 8, 48, 2, 2, 2.0, downsample=False, ops=ops).to(device)
    ys, xs = torch.meshgrid(torch.arange(10.0), torch.arange(10.0), indexing="ij")
    pos = torch.stack([xs, ys], 2).reshape(1, 100, 2).expand(2, -1, -1).to(device)
    table, radius = relative_position_table(40)
    feat = torch.randn(2, 100, 64, device=device)
    table = table.to(device)
    return stage, feat, lambda x: stage(pos, x, 10, 10, False, 2, table, radius)[1]


# one Function for the attention's rows, and, where the block kernels are not there, one for its query, key and value
@pytest.mark.parametrize("layered", [False, True])
def test_second_derivatives_of_local_attention(device, layered):
    """Against the same stage in operations that autograd records, all terms of every parameter; and a batch of gradients."""
    ops = SimpleNamespace(**{**vars(default_ops()), **({"block_tail": None} if layered else {})})
    results = []
    for these in (ops, RECORDED):
        stage, feat, call = local_stage(device, these)
        x = feat.clone().requires_grad_(True)
        out = call(x)
        names = {type(f).__name__ for f in walk(out.grad_fn)}
        assert ("_ClusterAttentionBackward" in names) == (layered and these is ops)
        assert ("_ClusterAttentionRowsBackward" in names) == (not layered and these is ops)
        wanted = [x] + list(stage.parameters())
        first = torch.autograd.grad(out.square().sum(), wanted, create_graph=True)
        second = torch.autograd.grad(sum(g.square().sum() for g in first), wanted)
        batch = torch.randn(2, *out.shape, generator=torch.Generator(device).manual_seed(1), device=device)
        batched = torch.autograd.grad(call(x), wanted, batch, is_grads_batched=True)
        results.append((first, second, batched))
    for kind, got, ref in zip(("first", "second", "batched"), *results):
        for (name, _), g, r in zip([("x", None)] + list(stage.named_parameters()), got, ref):
            assert norm_error(g, r) < 1e-4, (kind, name)


def walk(node):
    seen, todo = set(), [node]
    while todo:
        f = todo.pop()
        if f is not None and f not in seen:
            seen.add(f)
            todo += [g for g, _ in f.next_functions]
    return seen


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("local", [True, False])
def test_frozen_parameters(device, dt, local):
    """Gradients of a block some of whose parameters take none: those of the others are the same numbers."""
    grads = []
    for frozen in ((), ("attn.q.weight", "attn.q.bias", "mlp.fc1.bias", "norm1.weight", "attn.blank_k", "attn.pos_embed.weight")):
        mod, feat, call = local_stage(device, default_ops()) if local else dense_block(device)
        names = dict(mod.named_parameters())
        for name in names:
            names[name].requires_grad_(not name.endswith(frozen) if frozen else True)
        x = feat.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.float16 if dt == torch.float32 else dt, enabled=dt != torch.float32):
            out = call(x) if local else call(x)[0]
        out.float().square().sum().backward()
        grads.append({"x": x.grad, **{n: p.grad for n, p in names.items()}})
    for name, ref in grads[0].items():
        got = grads[1][name]
        assert (got is None) if name != "x" and name.endswith(frozen) else torch.equal(got, ref), name


@pytest.mark.parametrize("name", ["block_pack", "bias_table_grad", "cluster_pairs", "cluster_attention_plan", "norm_linear", "scatter_rows"])
def test_replaced_operations_are_called_in_training(device, name):
    """What a caller put in the place of an operation that a native call for a whole block stands for, with the same gradients."""
    calls = []

    def counted(*args, **kwargs):
        calls.append(name)
        return getattr(_native, name)(*args, **kwargs)

    results = []
    for ops in (default_ops(), SimpleNamespace(**{**vars(default_ops()), name: counted})):
        stage, feat, call = local_stage(device, ops)
        x = feat.clone().requires_grad_(True)
        results.append(torch.autograd.grad(call(x).square().sum(), [x, *stage.parameters()]))
    assert calls
    for got, ref in zip(*results):
        assert norm_error(got, ref) < 1e-5


@pytest.mark.parametrize("dt,stream", [(torch.float16, torch.float16), (torch.float16, torch.float32), (torch.bfloat16, torch.float32),
                                       (torch.float32, torch.float32)])
def test_factors_that_are_no_numbers_of_the_type(device, dt, stream):
    """Factors that fp16 and bf16 do not hold: both branches' are rounded to the type, in the backward as in the forward."""
    gen = torch.Generator(device).manual_seed(7)
    b, n, c, hidden = 3, 33, 64, 128

    def draw(*shape):
        return torch.randn(*shape, generator=gen, device=device)

    w_p, w_1, w_2 = draw(c, c) / 8, draw(hidden, c) / 8, draw(c, hidden) / 11
    packed, at = _native.block_pack(c, dt, [(w, t) for t in (False, True) for w in (w_p, w_1, w_2)])
    x, d_out, attn = draw(b, n, c).to(stream), draw(b, n, c).to(stream), draw(b, n, c).to(dt)
    norm_w, norm_b, zero = 1 + 0.2 * draw(c), draw(c), torch.zeros(hidden, device=device)
    scale = torch.tensor([[1 / 0.9, 1 / 0.7, 0.0], [1 / 0.6, 0.0, 1 / 0.9]], device=device)
    results = []
    for s in (scale, scale.to(dt).float()):
        out, x1, normed, hid, stats = _native.block_tail(attn, x, packed, at[:3], zero[:c], norm_w, norm_b, 1e-5, zero, zero[:c], s, keep=True)
        results.append((out, x1) + tuple(_native.block_tail_backward(d_out, x1, stats, norm_w, hid, packed, at[3:], s)))
    for got, ref in zip(*results):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("dt", DTYPES)
def test_what_a_training_step_is_made_of(device, dt):
    """A model's graph has a node of its own for every block and merge, and the layers' general form for none of what these stand for.
    In bf16 with local lists in every stage, as above."""
    net = build(default_ops(), device, 0.4, (48, 48, 24) if dt == torch.bfloat16 else (48, 48, 48, 48)).train()
    images = torch.randn(2, 3, 96, 96, generator=torch.Generator(device).manual_seed(1), device=device)
    with torch.autocast("cuda", dtype=torch.float16 if dt == torch.float32 else dt, enabled=dt != torch.float32):
        out = net(images)
    names = [type(f).__name__ for f in walk(out.grad_fn)]
    stages = [m for m in net.modules() if isinstance(m, BasicLayer)]
    merges = sum(m.downsample is not None for m in stages)
    local = names.count("_ClusterAttentionRowsBackward")
    if dt != torch.bfloat16:
        assert local + names.count("_DenseAttentionRowsBackward") == sum(len(m.blocks) for m in stages) and 0 < local < sum(len(m.blocks) for m in stages)
        assert "_NormLinearRowsBackward" not in names and "_BlockTailBackward" not in names
    else:
        assert local > 0
    for name in ("_MergeWeightsBackward", "_MergeTableBackward", "_RowScoreBackward"):
        assert names.count(name) == merges, name
    assert names.count("_LayerNormRowsBackward") == merges + 1       # of the merges and at the end; the patch embedding's 32 channels are not built


def test_global_attention_of_an_fp32_forward_is_one_kernel(device):
    """The stage's blocks by one call, and, issued one by one, the attention by its kernel."""
    calls = []

    def counted(name):
        def call(*args, **kwargs):
            calls.append(name)
            return getattr(_native, name)(*args, **kwargs)
        return call

    images, counts = torch.randn(2, 3, 96, 96, generator=torch.Generator(device).manual_seed(1), device=device), {}
    for name in ("blocks_forward", "dense_attention_train"):
        ops = SimpleNamespace(**{**vars(default_ops()), name: counted(name)})
        net = build(ops, device, 0.0, (48, 48, 48, 48)).eval()
        calls.clear()
        with torch.no_grad():
            net(images)
        counts[name] = len(calls)
    stages = [m for m in net.modules() if isinstance(m, BasicLayer)]
    assert counts["blocks_forward"] == len(stages)
    assert counts["dense_attention_train"] == sum(len(m.blocks) for m in stages[-2:])        # 36 and 9 tokens; 576 and 144 ahead of them


@pytest.mark.parametrize("masked", [True, False])
def test_second_derivatives_of_merge_weights(device, masked):
    """fp32 against the recorded formula: gradients, those of a backward that is itself recorded, and a batch of gradients."""
    from aff.model import _MergeWeights
    gen = torch.Generator(device).manual_seed(5)
    b, n, n_out, m, rows = 2, 50, 12, 48, 225
    table, prob = torch.randn(rows, 4, generator=gen, device=device), torch.rand(b, n, generator=gen, device=device)
    pe, idx = (torch.randint(k, (b, n_out, m), generator=gen, device=device) for k in (rows, n))
    mask = torch.randint(2, (b, n_out, m), generator=gen, device=device) if masked else None

    def recorded(t, p, *_):
        w = t[pe] * p.gather(1, idx.reshape(b, -1)).reshape(b, n_out, m, 1)
        return w if mask is None else w * mask.unsqueeze(3)

    derivatives_agree(lambda t, p: _MergeWeights.apply(t, p, pe, idx, mask, default_ops()), recorded, (table, prob), gen)


@pytest.mark.parametrize("c", [32, 128])
def test_second_derivatives_of_row_scores(device, c):
    from aff.model import _RowScore
    gen = torch.Generator(device).manual_seed(c)
    x, w, bias = (torch.randn(*s, generator=gen, device=device) * k for s, k in (((2, 33, c), 1.0), ((1, c), c ** -0.5), ((1,), 1.0)))
    derivatives_agree(lambda *a: _RowScore.apply(*a, torch.float32, default_ops()), lambda *a: F.linear(*a).sigmoid(), (x, w, bias), gen)


def derivatives_agree(fn, recorded, tensors, gen):
    results, batch = [], None
    for f in (fn, recorded):
        wanted = [t.clone().requires_grad_() for t in tensors]
        out = f(*wanted)
        batch = torch.randn(3, *out.shape, generator=gen, device=out.device) if batch is None else batch
        plain = torch.autograd.grad(out, wanted, batch[0], retain_graph=True)
        first = torch.autograd.grad(out, wanted, batch[0], create_graph=True)
        second = torch.autograd.grad(sum(g.square().sum() for g in first), wanted, allow_unused=True)
        results.append(plain + first + second + torch.autograd.grad(f(*wanted), wanted, batch, is_grads_batched=True))
    for got, ref in zip(*results):
        assert (got is None and ref is None) or norm_error(got, ref) < 1e-5


# every width; a row, a workgroup's rows and one more, and more rows than all workgroups take at once
@pytest.mark.parametrize("c,rows", [(64, 1), (64, 33), (64, 40000), (128, 17), (256, 9), (384, 1025), (512, 4101), (768, 8), (1024, 5000)])
@pytest.mark.parametrize("dt,dy", [(torch.float32, torch.float32), (torch.float32, torch.float16), (torch.float32, torch.bfloat16),
                                   (torch.float16, torch.float32), (torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                   (torch.bfloat16, torch.bfloat16)])
def test_layer_norm_in_training(device, c, rows, dt, dy):
    """Against float64.  A result stored in 16 bits: one rounding, 4e-4 / 3e-3; fp32: 1e-6 (a row's two sums); column sums: 2e-6 of the
    root of the sum of the squared terms, which is what roundings of 2^-24 of running sums over up to 40 rows a lane add up to."""
    gen = torch.Generator(device).manual_seed(rows + c)
    x, d = (torch.randn(1, rows, c, generator=gen, device=device).to(t) for t in (dt, dy))
    w, b = 1 + 0.2 * torch.randn(c, generator=gen, device=device), torch.randn(c, generator=gen, device=device)
    ref = [t.double().requires_grad_() for t in (x, w, b)]
    y = torch.nn.functional.layer_norm(ref[0], (c,), ref[1], ref[2], 1e-5)
    d_x, d_w, d_b = torch.autograd.grad(y, ref, d.double())
    bar = {torch.float32: 1e-6, torch.float16: 4e-4, torch.bfloat16: 3e-3}
    out, stats = _native.layer_norm_train(x, w, b, 1e-5, dy)
    got = _native.layer_norm_backward(d, x, stats, w)
    assert (out.double() - y).norm() <= bar[dy] * y.norm() and (got[0].double() - d_x).norm() <= bar[dt] * d_x.norm() + 1e-12
    h = ((y - ref[2]) / ref[1]).detach()
    for g, want, terms in ((got[1], d_w, d.double() * h), (got[2], d_b, d.double())):
        assert ((g.double() - want).abs() <= 2e-6 * terms.square().sum((0, 1)).sqrt() + 1e-12).all()


@pytest.mark.parametrize("amp", [torch.float16, torch.bfloat16, None])
def test_layer_norm_module_in_training(device, amp):
    """The module through the kernels: strided rows, a gradient that is an expanded view, a backward that is itself differentiated."""
    from aff.model import _layer_norm, default_ops
    norm = torch.nn.LayerNorm(64).to(device)
    base = torch.randn(3, 64, 50, device=device, generator=torch.Generator(device).manual_seed(3)).to(amp or torch.float32).requires_grad_()

    def grads(fn, create):
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            y = fn(base.transpose(1, 2))
        assert y.dtype == torch.float32
        return torch.autograd.grad(y.mean(1).pow(3).sum(), (base, norm.weight, norm.bias), create_graph=create)

    mine, theirs = grads(lambda x: _layer_norm(norm, x, default_ops()), False), grads(norm, False)
    twice = grads(lambda x: _layer_norm(norm, x, default_ops()), True)
    for a, b, c in zip(mine, theirs, twice):
        bar = 2e-5 if a.dtype == torch.float32 else 2 * BAR[a.dtype]
        assert a.dtype == b.dtype == c.dtype and (a - b).norm() <= bar * b.norm() and (c - b).norm() <= bar * b.norm() and c.requires_grad
