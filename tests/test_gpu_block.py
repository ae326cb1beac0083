"""GPU parity of the block kernels (`clusten_norm_linear_forward`, `clusten_block_tail_forward`) against the layers they stand
for (`norm1` + q / kv projections and proj + residual + `norm2` + MLP + residual, models/aff_transformer.py:103-106, 157-158,
219-232), evaluated in fp32 from the same rounded operands with the intermediates rounded where the layers store them.

Bar, max|x - ref| / max|ref|: 2e-3 fp16, 1e-2 bf16 (a handful of roundings of 2^-11 / 2^-8 on the way, those of the hidden
layer averaged over its channels), 1e-5 fp32.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from clusten import _native
from oracle import clusten_oracle as oracle

pytestmark = pytest.mark.gpu

BAR = {torch.float16: 2e-3, torch.bfloat16: 1e-2, torch.float32: 1e-5}
# fp32 and 16-bit token streams; row counts below a tile, across tiles, and enough for 2, 3 and 4 tiles a workgroup
CASES = [(torch.float16, torch.float16), (torch.float16, torch.float32), (torch.bfloat16, torch.bfloat16),
         (torch.float32, torch.float32)]
SHAPES = [(32, 64, 1), (32, 96, 70), (64, 192, 16), (64, 128, 16 * 1024 + 3), (128, 384, 33), (128, 128, 8192 + 17),
          (256, 768, 49), (256, 512, 16 * 1024 + 1), (512, 1536, 15), (512, 1024, 8192 - 5), (512, 512, 4096 + 1),
          (512, 512, 9217), (256, 256, 33 * 1024 + 7)]


class Block:
    """Random parameters of one block on the device, and its weights packed."""

    def __init__(self, c, hidden, dt, device, seed):
        gen = torch.Generator().manual_seed(seed)

        def draw(*shape, scale=1.0):
            return (torch.randn(*shape, generator=gen) * scale).to(device)

        self.c, self.hidden, self.dt = c, hidden, dt
        self.w = [draw(c, c, scale=c ** -0.5), draw(2 * c, c, scale=c ** -0.5), draw(c, c, scale=c ** -0.5),
                  draw(hidden, c, scale=c ** -0.5), draw(c, hidden, scale=hidden ** -0.5)]
        self.b = [draw(t.shape[0], scale=0.3) for t in self.w]
        self.norm = [1 + 0.2 * draw(c), 0.2 * draw(c), 1 + 0.2 * draw(c), 0.2 * draw(c)]
        self.packed, self.at = _native.block_pack(c, dt, [(t, False) for t in self.w])

    def rounded(self, t):
        return t.to(self.dt).float()

    def linear(self, x, i):
        return self.rounded(F.linear(x, self.rounded(self.w[i]), self.rounded(self.b[i])))

    def head(self, x):
        y = self.rounded(F.layer_norm(x.float(), (self.c,), self.norm[0], self.norm[1]))
        return torch.cat([self.linear(y, 0), self.linear(y, 1)], -1)

    def tail(self, attn, x, scale=None):
        s = 1.0 if scale is None else self.rounded(scale)[:, None, None]
        x1 = (x.float() + self.rounded(self.linear(attn.float(), 2) * s)).to(x.dtype).float()
        y = self.rounded(F.layer_norm(x1, (self.c,), self.norm[2], self.norm[3]))
        h = self.rounded(F.gelu(F.linear(y, self.rounded(self.w[3]), self.rounded(self.b[3]))))
        return x1 + self.rounded(self.linear(h, 4) * s)

    def run_head(self, x):
        return _native.norm_linear(x, self.norm[0], self.norm[1], 1e-5, self.packed, self.at[0], self.b[0], self.b[1],
                                   3 * self.c)

    def run_tail(self, attn, x, scale=None):
        return _native.block_tail(attn, x, self.packed, self.at[2:], self.b[2], self.norm[2], self.norm[3], 1e-5, self.b[3],
                                  self.b[4], scale)


@pytest.mark.parametrize("dt,stream", CASES)
@pytest.mark.parametrize("c,hidden,rows", SHAPES)
def test_against_the_layers(device, dt, stream, c, hidden, rows):
    block = Block(c, hidden, dt, device, c + rows)
    gen = torch.Generator().manual_seed(rows)
    x = (torch.randn(1, rows, c, generator=gen) * 2 + 0.5).to(device).to(stream)
    attn = torch.randn(1, rows, c, generator=gen).to(device).to(dt)
    got = block.run_head(x)
    assert got.dtype == dt and got.shape == (1, rows, 3 * c)
    assert oracle.rel_err(got.float(), block.head(x)) <= BAR[dt]
    got = block.run_tail(attn, x)
    assert got.dtype == stream and got.shape == x.shape
    assert oracle.rel_err(got.float(), block.tail(attn, x)) <= BAR[dt]


@pytest.mark.parametrize("c,hidden,rows", [(32, 96, 17), (64, 192, 513), (64, 192, 25089), (128, 384, 4095), (128, 256, 6273),
                                           (256, 768, 47), (256, 768, 784), (256, 768, 1569), (256, 768, 3137), (256, 768, 8193),
                                           (256, 512, 12289), (512, 1536, 393), (512, 1024, 2450), (512, 512, 4097)])
def test_fp32_against_float64(device, c, hidden, rows):
    """fp32 products are sums over three bf16 parts of every operand, over 1 to 4 row tiles a workgroup, the outputs shared
    among 1 to 3 of them: the parts hold all 24 bits, so what is left is the rounding of fp32 sums.  Relative 2-norm from
    float64: fp32 instructions 4.6e-7 at 512 channels, the parts 1.1e-7 (64 sums of 32 terms, each rounded to nearest)."""
    block = Block(c, hidden, torch.float32, device, c + rows)
    gen = torch.Generator().manual_seed(rows)
    x = (torch.randn(1, rows, c, generator=gen) * 2 + 0.5).to(device)
    x[0, -1] *= 1e-30                                            # far below and above the other rows
    attn = torch.randn(1, rows, c, generator=gen).to(device)
    attn[0, 0] *= 1e25
    w, b, norm = ([t.double() for t in ts] for ts in (block.w, block.b, block.norm))
    got, ref = block.run_head(x), F.layer_norm(x.double(), (c,), norm[0], norm[1])
    ref = torch.cat([F.linear(ref, w[0], b[0]), F.linear(ref, w[1], b[1])], -1)
    assert (got.double() - ref).norm() <= 1.5e-7 * ref.norm()
    got, x1 = block.run_tail(attn, x), x.double() + F.linear(attn.double(), w[2], b[2])
    ref = F.gelu(F.linear(F.layer_norm(x1, (c,), norm[2], norm[3]), w[3], b[3]))
    ref = x1 + F.linear(ref, w[4], b[4])
    assert ((got.double() - ref).norm(dim=-1) <= 3e-7 * ref.norm(dim=-1)).all()


@pytest.mark.parametrize("dt,stream", CASES)
def test_factors_of_the_images(device, dt, stream):
    """Stochastic depth: a factor per image on both branches, 0 leaving the image's rows as they are."""
    block = Block(64, 192, dt, device, 5)
    gen = torch.Generator().manual_seed(6)
    x = torch.randn(3, 37, 64, generator=gen).to(device).to(stream)
    attn = torch.randn(3, 37, 64, generator=gen).to(device).to(dt)
    scale = torch.tensor([1.25, 0.0, 1.25], device=device)
    got = block.run_tail(attn, x, scale)
    assert torch.equal(got[1], x[1])
    assert oracle.rel_err(got.float(), block.tail(attn, x, scale)) <= BAR[dt]


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_gelu_of_every_16_bit_number(device, dt):
    """With a norm of weight 0 the hidden layer is the norm's bias times the weights: identity weights bring every finite 16-bit
    number to the GELU and its result to the output, at most one unit in the last place from the exactly rounded value (below
    fp32's smallest normal number, which only bf16 results reach, it may be 0)."""
    from scipy.special import ndtr
    c = 512
    eye, zero = torch.eye(c, device=device), torch.zeros(c, device=device)
    packed, at = _native.block_pack(c, dt, [(torch.zeros(c, c, device=device), False), (eye, False), (eye, False)])
    values = torch.arange(-32768, 32768, dtype=torch.int16).view(dt)
    values = values[values.isfinite()]
    count = values.numel()
    x = torch.zeros(1, 1, c, device=device, dtype=dt)
    got = []
    for v in F.pad(values, (0, -count % c)).to(device).float().split(c):
        got.append(_native.block_tail(x, x, packed, at, zero, zero, v.contiguous(), 1e-5, zero, zero).reshape(-1))
    got = torch.cat(got)[:count].cpu()
    exact64 = values.double().numpy() * ndtr(values.double().numpy())
    exact = torch.from_numpy(exact64).to(dt)
    steps = (got.view(torch.int16).int() - exact.view(torch.int16).int()).abs()
    tiny = torch.from_numpy(np.abs(exact64) < 2.0 ** -126)
    assert ((steps <= 1) | ((got == 0) & ((exact == 0) | tiny))).all()
    assert ((torch.signbit(got) == torch.signbit(exact)) | (got == 0)).all()
    for bias in (torch.full((c,), float("nan"), device=device), zero):
        inf = torch.full((c,), -float("inf"), device=device)         # of a hidden layer: NaN, like the formula's 0 * inf
        assert torch.isnan(_native.block_tail(x, x, packed, at, zero, zero, bias, 1e-5, inf, zero)).all()


def test_gelu_in_fp32(device):
    """The erf formula in fp32 leaves the roundings of an error function, a sum and a product: 4.1e-8 of the result's root mean
    square over normal numbers of deviation 0.3, in the forward kernel as in the one ahead of the backward's products."""
    c = 512
    eye, zero = torch.eye(c, device=device), torch.zeros(c, device=device)
    packed, at = _native.block_pack(c, torch.float32, [(torch.zeros(c, c, device=device), False), (eye, False), (eye, False)])
    v = 0.3 * torch.randn(64 * c, generator=torch.Generator(device).manual_seed(1), device=device)
    x = torch.zeros(1, 1, c, device=device)
    rows = [_native.block_tail(x, x, packed, at, zero, zero, part.contiguous(), 1e-5, zero, zero).reshape(-1) for part in v.split(c)]
    exact = v.double() * 0.5 * torch.erfc(-v.double() * 0.5 ** 0.5)
    for got in (torch.cat(rows), _native.gelu_backward(v, torch.ones_like(v))[0]):
        assert (got.double() - exact).norm() <= 5e-8 * exact.norm()


@pytest.mark.parametrize("dt", list(BAR))
@pytest.mark.parametrize("c,count", [(32, 1), (256, 70)])
def test_packed_from_a_transpose(device, dt, c, count):
    """A matrix given as its transpose is packed as the matrix; more of them than one launch takes."""
    gen = torch.Generator().manual_seed(c)
    weights = [torch.randn(2 * c if i % 2 else c, c, generator=gen).to(device) for i in range(count)]
    want, at = _native.block_pack(c, dt, [(w, False) for w in weights])
    got, at_t = _native.block_pack(c, dt, [(w.t().contiguous(), True) for w in weights])
    assert at == at_t and torch.equal(got, want)
    assert torch.equal(got.float().sort().values, torch.cat([w.reshape(-1) for w in weights]).to(dt).float().sort().values)


def test_what_is_refused(device):
    block = Block(64, 192, torch.float16, device, 7)
    x = torch.randn(2, 8, 64, device=device)
    with pytest.raises(RuntimeError):
        block.run_head(x.to(torch.bfloat16))                      # neither fp32 nor the weights' type
    with pytest.raises(RuntimeError):
        block.run_head(torch.randn(2, 8, 48, device=device))      # width without a kernel
    with pytest.raises(RuntimeError):
        block.run_tail(x, x)                                      # attn not of the weights' type
    with pytest.raises(RuntimeError):
        _native.block_pack(64, torch.float16, [(torch.randn(64, 40, device=device), False)])


@pytest.mark.parametrize("amp", [torch.float16, torch.bfloat16, None])
def test_blocks_issued_by_one_call_equal_the_blocks_one_by_one(device, amp):
    """Local stages with shared and with per-image lists, short last clusters and masks (196 tokens), and the global stage of
    49 tokens: the same kernels on the same values, so bit for bit, and again after a parameter changed in place."""
    from aff.model import aff_tiny, default_ops
    torch.manual_seed(0)
    net = aff_tiny().to(device).eval()
    single_ops = default_ops()
    del single_ops.blocks_forward
    single = aff_tiny(ops=single_ops).to(device).eval()
    single.load_state_dict(net.state_dict())
    x = torch.randn(3, 3, 224, 224, generator=torch.Generator().manual_seed(1)).to(device)

    def run(m):
        with torch.no_grad(), torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            return m(x)

    first = run(net)
    assert torch.isfinite(first).all() and torch.equal(first, run(single))
    with torch.no_grad():
        for m in (net, single):
            m.layers[2].blocks[4].mlp.fc1.weight.mul_(1.5)
            m.layers[1].blocks[0].attn.pos_embed.bias.add_(0.25)
    second = run(net)
    assert not torch.equal(first, second) and torch.equal(second, run(single))


def test_models_copied_and_changed_after_a_forward(device):
    """A model is copied and pickled after a forward that kept packed weights and addresses, new parameters in the place of old
    ones are seen, and a block with another hidden width keeps its stage off the call that has one width for all."""
    import copy
    import io
    from aff.model import Mlp, aff_tiny
    torch.manual_seed(0)
    net = aff_tiny().to(device).eval()
    x = torch.randn(2, 3, 224, 224, generator=torch.Generator().manual_seed(1)).to(device)

    def run(m):
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            return m(x)

    first = run(net)
    assert torch.equal(first, run(copy.deepcopy(net)))
    torch.save(net.layers[2].blocks[0].__dict__.get("_pack_cache"), io.BytesIO())
    torch.save(net.layers[2].__dict__.get("_issue_cache"), io.BytesIO())
    fc1 = net.layers[2].blocks[4].mlp.fc1
    for factor in (1.5, 0.5):
        value = (fc1.weight.detach() * factor).cpu()
        fc1.weight = None                                        # its memory may be what the next one gets
        fc1.weight = torch.nn.Parameter(value.to(device))
        fresh = aff_tiny().to(device).eval()
        fresh.load_state_dict(net.state_dict())
        assert torch.equal(run(net), run(fresh))
    blk = net.layers[2].blocks[3]
    blk.mlp = Mlp(256, 256, ops=blk.mlp.ops).to(device).eval()    # narrower than the other blocks'
    out = run(net)
    calls = []
    blk.register_forward_hook(lambda *_: calls.append(1))        # with a hook every block is called by itself
    assert torch.equal(out, run(net)) and calls
    blk = net.layers[1].blocks[2]
    blk.forward = lambda *a, f=blk.forward: (calls.clear(), f(*a))[1]
    assert torch.equal(out, run(net)) and len(calls) == 1        # by the hooked block behind it only
    blk.mlp.forward = lambda x, f=blk.mlp.forward: 0 * f(x)
    assert not torch.equal(out, run(net))


def test_stages_with_active_dropout_are_not_issued_by_one_call(device):
    """Dropout in training mode somewhere in a model in eval mode drops."""
    from aff.model import AutoFocusFormer, default_ops
    torch.manual_seed(0)
    net = AutoFocusFormer(img_size=96, embed_dim=(32, 64, 128, 256), num_heads=(1, 2, 4, 8), depths=(1, 2, 2, 1), mlp_ratio=2.0,
                          nbhd_size=(48, 48, 48, 48), num_classes=40, drop_rate=0.5, attn_drop_rate=0.5, drop_path_rate=0.5,
                          ops=default_ops()).to(device).eval()
    x = torch.randn(2, 3, 96, 96, generator=torch.Generator().manual_seed(1)).to(device)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            return net(x)

    plain = run()
    for name in ("mlp.drop", "attn.proj_drop", "attn.attn_drop", "drop_path"):
        for stage in (1, 2):                                     # local and global attention; the stages' second blocks
            net.layers[stage].blocks[1].get_submodule(name).train()
            assert not torch.equal(run(), plain), (name, stage)
            net.eval()
            assert torch.equal(run(), plain)


@pytest.mark.parametrize("amp", [torch.float16, None])
def test_stages_that_one_call_does_not_fit(device, amp):
    """A later block without a bias, and one with operators of its own, go block by block; a stage without blocks has none."""
    from types import SimpleNamespace
    from aff.model import AutoFocusFormer, default_ops
    cfg = dict(img_size=96, embed_dim=(32, 64, 128, 256), num_heads=(1, 2, 4, 8), mlp_ratio=2.0, nbhd_size=(48, 48, 48, 48),
               num_classes=40)
    x = torch.randn(2, 3, 96, 96, generator=torch.Generator().manual_seed(1)).to(device)

    def run(net):
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=amp is not None):
            return net(x)

    torch.manual_seed(0)
    net = AutoFocusFormer(depths=(1, 2, 2, 1), ops=default_ops(), **cfg).to(device).eval()
    want = run(net)
    calls = []
    other = SimpleNamespace(**vars(default_ops()))
    other.block_tail = lambda *a, f=other.block_tail, **kw: (calls.append(1), f(*a, **kw))[1]
    blk = net.layers[1].blocks[1]
    blk.attn.ops = blk.mlp.ops = other
    assert torch.equal(run(net), want) and calls
    net.layers[2].blocks[1].attn.proj.bias = None                # zeros so far
    assert torch.isfinite(run(net)).all()
    assert (run(net) - want).norm() <= (1e-5 if amp is None else 4e-3) * want.norm()
    net = AutoFocusFormer(depths=(0, 1, 0, 1), ops=default_ops(), **cfg).to(device).eval()
    assert torch.isfinite(run(net)).all()
