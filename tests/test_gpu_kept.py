"""What a model keeps between inference forwards - packed weights, 16-bit copies, tables, argument arrays - against models that
have kept nothing: after writes that the keys cannot see, in recordings, and on other streams."""
from types import SimpleNamespace

import pytest
import torch

from aff.model import AutoFocusFormer, CapturedForward, default_ops

pytestmark = pytest.mark.gpu

# 576 and 144 tokens with local lists, 36 and 9 with global attention
CFG = dict(img_size=96, embed_dim=(32, 64, 128, 256), num_heads=(1, 2, 4, 8), depths=(1, 2, 2, 1), mlp_ratio=2.0, cluster_size=8,
           nbhd_size=(48, 48, 48, 48), num_classes=40)


def build(device, ops=None, seed=5):
    torch.manual_seed(seed)
    return AutoFocusFormer(ops=ops or default_ops(), **CFG).to(device).eval()


def images(device, b=3):
    return torch.randn(b, 3, 96, 96, generator=torch.Generator().manual_seed(b)).to(device)


def run(net, x, amp=None):
    with torch.no_grad(), torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        return net(x)


def fresh_copy(net, device, ops=None):
    other = build(device, ops, seed=6)
    other.load_state_dict(net.state_dict())
    return other


def block_weights(net):
    for layer in net.layers:
        for blk in layer.blocks:
            yield from (blk.attn.q.weight, blk.attn.kv.weight, blk.attn.proj.weight, blk.mlp.fc1.weight, blk.mlp.fc2.weight)


@pytest.mark.parametrize("one_call", [True, False])
def test_fp32_forwards_read_the_parameters_as_they_are(device, one_call):
    """A write through `.data` leaves address and version as they were: forwards without mixed precision see it all the same,
    with the blocks of a stage issued by one call and one by one, and so do replays of a recording."""
    ops = default_ops() if one_call else SimpleNamespace(**{**vars(default_ops()), "blocks_forward": None})
    net, x = build(device, ops), images(device)
    first = run(net, x)
    recorded = CapturedForward(net, x, autocast_dtype=None)
    assert torch.equal(recorded(x), first)
    for factor in (1.25, 0.5):
        for w in block_weights(net):
            w.data.mul_(factor)
        want = run(fresh_copy(net, device, ops), x)
        assert not torch.equal(want, first)
        assert torch.equal(run(net, x), want)
        assert torch.equal(recorded(x), want)


def churn(net, x):
    """What drops a kept value: forwards in other types, a changed weight; and memory for whoever asks for it, not zeros."""
    for amp in (torch.bfloat16, None, torch.float16):
        run(net, x, amp)
    with torch.no_grad():
        for w in block_weights(net):
            w.mul_(1.5)
    run(net, x, torch.float16)
    run(net, x)
    return [torch.full((1 << k,), float("nan"), device=x.device) for k in range(6, 22) for _ in range(8)]


@pytest.mark.parametrize("amp", [torch.float16, torch.bfloat16])
def test_recordings_outlive_what_the_model_keeps(device, amp):
    """16-bit weights are part of a recording: its replays repeat bit for bit after forwards in other types and changes of the
    weights have replaced what the model keeps."""
    net, x = build(device), images(device)
    recorded = CapturedForward(net, x, autocast_dtype=amp)
    first = recorded(x).clone()
    assert torch.equal(first, run(net, x, amp))
    junk = churn(net, x)
    for _ in range(3):
        assert torch.equal(recorded(x), first)
    del junk


@pytest.mark.parametrize("amp", [torch.float16, None])
def test_a_recording_of_the_callers_own(device, amp):
    """Recorded by `torch.cuda.graph` itself, of a model that has kept nothing yet: forwards between recording and first replay
    take nothing from it, and replays read the parameters as they are."""
    x = images(device)
    run(build(device, seed=7), x, amp)                           # library handles and kernel choices
    net = build(device)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(net, x, amp)
    want = run(fresh_copy(net, device), x, amp)
    assert torch.equal(run(net, x, amp), want)
    graph.replay()
    assert torch.equal(out, want)
    junk = churn(net, x)
    want = run(fresh_copy(net, device), x, amp)
    for _ in range(3):
        graph.replay()
        assert torch.equal(out, want)
    del junk


def delayed(stream):
    """Makes `stream` start what comes next some 30 ms late."""
    with torch.cuda.stream(stream):
        torch.cuda._sleep(60_000_000)


@pytest.mark.parametrize("amp", [torch.float16, None])
def test_kept_values_on_other_streams(device, amp):
    """What one stream is still to compute another one waits for, and what one stream is still to read is not overwritten when
    another one drops it."""
    x = images(device)
    want = run(build(device), x, amp)
    net, side = build(device), torch.cuda.Stream()
    torch.cuda.synchronize()
    delayed(side)
    with torch.cuda.stream(side):
        first = run(net, x, amp)
    second = run(net, x, amp)                                    # by the lists, tables and weights the other stream makes
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)
    delayed(side)
    with torch.cuda.stream(side):
        third = run(net, x, amp)
    for other in (torch.bfloat16, torch.float16, None):
        run(net, x, other)
    junk = [torch.full((1 << k,), float("nan"), device=device) for k in range(6, 22) for _ in range(8)]
    torch.cuda.synchronize()
    assert torch.equal(third, want)
    del junk


@pytest.mark.parametrize("amp", [torch.float16, None])
def test_a_model_that_leaves_takes_everything_along(device, amp):
    """Moved to the CPU a model leaves nothing behind but the lists of its grid."""
    x = images(device)
    run(build(device, seed=7), x, amp)                           # library workspaces
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    net = build(device)
    want = run(net, x, amp)
    net.cpu()
    grid = [t for layer in net.layers for kept in layer._grid_cache.values() for t in kept.made]
    lists = sum({t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() + 512 for t in grid}.values())
    # 512: allocations are rounded up; the result of the forward, the table of positions
    assert torch.cuda.memory_allocated() - before <= lists + 512 * 2
    assert torch.equal(run(net.to(device), x, amp), want)
