"""The C++ launch path (kotflash_amd._native) against the Python path it
stands in for: the same bits for every form both accept, the same refusals,
and autograd's hooks, checkpointing and streams as with a Python Function."""
import copy
import pickle

import pytest
import torch
from torch.utils.checkpoint import checkpoint

import kotflash_amd as kf
from kotflash_amd import _hip
from kotflash_amd.cache import PreallocatedKVCache, RaggedKVCache
from tests.gpu_helpers import seeded

pytestmark = pytest.mark.gpu
F16, BF16 = torch.float16, torch.bfloat16


@pytest.fixture
def python_path(monkeypatch):
    """Runs a call with the native entries answering NotImplemented."""
    def run(fn, *args, **kwargs):
        with monkeypatch.context() as mp:
            mp.setattr(_hip, "_NATIVE", _hip._NoNative())
            return fn(*args, **kwargs)
    return run


def _layout(t, layout):
    if layout == "bshd":
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    if layout == "padded":       # a prefix view of longer rows
        return torch.cat((t, t[:, :, :1]), 2)[:, :, :-1]
    if layout == "odd":          # strides the kernels cannot read in place
        return torch.cat((t, t[..., :3]), 3)[..., :-3]
    return t


@pytest.mark.parametrize("layout", ["plain", "bshd", "padded", "odd"])
@pytest.mark.parametrize("shape", [
    (2, 8, 2, 130, 130, 64, True, F16), (1, 4, 4, 33, 257, 72, False, BF16),
    (1, 4, 2, 1, 1500, 64, False, F16), (2, 4, 1, 16, 1024, 128, False, BF16),
    (1, 2, 2, 5, 3, 8, True, F16), (1, 2, 2, 40, 40, 20, False, F16),
])
def test_same_bits_as_the_python_path(python_path, shape, layout):
    b, hq, hkv, sq, sk, d, causal, dtype = shape
    q, k, v, do = (_layout(seeded(s, 40 + i, dtype=dtype), layout) for i, s in enumerate(
        ((b, hq, sq, d), (b, hkv, sk, d), (b, hkv, sk, d), (b, hq, sq, d))))

    def infer(**kw):
        return kf.attention(q, k, v, causal=causal, **kw)

    def train(**kw):
        leaves = [t.detach().requires_grad_() for t in (q, k, v)]
        out = kf.attention(*leaves, causal=causal, backend="hip", **kw)
        return (out, *torch.autograd.grad(out, leaves, do))

    for kw in ({}, {"scale": -0.3}):
        assert torch.equal(infer(**kw), python_path(infer, **kw))
        for a, e in zip(train(**kw), python_path(train, **kw)):
            assert torch.equal(a, e) and a.stride() == e.stride()


def test_gradients_through_hooks_checkpoint_and_expanded_grad(python_path):
    q, k, v = (seeded((1, 4, 200, 64), 60 + i, dtype=F16) for i in range(3))

    def step(how):
        leaves = [t.clone().requires_grad_() for t in (q, k, v)]
        packed = []
        call = lambda *t: kf.attention(*t, causal=True, backend="hip")  # noqa: E731
        if how == "saved hooks":
            with torch.autograd.graph.saved_tensors_hooks(
                    lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
                out = call(*leaves)
        elif how == "checkpoint":
            out = checkpoint(call, *leaves, use_reentrant=False)
        else:
            out = call(*leaves)
        if how == "tensor hook":
            out.register_hook(lambda g: g * 2)
        out.sum().backward()  # an expanded, stride-0 grad_out
        return packed, [t.grad for t in leaves]

    for how in ("plain", "saved hooks", "checkpoint", "tensor hook"):
        (pa, a), (pe, e) = step(how), python_path(step, how)
        assert pa == pe
        for x, y in zip(a, e):
            assert torch.equal(x, y), how


def test_refusals_stay(python_path):
    q, k, v = (seeded((1, 4, 64, 64), 70 + i, dtype=F16) for i in range(3))
    leaf = q.clone().requires_grad_()

    def second_order():
        g, = torch.autograd.grad(kf.attention(leaf, k, v, backend="hip").sum(), leaf, create_graph=True)
        torch.autograd.grad(g.sum(), leaf)

    def saved_mutated():
        x = leaf * 1
        out = kf.attention(x, k, v, backend="hip")
        x.mul_(2)
        out.sum().backward()

    calls = [
        lambda: kf.attention(q, k, v, backend="hip", scale=float("nan")),
        lambda: kf.attention(q, k, v, causal=1),
        lambda: kf.attention(q, k, v[:, :2]),
        lambda: kf.attention(q, k, v.bfloat16()),
        lambda: kf.attention(q, k, v.cpu()),
        lambda: kf.attention(q.float(), k.float(), v.float(), backend="hip"),
        lambda: kf.attention(q, k, v, backend="nope"),
        lambda: torch.vmap(lambda t: kf.attention(t[None], k, v, backend="hip"))(q),
        lambda: torch.func.grad(lambda t: kf.attention(t, k, v, backend="hip").sum())(q),
        lambda: torch.func.jvp(lambda t: kf.attention(t, k, v, backend="hip"), (q,), (q,)),
        second_order, saved_mutated,
    ]
    for i, call in enumerate(calls):
        with pytest.raises(Exception) as native:
            call()
        with pytest.raises(Exception) as python:
            python_path(call)
        assert type(native.value) is type(python.value), i
        assert str(native.value)[:60] == str(python.value)[:60], i


@pytest.mark.parametrize("kind", [PreallocatedKVCache, RaggedKVCache])
def test_cache_steps_match_the_python_path(python_path, kind):
    b, hkv, cap, d = 3, 2, 1400, 64
    full = [seeded((b, hkv, cap, d), 80 + i, dtype=BF16) for i in range(2)]
    n = 1 if kind is PreallocatedKVCache else 3
    q = seeded((b, 8, n, d), 82, dtype=BF16)
    new = [seeded((b, hkv, n, d), 83 + i, dtype=BF16) for i in range(2)]

    def steps():
        cache = kind(b, hkv, cap, d, device="cuda", dtype=BF16)
        cache.k.copy_(full[0])
        cache.v.copy_(full[1])
        if kind is RaggedKVCache:
            cache.set_lengths([0, 1200, 700])
        outs = [cache.append_and_attend(q, *new) for _ in range(3)]
        outs.append(cache.attend(q))
        with pytest.raises(ValueError, match="KV cache full"):
            if kind is RaggedKVCache:
                cache.set_lengths([0, cap - n + 1, 700])
            else:
                cache.length = cap
            cache.append_and_attend(q, *new)
        state = [cache.k, cache.v]
        if kind is RaggedKVCache:
            state += [cache.seqlens, cache.starts]
        return outs + state

    for i, (a, e) in enumerate(zip(steps(), python_path(steps))):
        assert torch.equal(a, e), i


def _ragged(b, cap, lengths, dtype=F16):
    cache = RaggedKVCache(b, 1, cap, 64, device="cuda", dtype=dtype)
    cache.k.copy_(seeded((b, 1, cap, 64), 93, dtype=dtype))
    cache.v.copy_(seeded((b, 1, cap, 64), 94, dtype=dtype))
    cache.set_lengths(lengths)
    return cache


def test_ragged_lengths_across_streams():
    """A step on another stream finds the last append's tokens and lengths;
    set_lengths returns with the mirrors written."""
    b, cap = 300, 64  # two launches of the lengths kernel
    cache = _ragged(b, cap, [i % 50 for i in range(b)])
    new = [seeded((b, 1, 2, 64), 90 + i, dtype=F16) for i in range(2)]
    q = seeded((b, 1, 1, 64), 92, dtype=F16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda._sleep(20_000_000)
    cache.append(*new)
    with torch.cuda.stream(side):
        got = cache.attend(q)
        lens = cache.seqlens.clone()
    torch.cuda.synchronize()
    assert lens.tolist() == cache.lengths == [i % 50 + 2 for i in range(b)]
    assert torch.isfinite(got).all() and torch.equal(got, cache.attend(q))
    assert cache.starts.tolist() == cache.lengths


@pytest.mark.parametrize("fused", [False, True])
def test_ragged_append_returns_with_its_work_done(fused):
    """An append behind queued work of its stream: whatever another stream
    does next, without a wait of its own, sees the append's tokens, lengths and
    output, and lengths set from there stay set."""
    b, cap, lengths = 3, 1200, [0, 1100, 700]
    cache = _ragged(b, cap, lengths)
    new = [seeded((b, 1, 3, 64), 95 + i, dtype=F16) for i in range(2)]
    q = seeded((b, 4, 3, 64), 97, dtype=F16)
    held = cache.k[:, :, :], cache.seqlens[:], cache.starts[:]  # taken before the append
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        out = cache.append_and_attend(q, *new) if fused else cache.append(*new)
    k, seqlens, starts = (t.clone() for t in held)
    got = out.clone() if fused else None
    cache.set_lengths(lengths)  # drop the tokens again, from this stream
    torch.cuda.synchronize()
    assert seqlens.tolist() == starts.tolist() == [x + 3 for x in lengths]
    for i, n in enumerate(lengths):
        assert torch.equal(k[i, :, n:n + 3], new[0][i])
    assert cache.seqlens.tolist() == cache.starts.tolist() == cache.lengths == lengths
    if fused:
        again = cache.append_and_attend(q, *new)
        assert torch.isfinite(got).all() and torch.equal(got, again)


def test_ragged_copies_carry_no_stream():
    """A copied or unpickled cache holds the tokens and lengths appended on
    another stream."""
    cache = _ragged(2, 1200, [5, 1100])
    side = torch.cuda.Stream()
    new = [seeded((2, 1, 3, 64), 95 + i, dtype=F16) for i in range(2)]
    q = seeded((2, 1, 1, 64), 97, dtype=F16)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        cache.append(*new)
    for other in (copy.copy(cache), copy.deepcopy(cache), pickle.loads(pickle.dumps(cache))):
        assert other.lengths == cache.lengths
        assert other.seqlens.tolist() == other.starts.tolist() == [8, 1103]
        assert torch.equal(other.attend(q), cache.attend(q))
