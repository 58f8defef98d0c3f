"""The natively prepared calls (csrc/host_calls.cpp): inputs the kernels cannot
read in place are copied, refusals keep their exception types, and streams,
threads, saved-tensor hooks and caches that are not KVCache itself behave as
with calls prepared in Python."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from kernels import _native
from kernels.BlockSparseDecodeAttention import block_sparse_decode_attention
from kernels.BlockSparseFlashAttention import BlockSparseFlashAttention
from kernels.dit_glue import gate_residual, gate_residual_ln_modulate, ln_modulate
from kernels.kv_cache import KVCache, attention_inputs, rope_tables
from kernels.sampling import PhiloxStream, subs_sample_step
from kernels.SplitKVDecodeAttention import split_kv_decode_attention

BF = torch.bfloat16


def test_argument_errors_without_a_gpu():
    host = _native.host()
    t = torch.zeros(1, 1, 256, 64, dtype=BF)
    with pytest.raises(TypeError, match="number of arguments"):
        host.decode(t, t, t, 16)
    with pytest.raises(TypeError, match="tensor"):
        host.decode(t, t, 3, 16, 0)
    with pytest.raises(OverflowError):
        host.decode(t, t, t, 1 << 40, 0)
    with pytest.raises(KeyError):
        host.bind({})


def test_operands_off_the_gpu_are_refused_without_one():
    """CPU addresses never reach a launch: the calls raise as they did when
    the stream was looked up in Python, on a machine with or without a GPU."""
    import kernels.ops  # noqa: F401
    host = _native.host()
    q, lse = torch.zeros(1, 1, 256, 64, dtype=BF), torch.zeros(1, 1, 256)
    x, m, w = torch.zeros(1, 2, 64, dtype=BF), torch.zeros(1, 64, dtype=BF), torch.zeros(64, dtype=BF)
    qkv, table = torch.zeros(1, 4, 192, dtype=BF), torch.zeros(8, 32)
    block = torch.zeros(1, 2, dtype=torch.int64)
    for call in (
        lambda: torch.ops.bd3.attn_bwd(q, q, q, q, lse, q, 16),
        lambda: host.attn_fwd(q, q, q, 16),
        lambda: host.attn_bwd(q, q, q, q, lse, q, 16),
        lambda: host.decode(q, q, q, 16, 0),
        lambda: host.qkv_rope(qkv, 1, table, table, None, 0, None, None, 0),
        lambda: host.subs_sample(x, block, 63, 0.5, None, 0, 0),
        lambda: host.ln_modulate(x, w, m, m, 1e-5, -1),
        lambda: host.gate_residual(x, m, x, None),
        lambda: host.gate_residual_ln_modulate(x, m, x, w, m, m, 1e-5, -1, None),
    ):
        with pytest.raises(AssertionError, match="CUDA"):
            call()


def test_seeds_are_taken_modulo_2_64():
    """A generator whose seed or offset was set by hand to a negative, large or
    numpy integer is accepted, as it was by ctypes (the call gets as far as the
    refusal of its CPU tensors)."""
    host = _native.host()
    x, block = torch.zeros(1, 2, 64), torch.zeros(1, 2, dtype=torch.int64)
    for seed, offset in ((-1, 0), (1 << 64, -5), (np.int64(-7), np.uint64(1 << 63))):
        with pytest.raises(AssertionError, match="CUDA"):
            host.subs_sample(x, block, 63, 0.5, None, seed, offset)
    with pytest.raises(TypeError):
        host.subs_sample(x, block, 63, 0.5, None, 1.5, 0)


def rnd(dev, *shape, seed=0, dtype=BF):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dev, dtype)


def layouts(t):
    """t with a last stride of 2, and with outer strides that are not
    multiples of 8 elements."""
    wide = torch.empty(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype, device=t.device)[..., ::2]
    odd = torch.empty(*t.shape[:-1], t.shape[-1] + 3, dtype=t.dtype, device=t.device)[..., :t.shape[-1]]
    for x in (wide, odd):
        x.copy_(t)
        yield x


@pytest.mark.gpu
def test_inputs_that_need_a_copy(cuda):
    q, k, v, do = (rnd(cuda, 1, 2, 256, 64, seed=s) for s in range(4))

    def train(q, k, v, do):
        q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
        o = BlockSparseFlashAttention.apply(q, k, v, 16)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))

    qkv, x, y, w = rnd(cuda, 2, 16, 384, seed=4), rnd(cuda, 2, 5, 64, seed=5), rnd(cuda, 2, 5, 64, seed=6), rnd(cuda, 64)
    m = rnd(cuda, 2, 64, seed=7)
    logits, block = rnd(cuda, 3, 40, seed=8), torch.full((3,), 39, device=cuda)
    tables = rope_tables(64, 32, device=cuda)
    calls = [
        (train, (q, k, v, do)),
        (lambda *a: block_sparse_decode_attention(*a, 16), (q[:, :, :16], k, v)),
        (lambda *a: split_kv_decode_attention(*a, 16, n_splits=3), (q[:, :, :16], k, v)),
        (lambda *a: attention_inputs(*a, 2, *tables, positions=torch.arange(15, -1, -1)), (qkv,)),
        (lambda *a: ln_modulate(*a), (x, w, m, m)),
        (lambda *a: gate_residual(*a), (x, m, y)),
        (lambda *a: gate_residual_ln_modulate(*a), (x, m, y, w, m, m)),
        (lambda a: subs_sample_step(a, block, 39, 0.5, generator=PhiloxStream(1)), (logits,)),
    ]
    for i, (call, args) in enumerate(calls):
        print(f"call {i}", flush=True)
        flat = lambda r: r if isinstance(r, tuple) else (r,)  # noqa: E731
        want = flat(call(*(a.contiguous() for a in args)))
        for moved in zip(*(layouts(a) for a in args)):
            assert all(torch.equal(a, b) for a, b in zip(want, flat(call(*moved))))


@pytest.mark.gpu
def test_refusals_keep_their_types(cuda):
    q = rnd(cuda, 1, 2, 256, 64)
    x, m = rnd(cuda, 2, 5, 64), rnd(cuda, 2, 64)
    tables = rope_tables(64, 32, device=cuda)
    off = torch.empty(q.numel() + 1, dtype=BF, device=cuda)[1:].view(q.shape)  # contiguous, base 2 bytes off
    for call in (
        lambda: BlockSparseFlashAttention.apply(off, q, q, 16),
        lambda: BlockSparseFlashAttention.apply(q, q, q, 0),
        lambda: block_sparse_decode_attention(q, q, q, 0),
        lambda: attention_inputs(rnd(cuda, 1, 16, 384), 2, *tables, positions=17),  # past the table
        lambda: ln_modulate(x, m[0], m[:1], m),
        lambda: ln_modulate(x, m[0], m.float(), m),
        lambda: ln_modulate(x, m[0], m[:, None].expand(2, 5, 64), m),
        lambda: ln_modulate(x, m[0], m, m, out_dtype=torch.float32),  # bf16 modulation has a bf16 result
        lambda: gate_residual(x, m, x, out=x.float()),
        lambda: gate_residual_ln_modulate(x, m, x, m[0], m.float(), m),
        lambda: subs_sample_step(x, torch.zeros(2, 5, device=cuda, dtype=torch.int64), 64, 0.5),
    ):
        with pytest.raises(AssertionError):
            call()
    with pytest.raises(KeyError):
        ln_modulate(x.half(), m[0], m, m)
    with pytest.raises(KeyError):
        ln_modulate(x, m[0], m, m, out_dtype=torch.float16)


@pytest.mark.gpu
def test_one_operand_off_the_gpu_is_refused(cuda):
    """Every operand is looked at, not the first alone; the backward op also
    refuses the shapes and dtypes its forward would not have saved."""
    import kernels.ops  # noqa: F401
    q, lse = rnd(cuda, 1, 1, 256, 64), torch.zeros(1, 1, 256, device=cuda)
    x, m, w = rnd(cuda, 2, 5, 64), rnd(cuda, 2, 64), rnd(cuda, 64)
    sin, cos = rope_tables(64, 32, device=cuda)
    block = torch.full((2, 5), 63, device=cuda)

    def train(q, k, v, o, lse, do):
        return torch.ops.bd3.attn_bwd(q, k, v, o, lse, do, 16)

    calls = [
        (train, (q, q, q, q, lse, q)),
        (lambda *a: BlockSparseFlashAttention.apply(*a, 16), (q, q, q)),
        (lambda *a: block_sparse_decode_attention(*a, 16), (q, q, q)),
        (lambda *a: split_kv_decode_attention(*a, 16, n_splits=2), (q, q, q)),
        (lambda qkv, s, c: attention_inputs(qkv, 1, s, c), (rnd(cuda, 1, 4, 192), sin, cos)),
        (lambda *a: ln_modulate(*a), (x, w, m, m)),
        (lambda *a: gate_residual(*a), (x, m, x, x.clone())),
        (lambda *a: gate_residual_ln_modulate(*a), (x, m, x, w, m, m)),
        (lambda lg, u: subs_sample_step(lg, block, 63, 0.5, u=u), (x, torch.rand(2, 5, 64, device=cuda).double())),
    ]
    for call, args in calls:
        for i in range(len(args)):
            with pytest.raises(AssertionError):
                call(*(a.cpu() if i == j else a for j, a in enumerate(args)))
    for bad in ((q, q, q, q.float(), lse, q), (q, q, q, q, lse.double(), q), (q, q, q, q, lse[..., :128], q),
                (q, q[:, :, :128], q, q, lse, q), (q.half(), q, q, q, lse, q), (q, q, q, q, lse, q[:, :, :128])):
        with pytest.raises(AssertionError):
            train(*bad)


@pytest.mark.gpu
def test_negative_seed_is_its_value_modulo_2_64(cuda):
    logits, block = rnd(cuda, 8, 3000, seed=9), torch.full((8,), 2999, device=cuda)
    outs = []
    for seed, offset in ((-3, -2), ((1 << 64) - 3, (1 << 64) - 2)):
        g = PhiloxStream(0)
        g.seed, g.offset = seed, offset
        outs.append(subs_sample_step(logits, block, 2999, 0.1, generator=g))
    assert torch.equal(*outs)


@pytest.mark.gpu
def test_saved_tensor_hooks_see_the_saved_tensors(cuda):
    q, k, v = (rnd(cuda, 1, 1, 256, 64, seed=s).requires_grad_() for s in range(3))
    do = rnd(cuda, 1, 1, 256, 64, seed=3)
    want = torch.autograd.grad(BlockSparseFlashAttention.apply(q, k, v, 16), (q, k, v), do)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(cuda)):
        o = BlockSparseFlashAttention.apply(q, k, v, 16)
    got = torch.autograd.grad(o, (q, k, v), do)
    assert len(packed) == 5 and all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.gpu
def test_side_streams_and_threads(cuda):
    q, k, v = rnd(cuda, 2, 3, 16, 64, seed=1), rnd(cuda, 2, 3, 2000, 64, seed=2), rnd(cuda, 2, 3, 2000, 64, seed=3)
    want = block_sparse_decode_attention(q, k, v, 16)
    torch.cuda.synchronize()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(20):
                if not torch.equal(block_sparse_decode_attention(q, k, v, 16), want):
                    bad.append(1)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.gpu
def test_cache_subclass_goes_through_its_methods(cuda):
    calls = []

    class Counting(KVCache):
        def slot(self, *a):
            calls.append("slot")
            return super().slot(*a)

        def prefix_and_slot(self, *a):
            calls.append("prefix")
            return super().prefix_and_slot(*a)

    tables = rope_tables(64, 600, device=cuda)
    plain, counting = KVCache.empty(1), Counting.empty(1)
    for step in range(3):  # 3 x 200 tokens: past the first capacity of 256
        qkv = rnd(cuda, 2, 200, 3 * 128, seed=step)
        a = attention_inputs(qkv, 2, *tables, positions=200 * step, kv_cache=plain, store=True)
        b = attention_inputs(qkv, 2, *tables, positions=200 * step, kv_cache=counting, store=True)
        assert all(torch.equal(x, y) for x, y in zip(a, b))
        assert a[1].shape[2] == 200 * (step + 1) and plain.length == counting.length == 200 * (step + 1)
    assert calls == ["slot", "prefix"] * 3
