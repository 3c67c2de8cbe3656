"""The extension module of the plain calls (csrc/pyfast.cpp) against the general
path of api.py.

CPU tier: what is not the plain case is refused (None) and reaches the general
path's errors. GPU tier: every entry point, on plain arguments and on forms that
only the general path takes (strided, offset, other scale and flag types),
gives the same bytes either way, and the plain case is the module's.
"""
import pytest
import torch

import cuda_amd._lib as L
import cuda_amd.api as api
import cuda_llm
from _util import build_paged, mx_inputs, qkv


@pytest.fixture
def general(monkeypatch):
    """Calls f through the general path."""
    def run(f):
        with monkeypatch.context() as m:
            m.setattr(api, "_native_module", L._General())
            m.setattr(api, "_native", lambda: api._native_module)
            return f()
    return run


def test_refuses_what_is_not_plain():
    n = L.native()
    if isinstance(n, L._General):
        pytest.skip("library not built")
    q = torch.zeros(1, 2, 4, 64, dtype=torch.bfloat16)
    assert n.flash_attention_forward(q, q, q, False, None) is None       # CPU
    assert n.flash_attention_forward(q, q, None, False, None) is None    # no tensor
    assert n.flash_attention_forward(q, q) is None                       # arguments missing
    assert n.async_flash_decode(q, q, q, "x") is None
    assert n.paged_kv_append(*[q] * 4, *[None] * 5) is None
    with pytest.raises(RuntimeError, match="Inputs must be on CUDA"):
        cuda_llm.flash_attention(q, q, q)
    with pytest.raises(TypeError):
        n.bind(1)


def test_decode_workspace_sizes():
    """The best workspace is never less than the least one; invalid sizes are 0."""
    lib = L.load()
    for n, hq, hkv, d, blocks in ((1, 32, 8, 128, 3), (3, 32, 8, 128, 256), (64, 32, 8, 64, 512), (1, 1, 1, 64, 2 ** 26)):
        least = lib.ca_decode_workspace_bytes(n, hq, d, 16 * blocks)
        for dt in (L.CA_F32, L.CA_F16, L.CA_BF16):
            for fp8 in (0, 1):
                assert lib.ca_paged_decode_workspace_bytes(dt, fp8, n, hq, hkv, d, blocks) >= least
            assert lib.ca_flash_decode_workspace_bytes(dt, n, hq, hkv, 16 * blocks, d) >= least
    big = 2 ** 31 - 1
    for bad in ((0, 32, 8, 128, 4), (1, 32, 5, 128, 4), (1, 32, 8, 96, 4), (1, 32, 8, 128, -1), (big, big, 1, 128, big)):
        assert lib.ca_paged_decode_workspace_bytes(L.CA_BF16, 0, *bad) == 0
        assert lib.ca_flash_decode_workspace_bytes(L.CA_BF16, *bad[:3], bad[4], bad[3]) == 0


def _same(a, b):
    a, b = ([x] if torch.is_tensor(x) else list(x) for x in (a, b))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and x.is_contiguous()
        assert not x.requires_grad
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))


def _offset(t):
    """The same values, contiguous, one element past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.flatten()
    return buf[1:].view(t.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hq,hkv,s,d", [(4, 4, 100, 64), (8, 2, 333, 128), (3, 1, 1, 128)])
def test_prefill_entry_points(dev, general, dtype, hq, hkv, s, d):
    q, k, v = qkv(2, hq, s, d, dtype, dev, hkv=hkv)
    for causal in (False, True):
        for scale in (None, 0.3, -0.2):
            for f in (cuda_llm.flash_attention_forward, cuda_llm.flash_attention_forward_lse):
                _same(f(q, k, v, causal, scale), general(lambda: f(q, k, v, causal, scale)))
    nat = api._native()
    assert nat.flash_attention_forward(q, k, v, True, None) is not None
    o, lse = cuda_llm.flash_attention_forward_lse(q, k, v, True)
    do = torch.randn_like(q)
    _same(cuda_llm.flash_attention_backward(do, q, k, v, o, lse, True),
          general(lambda: cuda_llm.flash_attention_backward(do, q, k, v, o, lse, True)))
    cos, sin = torch.rand(s, d, device=dev), torch.rand(s, d, device=dev)
    _same(cuda_llm.fused_rope_flash_attention(q, k, v, cos, sin),
          general(lambda: cuda_llm.fused_rope_flash_attention(q, k, v, cos, sin)))
    # the general path's forms: offset data, integer flags and scales, other table types
    _same(cuda_llm.flash_attention_forward(_offset(q), _offset(k), v, 1, 1),
          cuda_llm.flash_attention_forward(q, k, v, True, 1.0))
    assert nat.flash_attention_forward(_offset(q), k, v, True, None) is None
    assert nat.flash_attention_forward(q, k, v, 1, None) is None
    _same(cuda_llm.flash_attention_backward(do.transpose(1, 2).contiguous().transpose(1, 2), q, k, v, o,
                                            lse.double(), True),
          cuda_llm.flash_attention_backward(do, q, k, v, o, lse, True))
    for bad in ((q[:, :, :, ::2], k, v), (q, k[:, :, :0], v), (q, k.half() if dtype != torch.float16 else k.float(), v)):
        with pytest.raises(RuntimeError):
            cuda_llm.flash_attention_forward(*bad)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 64), (32, 8, 128), (40, 2, 128)])
def test_decode_entry_points(dev, general, dtype, hq, hkv, d):
    nat = api._native()
    q = torch.randn(3, hq, 1, d, device=dev).to(dtype)
    k, v = (torch.randn(3, hkv, 1100, d, device=dev).to(dtype) for _ in range(2))
    _same(cuda_llm.flash_decode(q, k, v), general(lambda: cuda_llm.flash_decode(q, k, v)))
    kt = k.transpose(1, 2).contiguous().transpose(1, 2)
    assert nat.async_flash_decode(q, kt, v, None) is None
    _same(cuda_llm.flash_decode(q, kt, v, 0.1), cuda_llm.flash_decode(q, k, v, 0.1))
    for fp8, per_block in ((False, True), (True, True), (True, False)):
        c = build_paged([5, 1030, 0], hq, hkv, d, dtype, dev, fp8=fp8, per_block=per_block, pool=200)
        args = (c["query"], c["key_cache"], c["value_cache"])
        meta = (c["block_tables"], c["context_lens"])
        if fp8:
            f = lambda *x: cuda_llm.fp8_paged_attention(*x[:3], c["k_scale"], c["v_scale"], *x[3:])
            assert nat.fp8_paged_attention_forward(*args, c["k_scale"], c["v_scale"], *meta, None) is not None
            view = [args[0]] + [t.view(torch.float8_e4m3fn) for t in args[1:]]
            _same(f(*view, *meta), f(*args, *meta))
        else:
            f = cuda_llm.paged_attention
            assert nat.paged_attention_forward(*args, *meta, None) is not None
        _same(f(*args, *meta), general(lambda: f(*args, *meta)))
        _same(f(_offset(args[0]), *args[1:], meta[0].repeat(1, 2)[:, :meta[0].shape[1]], meta[1]), f(*args, *meta))
        with pytest.raises(RuntimeError, match="int32"):
            f(*args, meta[0].long(), meta[1])


@pytest.mark.gpu
@pytest.mark.parametrize("fp8,per_block", [(False, False), (True, False), (True, True)])
def test_append_and_debug_check(dev, general, monkeypatch, fp8, per_block):
    new = [torch.randn(2, 4, 3, 64, device=dev).half() for _ in range(2)]

    def run(lens_t, **kw):
        c = build_paged([30, 20], 8, 4, 64, torch.float16, dev, fp8=fp8, per_block=per_block, seed=3)
        sc = dict(k_scale=c["k_scale"], v_scale=c["v_scale"]) if fp8 else {}
        cuda_llm.paged_kv_append(*new, c["key_cache"], c["value_cache"], c["block_tables"], lens_t, **sc, **kw)
        return [c["key_cache"], c["value_cache"], *sc.values()]

    lens = torch.tensor([25, 13], dtype=torch.int32, device=dev)
    want = general(lambda: run(lens))
    _same(run(lens), want)
    _same(run(lens.long()), want)
    some = torch.tensor([1, 3], dtype=torch.int32, device=dev)
    _same(run(lens, new_lens=some), general(lambda: run(lens, new_lens=some)))
    if not fp8:
        c = build_paged([30, 20], 8, 4, 64, torch.float16, dev)
        args = (c["query"], c["key_cache"], c["value_cache"], c["block_tables"] + 1000, c["context_lens"])
        cuda_llm.paged_attention(*args)  # clamped
        monkeypatch.setenv("CUDA_LLM_CHECK_BLOCK_TABLES", "1")
        with pytest.raises(RuntimeError):
            cuda_llm.paged_attention(*args)


@pytest.mark.gpu
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
def test_microscaled(dev, general, out_dtype):
    x = mx_inputs(1, 2, 130, 128, dev)
    args = [x["q"], x["q_scale"], x["k"], x["k_scale"], x["v"], x["v_scale"]]
    f = lambda *a: cuda_llm.fused_microscaled_attention(*a, is_causal=True, out_dtype=out_dtype)
    assert api._native().fused_microscaled_attention(*args, True, None, False) is not None
    want = general(lambda: f(*args))
    _same(f(*args), want)
    _same(f(*[t.view(torch.float8_e8m0fnu) if i % 2 else t for i, t in enumerate(args)]), want)
    _same(f(*[_offset(t) if i == 0 else t for i, t in enumerate(args)]), want)
    with pytest.raises(RuntimeError, match="out_dtype"):
        cuda_llm.fused_microscaled_attention(*args, out_dtype=torch.float32)


@pytest.mark.gpu
def test_functorch_and_subclasses_go_the_general_way(dev):
    q, k, v = qkv(2, 2, 16, 64, torch.bfloat16, dev)
    nat = api._native()

    class Sub(torch.Tensor):
        pass

    assert nat.flash_attention_forward(q.as_subclass(Sub), k, v, False, None) is None
    seen = []

    def inner(x):
        seen.append(nat.flash_attention_forward(x, x, x, False, None))
        return x

    torch.func.vmap(inner)(q[None])
    torch.func.grad(lambda x: inner(x).float().sum())(q)
    assert seen == [None, None]
