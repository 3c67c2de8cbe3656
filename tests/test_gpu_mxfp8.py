"""GPU tier: fused_microscaled_attention (MXFP8) vs the oracle on the
dequantised tensors (tolerance max-abs 5e-2).

The reference declares this entry point but ships no kernel or test, so parity
is pinned by the OCP MX definition (golden vectors from float64 loops over the
decoded codes) rather than by a reference vector.
"""
import os

import numpy as np
import pytest
import torch

import cuda_llm
import oracle
from _util import TOL_FP8, assert_close, mx_inputs, to_np

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "golden.npz")


def _ref(x, heads=None):
    deq = {n: oracle.mx_dequantize(x[n].cpu().numpy(), x[n + "_scale"].cpu().numpy()) for n in "qkv"}
    if heads is not None:
        deq = {n: a[heads[0]:heads[0] + 1, heads[1]:heads[1] + 1] for n, a in deq.items()}
    return deq


def _run(x, causal, **kw):
    return cuda_llm.fused_microscaled_attention(x["q"], x["q_scale"], x["k"], x["k_scale"],
                                                x["v"], x["v_scale"], is_causal=causal, **kw)


def test_golden_mx(dev):
    g = np.load(GOLDEN, allow_pickle=False)
    c = {k.split("/", 1)[1]: g[k] for k in g.files if k.startswith("mx_causal/")}
    x = {n: torch.from_numpy(c[n]).to(dev) for n in ("q", "k", "v", "q_scale", "k_scale", "v_scale")}
    out = _run(x, bool(c["causal"]))
    torch.cuda.synchronize()
    assert_close(to_np(out), c["out"], **TOL_FP8, name="golden mx")


@pytest.mark.parametrize("s", [1, 100, 256, 777])
@pytest.mark.parametrize("causal", [False, True])
def test_mx_vs_oracle(dev, s, causal):
    x = mx_inputs(2, 3, s, 128, dev, seed=s)
    out = _run(x, causal)
    torch.cuda.synchronize()
    d = _ref(x)
    ref = oracle.attention(d["q"], d["k"], d["v"], is_causal=causal)
    assert_close(to_np(out), ref, **TOL_FP8, name=f"mx S={s}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("profile", ["ramp", "jump"])
def test_mx_running_max_growth(dev, causal, profile):
    """Logits that grow along the keys: tiles after a wave's first take their
    weights against the running max as it stands, and a tile whose bf16
    weights sum past 2^48 (ramp: about +33 log2 units per 64-key tile) or
    overflow (jump: +130 log2 units at key 512) takes the full max, rescale
    and weights again. The MX block scales carry the growing key norms."""
    g = torch.Generator(device="cpu").manual_seed(12)
    b, h, s, d = 1, 2, 1024, 128
    u = torch.randn(d, generator=g)
    u = u / u.norm()
    j = torch.arange(s, dtype=torch.float32)
    amp = 0.5 * j if profile == "ramp" else torch.where(j < 512, torch.ones_like(j),
                                                         torch.full_like(j, 130.0))
    raw = {"k": amp[:, None] * u + 0.1 * torch.randn(b, h, s, d, generator=g),
           "q": 8 * u + 0.1 * torch.randn(b, h, s, d, generator=g),
           "v": torch.randn(b, h, s, d, generator=g)}
    x = {}
    for n, t in raw.items():
        codes, sc = oracle.mx_quantize(t.numpy())
        x[n] = torch.from_numpy(codes).to(dev)
        x[n + "_scale"] = torch.from_numpy(sc).to(dev)
    out = _run(x, causal)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    dq = _ref(x)
    ref = oracle.attention(dq["q"], dq["k"], dq["v"], is_causal=causal)
    assert_close(to_np(out), ref, **TOL_FP8, name=f"mx {profile} causal={causal}")


def test_mx_scale_formats_agree(dev):
    """e8m0 bytes, float8_e8m0fnu and float powers of two give identical output."""
    x = mx_inputs(1, 2, 130, 128, dev, seed=3)
    a = _run(x, True)
    y = dict(x)
    for n in ("q_scale", "k_scale", "v_scale"):
        y[n] = torch.ldexp(torch.ones_like(x[n], dtype=torch.float32), x[n].to(torch.int32) - 127)
    b = _run(y, True)
    z = dict(x)
    for n in ("q_scale", "k_scale", "v_scale"):
        z[n] = x[n].view(torch.float8_e8m0fnu)
    c = _run(z, True)
    torch.cuda.synchronize()
    assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("causal", [False, True])
def test_mx_zero_scale_is_running_mean(dev, causal):
    """softmax_scale = 0: O is the running mean (causal) or the mean of the
    dequantised V rows, a closed form that needs no oracle."""
    x = mx_inputs(1, 2, 700, 128, dev)
    out = _run(x, causal, softmax_scale=0.0)
    torch.cuda.synchronize()
    v = torch.from_numpy(_ref(x)["v"]).to(dev).double()
    s = v.shape[2]
    if causal:
        ref = v.cumsum(2) / torch.arange(1, s + 1, device=dev, dtype=torch.float64)[:, None]
    else:
        ref = v.mean(2, keepdim=True).expand_as(v)
    assert_close(to_np(out), ref.cpu().numpy(), **TOL_FP8, name=f"mx zero scale causal={causal}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
def test_mx_negative_scale(dev, causal, out_dtype):
    """A negative softmax scale (the kernel takes |scale| on -Q, the codes'
    signs flipped per query tile, so every tile of a multi-tile grid, the
    first and the ones a walk's last iteration loads, is checked)."""
    x = mx_inputs(2, 3, 700, 128, dev, seed=7)
    out = _run(x, causal, softmax_scale=-0.06, out_dtype=out_dtype)
    torch.cuda.synchronize()
    d = _ref(x)
    ref = oracle.attention(d["q"], d["k"], d["v"], is_causal=causal, scale=-0.06)
    assert_close(to_np(out), ref, **TOL_FP8, name=f"mx scale -0.06 causal={causal}")


def test_mx_limits_fail_before_launch(dev):
    """seq_len >= 2^22 and a non-finite softmax scale are rejected with
    CA_INVALID_ARGUMENT before anything is launched (dummy pointers, never
    read)."""
    import ctypes
    from cuda_amd import _lib as L
    P = ctypes.c_void_p(256)
    lib = L.load()
    for s, sc in ((1 << 22, 0.1), (64, float("inf")), (64, float("nan"))):
        ws = lib.ca_mx_workspace_bytes(L.CA_SCALE_E8M0, 1, 1, s, 128)
        st = lib.ca_fused_microscaled_attention(L.CA_BF16, P, P, P, P, P, P, L.CA_SCALE_E8M0, P, 1, 1, s, 128,
                                                ctypes.c_float(sc), 1, P, ws, None)
        assert st == L.CA_INVALID_ARGUMENT, (s, sc)
    torch.cuda.synchronize()


def test_mx_fp16_output(dev):
    x = mx_inputs(1, 2, 64, 128, dev, seed=4)
    out = _run(x, False, out_dtype=torch.float16)
    torch.cuda.synchronize()
    d = _ref(x)
    assert_close(to_np(out), oracle.attention(d["q"], d["k"], d["v"]), **TOL_FP8, name="fp16 out")


@pytest.mark.parametrize("b,h,s,causal", [(1, 64, 2048, False), (2, 24, 3640, True)])
def test_mx_persistent_grid(dev, b, h, s, causal):
    """Grids of more than 256 work items (512 non-causal query tiles; 360
    causal pairs, the first tile of each head 64 rows): each workgroup of the
    persistent launch takes several, draining and refilling its ring between
    them. Sampled heads against the oracle."""
    x = mx_inputs(b, h, s, 128, dev, seed=s)
    out = _run(x, causal)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    for (bi, hi) in [(0, 0), (b - 1, h - 1)]:
        d = _ref(x, heads=(bi, hi))
        ref = oracle.attention(d["q"], d["k"], d["v"], is_causal=causal)
        assert_close(to_np(out[bi:bi + 1, hi:hi + 1]), ref, **TOL_FP8, name=f"head {bi},{hi}")


def test_baseline_c5_shape(dev):
    """C5: B=1, H=16, S=8192, D=128, causal; every head vs the oracle."""
    x = mx_inputs(1, 16, 8192, 128, dev, seed=0)
    out = _run(x, True)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    for h in range(16):
        d = _ref(x, heads=(0, h))
        ref = oracle.attention(d["q"], d["k"], d["v"], is_causal=True)
        assert_close(to_np(out[:, h:h + 1]), ref, **TOL_FP8, name=f"C5 head {h}")


def _abi_call(x, kind, scales, out, causal=True):
    """ca_fused_microscaled_attention through ctypes with the given scale
    tensors and scale kind; returns the status (no raise)."""
    import ctypes
    import cuda_amd._lib as L
    b, h, s, d = x["q"].shape
    ws = torch.empty(int(L.load().ca_mx_workspace_bytes(kind, b, h, s, d)), dtype=torch.uint8,
                     device=x["q"].device)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    return L.load().ca_fused_microscaled_attention(
        L.CA_BF16, p(x["q"]), p(scales[0]), p(x["k"]), p(scales[1]), p(x["v"]), p(scales[2]), kind,
        p(out), b, h, s, d, 1.0 / d ** 0.5, int(causal), p(ws), ws.numel(),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))


def _check_scales(x, scales):
    import ctypes
    import cuda_amd._lib as L
    b, h, s, d = x["q"].shape
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    return L.load().ca_check_mx_scales(p(scales[0]), p(scales[1]), p(scales[2]), b, h, s, d,
                                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))


def test_mx_float_scale_form_of_the_c_abi(dev):
    """The reference's float-scale interface (kernels_api.h:103-108) at the C
    ABI: float32 powers of two give the e8m0 form's output bit for bit. The
    call is asynchronous in both forms: a scale that is not such a power of
    two is taken as the e8m0 NaN, so the outputs it reaches are not
    meaningful, and the separate, synchronous ca_check_mx_scales reports it."""
    import cuda_amd._lib as L
    x = mx_inputs(2, 2, 300, 128, dev, seed=7)
    e8 = [x[n + "_scale"].contiguous() for n in "qkv"]
    f32 = [torch.ldexp(torch.ones_like(t, dtype=torch.float32), t.to(torch.int32) - 127) for t in e8]
    a = torch.full_like(x["q"], 0, dtype=torch.bfloat16)
    b = torch.full_like(a, 0)
    assert _abi_call(x, L.CA_SCALE_E8M0, e8, a) == L.CA_OK
    assert _abi_call(x, L.CA_SCALE_F32, f32, b) == L.CA_OK
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert _check_scales(x, f32) == L.CA_OK
    d = _ref(x)
    assert_close(to_np(b), oracle.attention(d["q"], d["k"], d["v"], is_causal=True), **TOL_FP8,
                 name="float scales")
    for bad, which in ((3.0, 0), (0.0, 1), (-0.5, 2), (float("nan"), 1), (0.75, 2)):
        sc = [t.clone() for t in f32]
        sc[which].view(-1)[123] = bad          # row 30 of head (0, 0), block 3
        assert _check_scales(x, sc) == L.CA_INVALID_ARGUMENT
        assert b"powers of two" in L.load().ca_last_error()
        out = torch.full_like(a, 7.0)
        assert _abi_call(x, L.CA_SCALE_F32, sc, out) == L.CA_OK
        torch.cuda.synchronize()
        # what the bad scale cannot reach equals the valid output bit for bit:
        # the other heads, and for q the other query rows (what it reaches is
        # not meaningful and is not pinned)
        same = out == b
        assert same[1].all() and same[0, 1].all()
        if which == 0:
            assert same[0, 0, :30].all() and same[0, 0, 31:].all() and not same[0, 0, 30].all()
    # the smallest and largest e8m0 values are accepted in float form
    sc = [t.clone() for t in f32]
    sc[1].view(-1)[5] = 2.0 ** -127
    sc[1].view(-1)[6] = 2.0 ** 127
    assert _check_scales(x, sc) == L.CA_OK
    assert _abi_call(x, L.CA_SCALE_F32, sc, torch.empty_like(a)) == L.CA_OK


def test_mx_scale_check_opt_in(dev, monkeypatch):
    """CUDA_LLM_CHECK_MX_SCALES=1 makes the Python entry check float scales
    first and raise; by default the call goes through (the row the bad q
    scale reaches is not meaningful, the others are unchanged)."""
    x = mx_inputs(1, 1, 64, 128, dev, seed=3)
    f32 = [torch.ldexp(torch.ones_like(x[n + "_scale"], dtype=torch.float32),
                       x[n + "_scale"].to(torch.int32) - 127) for n in "qkv"]
    f32[0].view(-1)[0] = 0.3
    monkeypatch.setenv("CUDA_LLM_CHECK_MX_SCALES", "0")
    good = [t.clone() for t in f32]
    good[0].view(-1)[0] = 1.0
    ref = cuda_llm.fused_microscaled_attention(x["q"], good[0], x["k"], good[1], x["v"], good[2], is_causal=True)
    out = cuda_llm.fused_microscaled_attention(x["q"], f32[0], x["k"], f32[1], x["v"], f32[2], is_causal=True)
    torch.cuda.synchronize()
    assert torch.equal(out[0, 0, 1:], ref[0, 0, 1:]) and not torch.equal(out[0, 0, 0], ref[0, 0, 0])
    monkeypatch.setenv("CUDA_LLM_CHECK_MX_SCALES", "1")
    with pytest.raises(RuntimeError, match="powers of two"):
        cuda_llm.fused_microscaled_attention(x["q"], f32[0], x["k"], f32[1], x["v"], f32[2], is_causal=True)


@pytest.mark.parametrize("b,h,s", [(1, 101, 1200), (3, 12, 2300), (4, 16, 1500)])
def test_mx_causal_tile_orders(dev, b, h, s):
    """253 pairs of 256-row tiles; single tiles, the longest of all heads first,
    for head counts that 8 does not and does divide: row 0 of every head is
    V's row 0, sampled heads against the oracle."""
    x = mx_inputs(b, h, s, 128, dev, seed=s)
    out = _run(x, True)
    torch.cuda.synchronize()
    v0 = oracle.mx_dequantize(x["v"][:, :, :1].cpu().numpy(), x["v_scale"][:, :, :1].cpu().numpy())
    assert_close(to_np(out[:, :, :1]), v0, **TOL_FP8, name="row 0")
    for heads in ((0, 0), (b - 1, h - 1)):
        d = _ref(x, heads)
        ref = oracle.attention(d["q"], d["k"], d["v"], is_causal=True)
        assert_close(to_np(out[heads[0]:heads[0] + 1, heads[1]:heads[1] + 1]), ref, **TOL_FP8, name=f"head {heads}")
