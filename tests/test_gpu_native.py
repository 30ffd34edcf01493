"""The native host fast paths (csrc/native.cpp) against the Python forms of the
same calls: the same launches, so bit-equal results, over the layouts both
take; and what the fast paths leave to the Python forms is still taken or
refused there."""
import ctypes

import pytest
import torch

from dllm_serve_amd import _capi
from dllm_serve_amd.engine.sampler import RemaskSampler
from dllm_serve_amd.engine.sequence import PageAllocator, Sequence, prepare_step
from dllm_serve_amd.layers.attention import Attention
from dllm_serve_amd.layers.rotary_embedding import RotaryEmbedding
from dllm_serve_amd.sparse.state import SparseConfig
from dllm_serve_amd.utils.context import reset_context

pytestmark = pytest.mark.gpu
D = 128


@pytest.fixture
def both(monkeypatch):
    """Runs a call with the native module and without it."""
    assert _capi.native is not None, "the native module is not built"
    native = _capi.native

    def run(f):
        monkeypatch.setattr(_capi, "native", native)
        a = f()
        monkeypatch.setattr(_capi, "native", None)
        b = f()
        monkeypatch.setattr(_capi, "native", native)
        return a, b

    return run


@pytest.mark.parametrize("state", [0, 2])
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (14, 2)])
def test_attention_layouts(dev, both, state, Hq, Hkv):
    cfg = SparseConfig(enabled=True, default_block_len=32, retention_ratio=0.5)
    seqs = [Sequence([1] * p, 64, 7, cfg if state else None, device=dev) for p in (40, 333)]
    alloc = PageAllocator(range(8))
    for s in seqs:
        for _ in range(state):
            s.advance()
        alloc.allocate(s)
    attn = Attention(Hq, D, D ** -0.5, Hkv, causal=False)
    g = torch.Generator(device=dev).manual_seed(Hq + state)
    attn.k_cache, attn.v_cache = (torch.randn(8, 256, Hkv, D, generator=g, device=dev).bfloat16() for _ in range(2))
    n = sum(s.step_rows()[1] for s in seqs)
    fused = torch.randn(n, (Hq + 2 * Hkv) * D + 16, generator=g, device=dev).bfloat16()
    q, k, v = fused[:, :Hq * D], fused[:, Hq * D:(Hq + Hkv) * D], fused[:, (Hq + Hkv) * D:(Hq + 2 * Hkv) * D]
    shapes = {"slices": (q, k, v), "2d": tuple(x.contiguous() for x in (q, k, v)),
              "3d": (q.contiguous().view(n, Hq, D), k.view(n, Hkv, D), v.contiguous().view(n, Hkv, D)),
              "flat": tuple(x.contiguous().view(-1) for x in (q, k, v))}
    prepare_step(seqs, dev)
    try:
        for name, x in shapes.items():
            a, b = both(lambda: attn(*x))
            assert a.shape == b.shape == (n, Hq * D) and a.stride() == b.stride(), name
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), name
        for bad in ((q[1:], k, v), (q.float(), k, v), (q, k, v.cpu())):
            with pytest.raises((ValueError, TypeError, RuntimeError)):
                attn(*bad)
        if state:
            attn.k_cache = attn.k_cache.float()
            with pytest.raises(ValueError):
                attn(q, k, v)
    finally:
        reset_context()


@pytest.mark.parametrize("inplace", [False, True])
def test_rope_layouts(dev, both, inplace):
    rope = RotaryEmbedding(D, D, 64, 10000.0, inplace=inplace).to(dev)
    g = torch.Generator(device=dev).manual_seed(3)
    fused = torch.randn(9, 6 * D, generator=g, device=dev).bfloat16()
    pos = torch.randint(0, 64, (9,), generator=g, device=dev)
    for p in (pos, pos.to(torch.int32), torch.stack([pos, pos], 1)[:, 0]):
        for view in (lambda x: x, lambda x: x.unflatten(1, (-1, D))):
            def call():
                f = fused.clone()
                return rope(p, view(f[:, :4 * D]), view(f[:, 4 * D:]))
            (qa, ka), (qb, kb) = both(call)
            assert qa.shape == qb.shape and qa.stride() == qb.stride()
            assert torch.equal(qa, qb) and torch.equal(ka, kb)
    # in place is asked for by any true value
    rope.inplace = int(inplace)
    (qa, ka), (qb, kb) = both(call)
    assert torch.equal(qa, qb) and torch.equal(ka, kb)
    f = fused.clone()
    rope(pos, f[:, :4 * D], f[:, 4 * D:])
    assert torch.equal(f, fused) != inplace
    rope.head_size = 1 << 64  # past every C integer: left to the Python form, which refuses it
    with pytest.raises((ValueError, TypeError, RuntimeError)):
        rope(pos, fused[:, :4 * D], fused[:, 4 * D:])
    rope.head_size = D
    with pytest.raises(ValueError):
        rope(pos, fused.float(), fused)


def test_sampler_calls(dev, both):
    g = torch.Generator(device=dev).manual_seed(5)
    logits = torch.randn(48, 4104, generator=g, device=dev).bfloat16()[:, :4096]
    s = RemaskSampler(lambda h: logits, 9)
    (xa, pa), (xb, pb) = both(lambda: s.logits_max(torch.empty(48, 8, device=dev)))
    assert torch.equal(xa, xb) and torch.equal(pa, pb) and pa.dtype == torch.bfloat16
    bad = RemaskSampler(lambda h: logits.float(), 9)
    with pytest.raises(ValueError):
        bad.logits_max(torch.empty(48, 8, device=dev))


def _pend_hip_error():
    """Leaves an error of an unrelated host call pending, as any library may:
    the next check after a launch reports it, with the launch on the stream."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    hip = ctypes.CDLL(path)
    assert hip.hipSetDevice(1 << 20) != 0 and hip.hipPeekAtLastError() != 0


def test_runtime_error_after_a_launch_is_raised_once(dev):
    """A HIP error reported behind a launch raises; the call does not run a
    second time (rope in place would rotate twice, unmasking go on)."""
    assert _capi.native is not None, "the native module is not built"
    rope = RotaryEmbedding(D, D, 64, 10000.0).to(dev)
    ref = RotaryEmbedding(D, D, 64, 10000.0, inplace=False).to(dev)
    g = torch.Generator(device=dev).manual_seed(8)
    q, k = (torch.randn(5, n * D, generator=g, device=dev).bfloat16() for n in (4, 2))
    pos = torch.arange(5, device=dev)
    want = ref(pos, q, k)
    rope.inplace = True
    torch.cuda.synchronize()
    _pend_hip_error()
    with pytest.raises(RuntimeError, match="dllm_rope_neox failed"):
        rope(pos, q, k)
    assert torch.equal(q, want[0]) and torch.equal(k, want[1])

    tok = torch.full((1, 16), 9, dtype=torch.int64, device=dev)
    prm = torch.tensor([[0, 16, 0, 4, 0]], dtype=torch.int32, device=dev)
    x0 = torch.arange(100, 116, device=dev)
    conf = torch.rand(16, generator=g, device=dev).bfloat16()
    logits = torch.randn(16, 64, generator=g, device=dev).bfloat16()
    torch.cuda.synchronize()
    _pend_hip_error()
    with pytest.raises(RuntimeError, match="dllm_lowconf_unmask failed"):
        # (None would have sample_device_windows unmask a second time)
        _capi.native.unmask(tok, prm, 16, x0, conf, 9)
    assert int((tok != 9).sum()) == 4  # ceil(16 / 4): one step

    _pend_hip_error()
    with pytest.raises(RuntimeError, match="dllm_softmax_max failed"):
        RemaskSampler(lambda h: logits, 9).logits_max(logits)

    seqs = [Sequence([1] * 24, 8, 9, None, device=dev)]
    prepare_step(seqs, dev)
    try:
        attn = Attention(4, D, D ** -0.5, 4, causal=False)
        x = torch.randn(32, 4 * D, generator=g, device=dev).bfloat16()
        attn(x, x, x)
        torch.cuda.synchronize()
        _pend_hip_error()
        with pytest.raises(RuntimeError, match="dllm_attn_varlen_fwd failed"):
            attn(x, x, x)
        assert attn(x, x, x).shape == (32, 4 * D)
    finally:
        reset_context()
