"""The native front end against the Python path behind it: bit-equal results
for every form both take, and hands off (None) everything else."""
import os
import subprocess
import sys

import pytest
import torch

from nanovllm_amd import _native
from nanovllm_amd import kernels as K

BF16 = torch.bfloat16


class _Absent:
    """A front end that takes no call: the Python path alone."""

    def __getattr__(self, name):
        return lambda *args: None


class _Sub(torch.Tensor):
    pass


def test_hands_off_what_is_not_an_ordinary_gpu_call():
    f = _native.load_front_end()
    x, w = torch.zeros(2, 8, dtype=BF16), torch.ones(8, dtype=BF16)
    assert f.rms_norm(x, w, 1e-6, None) is None                 # on the CPU
    assert f.rms_norm(x.as_subclass(_Sub), w, 1e-6, None) is None
    assert f.rms_norm(x.to("meta"), w.to("meta"), 1e-6, None) is None
    assert f.rms_norm(None, w, 1e-6, None) is None
    assert f.rms_norm(x, w, "eps", None) is None
    assert f.add_rms_norm(x, x, w, 1) is None
    assert f.silu_mul([1.0]) is None
    assert f.place(x) is None and f.merge_heads(x) is None
    with pytest.raises(TypeError):
        f.rms_norm(x)


def test_refusals_are_the_python_paths():
    x = torch.zeros(2, 8, dtype=BF16)
    with pytest.raises(ValueError, match="cuda"):
        K.rms_norm(x, torch.ones(8), 1e-6)
    with pytest.raises(ValueError, match="cuda"):
        K.silu_mul(x)
    with pytest.raises(ValueError, match="causal"):
        K.paged_attention_varlen(x, x, x, x, x, 1, 1, 1.0, x, causal=False)
    assert K.place(x) == (None, 16)
    assert K.merge_heads(torch.zeros(2, 3, 4)).shape == (2, 12)
    assert K.merge_heads(torch.zeros(0, 3, 4)).shape == (0, 12)


def _both(monkeypatch, call):
    """(through the front end, through the Python path); the front end must
    have taken the call itself."""
    front = _native.load_front_end()
    taken = []

    class Watch:
        def __getattr__(self, name):
            def fn(*args):
                got = getattr(front, name)(*args)
                taken.append(got is not None)
                return got
            return fn

    monkeypatch.setattr(K, "_front", _Absent())
    want = call()
    monkeypatch.setattr(K, "_front", Watch())
    got = call()
    assert taken and all(taken)
    return got, want


def _same(got, want):
    if isinstance(want, tuple):
        assert len(got) == len(want)
        for g, w in zip(got, want):
            _same(g, w)
        return
    assert got.shape == want.shape and got.stride() == want.stride() and got.dtype == want.dtype
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_rows_equal_the_python_path(cuda, monkeypatch):
    g = torch.Generator(device=cuda).manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF16)
    w = r(200)
    for x in (r(7, 200), r(7, 480)[:, 8:208], r(1, 200), r(9, 203)[:, 1:201], r(0, 200)):
        y = r(*x.shape)
        _same(*_both(monkeypatch, lambda: K.rms_norm(x, w, 1e-6)))
        out = torch.empty(x.shape[0], 400, dtype=BF16, device=cuda)[:, 200:]
        _same(*_both(monkeypatch, lambda: K.rms_norm(x, w, 1e-6, out=out).clone()))
        _same(*_both(monkeypatch, lambda: K.add_rms_norm(x, y, w, 1e-6)))
        _same(*_both(monkeypatch, lambda: K.add_then_rms_norm(x, y, w, 1e-6)))
        _same(*_both(monkeypatch, lambda: K.silu_mul(x)))
    table = torch.arange(1003, device=cuda) * 3
    logits = r(6, 1003)
    K.argmax_rows(logits)
    for x, m in ((logits, None), (logits, table), (r(6, 1010)[:, :1003], table)):
        _same(*_both(monkeypatch, lambda: K.argmax_rows(x, m)))
        out = torch.zeros(9, dtype=torch.int64, device=cuda)
        _same(*_both(monkeypatch, lambda: K.argmax_rows(x, m, out=out).clone()))


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("head_major", [False, True])
def test_attention_equals_the_python_path(cuda, monkeypatch, fp8, head_major):
    g = torch.Generator(device=cuda).manual_seed(4)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF16)
    hq, hkv, nb, bs = 8, 2, 11, 64
    kv = r(nb, hkv, 2, bs, 128).permute(2, 0, 3, 1, 4) if head_major else r(2, nb, bs, hkv, 128)
    kv = kv.to(torch.float8_e4m3fn) if fp8 else kv
    one = torch.ones(1, device=cuda)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=cuda)
    table = i32([[4, 9, 0, 2, 1], [7, 3, -1, -1, -1], [5, 6, 8, -1, -1]])
    qkv = r(9, (hq + 2 * hkv) * 128 + 16)
    qkv = qkv[:, : (hq + 2 * hkv) * 128]
    pos = torch.tensor([5, 6, 7, 0, 3, 9, 10, 11, 12], device=cuda)
    cos = torch.randn(64, 128, generator=g, device=cuda)
    slots = i32([300, 301, 302, -1, 40, 500, 501, 502, nb * bs + 3])
    k, v = kv[0].clone(), kv[1].clone()
    norms = (r(128), r(128))
    for qn, kn in (norms, (None, None)):
        for ks, vs in ((None, None), (one * 0.5, one * 2)):
            def store():
                k.copy_(kv[0])
                v.copy_(kv[1])
                q = K.qk_norm_rope_store(qkv, pos, qn, kn, cos, hq, hkv, 128, 1e-6, k, v, slots, ks, vs)
                return q, k.float(), v.float()
            _same(*_both(monkeypatch, store))
    k, v = kv[0], kv[1]                   # the layout's own strides
    q = r(9, hq, 128)
    for args in ((i32([0, 3, 4, 9]), i32([0, 300, 410, 600]), 5, 320),
                 (i32([0, 1, 1, 9]), i32([0, 260, 270, 460]), 8, 300)):
        for scales in ({}, dict(k_scale=one * 0.5, v_scale=one)):
            varlen = lambda out=None: K.paged_attention_varlen(q, k, v, *args, 128 ** -0.5, table,
                                                               out=out, **scales)
            varlen()                      # the workspace is the Python path's to grow
            _same(*_both(monkeypatch, varlen))
            out = torch.zeros(9, hq, 256, dtype=BF16, device=cuda)[:, :, :128]
            _same(*_both(monkeypatch, lambda: varlen(out).clone()))
    lens = i32([310, 0, 190])
    for bound in (None, 320):
        decode = lambda: K.paged_attention_decode(q[:3], k, v, lens, table, 128 ** -0.5, bound,
                                                  k_scale=one, v_scale=one)
        decode()
        _same(*_both(monkeypatch, decode))


@pytest.mark.gpu
def test_sizes_past_32_bits_are_handed_off(cuda):
    """More rows than a C-ABI count holds (views of one row, no memory behind
    them): the front end hands the call back with the interpreter as it was,
    and the Python path refuses it."""
    f = _native.load_front_end()
    row = torch.ones(1, 8, device=cuda).to(BF16)
    w, out = torch.ones(8, device=cuda).to(BF16), torch.zeros(1, 8, device=cuda).to(BF16)
    n = 2 ** 31
    assert f.rms_norm(row.expand(n, 8), w, 1e-6, out.expand(n, 8)) is None
    with pytest.raises(ValueError):
        K.rms_norm(row.expand(n, 8), w, 1e-6, out=out.expand(n, 8))
    assert f.silu_mul(row.expand(n, 8)) is None
    assert f.add_rms_norm(row.expand(n, 8), row.expand(n, 8), w, 1e-6) is None
    assert f.argmax_rows(row.expand(n, 8), None, None, {}) is None
    assert K.rms_norm(row, w, 1e-6).shape == (1, 8)


LINEAR_SHAPES = [
    # rows around the 16-row tiles and the limit, K of one chunk, fewer chunks
    # than waves, a remainder of waves and of depth, N short of a tile
    (1, 16, 64), (2, 20, 128), (15, 64, 448), (16, 6144, 576), (17, 1024, 1600), (31, 100, 3072),
    (32, 6148, 256), (33, 4096, 1024), (48, 48, 64), (64, 6160, 2048), (7, 12288, 1024),
    (9, 12300, 512), (64, 1024, 16384),
]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", LINEAR_SHAPES)
def test_linear_rows_against_64_bits(cuda, m, n, k):
    """nva_linear over every tile shape: half a bf16 ulp of the result (bf16 has 8
    significant bits: at most 2^-8 of the value, rounded up to 1.01 of it here)
    plus fp32 sums of K terms, within (K / 32) 2^-24 of the sum of magnitudes
    (32 products a matrix instruction, chained)."""
    g = torch.Generator(device=cuda).manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=g, device=cuda).to(BF16)[:, :k]
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF16)
    guard = torch.full((m + 1, n + 4), 7.0, dtype=BF16, device=cuda)
    lib = _native.load()
    _native.check(lib.nva_linear(x.data_ptr(), x.stride(0), w.data_ptr(), guard.data_ptr(),
                                 guard.stride(0), m, n, k, K._stream()), "linear")
    want = x.double() @ w.double().t()
    bound = want.abs() * 1.01 * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * (k / 32) * 2.0 ** -24
    assert bool(((guard[:m, :n].double() - want).abs() <= bound + 1e-30).all())
    assert bool((guard[m:] == 7).all()) and bool((guard[:, n:] == 7).all())   # nothing else written
    got = K.linear(x, w)
    assert got.shape == (m, n) and got.is_contiguous()
    assert bool(((got.double() - want).abs() <= bound + 1e-30).all())


def test_where_the_few_row_kernel_is_preferred():
    """The lines of nva_linear_preferred, both sides of each."""
    f = _native.load().nva_linear_preferred
    yes = [(1, 16, 64), (1, 4096, 4096), (12, 5120, 4096), (16, 4096, 4096), (16, 24576, 4096),
           (16, 5120, 2048), (16, 6144, 3584), (16, 7168, 4096), (17, 4096, 4096), (32, 1024, 3072),
           (32, 5120, 2048), (32, 8192, 3072), (33, 4096, 2048), (64, 4096, 1024), (64, 6144, 2048),
           (64, 8192, 2048), (1, 512, 16448), (32, 5120, 25600), (32, 512, 32768), (64, 5120, 25600),
           (64, 2048, 20480)]
    no = [(0, 4096, 4096), (65, 4096, 1024), (-1, 16, 64), (1, 12, 64), (1, 18, 64), (1, 16, 32),
          (1, 16, 96), (1, 16, 0), (1, 4096, 4160), (16, 4096, 16384), (1, 64, 16448), (1, 508, 20480),
          (1, 6148, 32768), (1, 5120, 20416), (1, 1024, 32832), (13, 5120, 2112), (13, 6144, 4096),
          (17, 4100, 2112), (32, 6144, 3072), (32, 8192, 4096), (32, 8196, 64), (33, 1024, 2048),
          (33, 5120, 1024), (33, 4096, 2112), (64, 8196, 1024), (64, 1024, 20480), (33, 5120, 27648),
          (64, 1024, 16384)]
    for m, n, k in yes:
        assert f(m, n, k) == 1, (m, n, k)
    for m, n, k in no:
        assert f(m, n, k) == 0, (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (7, 12288, 1024), (16, 6144, 576), (17, 1024, 1600),
                                   (32, 4096, 4096), (33, 4096, 1024), (2, 512, 17408),
                                   (33, 1024, 2048), (16, 4096, 8192), (65, 4096, 1024)])
def test_linear_runs_where_it_is_preferred(cuda, m, n, k):
    """K.linear is the few-row kernel where nva_linear_preferred says so (its
    sums have one order, so its bits) and the library's product elsewhere."""
    g = torch.Generator(device=cuda).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=cuda).to(BF16)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF16)
    lib = _native.load()
    want = torch.nn.functional.linear(x, w)
    if lib.nva_linear_preferred(m, n, k):
        want = torch.empty_like(want)
        _native.check(lib.nva_linear(x.data_ptr(), k, w.data_ptr(), want.data_ptr(), n, m, n, k,
                                     K._stream()), "linear")
    assert torch.equal(K.linear(x, w), want)


@pytest.mark.gpu
def test_linear_takes_every_form_the_library_takes(cuda):
    import torch.nn.functional as F

    x, w = torch.randn(5, 128, device=cuda), torch.randn(32, 128, device=cuda)
    b = torch.randn(32, device=cuda).to(BF16)
    xb, wb = x.to(BF16), w.to(BF16)
    assert torch.equal(K.linear(x, w), F.linear(x, w))                       # float32
    assert torch.equal(K.linear(xb, wb, b), F.linear(xb, wb, b))             # bias
    three = xb.view(1, 5, 128).expand(2, 5, 128)
    assert torch.equal(K.linear(three, wb), F.linear(three, wb))
    odd = torch.randn(32, 129, device=cuda).to(BF16)[:, 1:]
    assert torch.equal(K.linear(xb, odd), F.linear(xb, odd))                 # strided, misaligned
    wg = w.clone().requires_grad_()
    K.linear(x, wg).sum().backward()
    assert wg.grad is not None
    wg = wb.clone().requires_grad_()
    K.linear(xb, wg).sum().backward()
    assert wg.grad is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert K.linear(xb, wb).dtype == torch.float16
    tangent = torch.autograd.forward_ad
    with tangent.dual_level():
        d = K.linear(tangent.make_dual(xb, xb), wb)
        assert tangent.unpack_dual(d).tangent is not None
    rows = torch.vmap(lambda r: K.linear(r, wb))(xb.view(5, 1, 128))
    assert rows.shape == (5, 1, 32)
    seen = []

    class Log(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, fn, types, args=(), kwargs=None):
            seen.append(fn)
            return fn(*args, **(kwargs or {}))

    with Log():
        K.linear(xb, wb)
    assert seen
    with pytest.raises(RuntimeError):
        K.linear(xb, wb[:, :64])


@pytest.mark.gpu
def test_other_forms_still_run(cuda):
    """Host lengths, a scale or bound of another number type: the Python path
    takes them behind the front end."""
    q = torch.randn(2, 4, 128, device=cuda).to(BF16)
    kv = torch.randn(2, 2, 32, 2, 128, device=cuda).to(BF16)
    table = torch.tensor([[0], [1]], dtype=torch.int32, device=cuda)
    lens = torch.tensor([20, 31], dtype=torch.int32)
    want = K.paged_attention_decode(q, kv[0], kv[1], lens.to(cuda), table, 0.5, 32)
    import numpy as np
    for n, s, b in ((lens, 0.5, 32), (lens.tolist(), 0.5, 32), (lens.to(cuda), np.float64(0.5), 32),
                    (lens.to(cuda), 0.5, np.int64(32))):
        assert torch.equal(K.paged_attention_decode(q, kv[0], kv[1], n, table, s, b), want)
    with pytest.raises(ValueError):
        K.paged_attention_decode(q, kv[0], kv[1], lens.tolist(), table, 0.5, 16)


def test_loads_in_a_process_that_has_not_imported_torch():
    """As a build check does: the module's own libraries include torch's."""
    code = "from nanovllm_amd import _native; _native.load_front_end()"
    pkg = os.path.dirname(os.path.dirname(os.path.abspath(_native.__file__)))
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300,
                   env={**os.environ, "PYTHONPATH": pkg})


def test_a_module_of_another_torch_or_python_is_refused(monkeypatch):
    """Its ABI is the interpreter's and torch's it was built against."""
    _native.load_front_end()
    monkeypatch.setattr(_native, "_front", None)
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "0.0.1")
        with pytest.raises(_native.NativeLibraryError, match="0.0.1.*build it again"):
            _native.load_front_end()
    with monkeypatch.context() as m:
        m.setattr(_native.sys, "hexversion", 0x03000000)
        with pytest.raises(_native.NativeLibraryError, match="0x300.*build it again"):
            _native.load_front_end()
    assert _native.load_front_end().built_for_torch == torch.__version__


def test_the_front_end_is_built_again_when_torch_changes(tmp_path):
    """make would run the module's rule for another interpreter's torch."""
    fake = tmp_path / "torch"
    fake.mkdir()
    (fake / "__init__.py").write_text("")
    (fake / "version.py").write_text("__version__ = '9.9.9'\n")
    out = subprocess.run(["make", "-n", "-C", _native.CSRC_DIR, f"PYTHON={sys.executable}"],
                         env={**os.environ, "PYTHONPATH": str(tmp_path)}, capture_output=True, text=True,
                         check=True, timeout=120).stdout
    assert "9.9.9" in out and f"-I{fake}" not in out and f"{fake}/include" in out
