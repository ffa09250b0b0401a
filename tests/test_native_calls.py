"""innova_amd._native (csrc/native_calls.cpp): the ordinary form of a call runs as one C function, everything else goes the way through
Python.  Both ways have to give the same results, errors included."""
import numpy as np
import pytest
import torch

import innova_amd as ia
from innova_amd import _lib, kernel, layers


class _Python:
    """Stands for the native module and takes nothing."""

    def __getattr__(self, name):
        return lambda *a: None


def _calls():
    rng = np.random.default_rng(5)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    w = {f: ia.DeviceWeights.quantize((rng.standard_normal(n * k) * 0.02).astype(np.float32), np.full(n * k // 256, int(ia.Format[f]), np.uint8), n, k)
         for f, n, k in (("OIL4", 40, 512), ("OIL8", 40, 512))}
    gu = ia.DeviceWeights.quantize((rng.standard_normal(512 * 512) * 0.02).astype(np.float32), np.full(1024, int(ia.Format.OIL4), np.uint8), 512, 512)
    down = ia.DeviceWeights.quantize((rng.standard_normal(512 * 256) * 0.02).astype(np.float32), np.full(512, int(ia.Format.OIL4), np.uint8), 512, 256)
    x, nw = dev(rng.standard_normal((4, 512)).astype(np.float32)), dev(rng.standard_normal(512).astype(np.float32) * 0.1)
    codes, act = dev(rng.integers(0, 256, 64 * 96, dtype=np.uint8)), dev(rng.standard_normal((64, 96)).astype(np.float32))
    cb8, cb4 = dev(rng.standard_normal(256).astype(np.float32)), dev(rng.standard_normal(16).astype(np.float16).view(np.int16))
    out = torch.empty(4, 40, device="cuda")
    o4 = w["OIL4"]
    cases = {
        "gemv1": lambda: o4.gemv(x[:1]), "gemv4": lambda: o4.gemv(x), "gemv 3d": lambda: o4.gemv(x.reshape(2, 2, 512)), "gemv out": lambda: o4.gemv(x, out=out),
        "gemv flat": lambda: o4.gemv(x[0]), "gemv grad": lambda: o4.gemv(x.clone().requires_grad_()),
        "gemv other": lambda: w["OIL8"].gemv(x[:3]), "bf16": lambda: o4.gemm_bf16(x.to(torch.bfloat16)), "f32": lambda: w["OIL8"].gemm_f32(x),
        "dequant": lambda: o4.dequant(), "embed": lambda: layers.embed_rows(o4, torch.tensor([3, 39, 0], dtype=torch.int32, device="cuda")),
        "norm1": lambda: layers.gemv_rmsnorm(o4, x[:1], nw), "norm4": lambda: layers.gemv_rmsnorm(o4, x, nw),
        "mlp": lambda: layers.mlp_step(gu, down, x[:2], norm_w=nw), "mlp plain": lambda: layers.mlp_step(gu, down, x[0]),
        "oil8": lambda: kernel.oil8_gemm(codes, cb8, act, 3, 64, 96), "oil4": lambda: kernel.oil4_gemm(codes, cb4, act, 2, 64, 96),
        "spark": lambda: kernel.gemv_spark_batch(codes, 0.5, act, 64, 2, 96), "prod4": lambda: kernel.gemv_oil4_batch(codes, cb4, 0.5, act, 64, 2, 96),
        "prod8": lambda: kernel.gemv_oil8_batch(codes, cb8, 1, act, 64, 2, 96), "engine": lambda: kernel.engine_quant_gemm(4, act, codes, cb8, 2, 64, 96),
        # refused or unusual: the way through Python decides
        "dtype": lambda: o4.gemv(x.half()), "strided": lambda: o4.gemv(x[:, ::2].expand(4, 256)), "not rows": lambda: o4.gemv(x[0, :300].clone()),
        "empty": lambda: o4.gemv(x[:0]), "cpu": lambda: o4.gemv(x.cpu()), "out size": lambda: o4.gemv(x, out=out[:3]), "out type": lambda: o4.gemv(x, out=out.half()),
        "numpy": lambda: kernel.oil8_gemm(codes.cpu().numpy(), cb8.cpu().numpy(), act.cpu().numpy(), 3, 64, 96),
        "numpy ints": lambda: kernel.oil8_gemm(codes, cb8, act, np.int64(3), 64, 96), "bits": lambda: kernel.engine_quant_gemm(3, act, codes, cb8, 2, 64, 96),
        "book": lambda: kernel.engine_quant_gemm(8, act, codes, cb8[:16], 2, 64, 96), "negative": lambda: kernel.oil8_gemm(codes, cb8, act, -1, 64, 96),
    }
    return cases


def _outcome(f):
    try:
        r = f()
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)
    torch.cuda.synchronize()
    return (tuple(r.shape), str(getattr(r, "dtype", "")), bool(getattr(r, "requires_grad", False)), np.asarray(r.cpu() if isinstance(r, torch.Tensor) else r).tobytes())


@pytest.mark.gpu
def test_same_results_and_errors_as_through_python(monkeypatch):
    for name, f in _calls().items():
        monkeypatch.setattr(_lib, "_native", None)
        native = _outcome(f)
        monkeypatch.setattr(_lib, "_native", _Python())
        assert native == _outcome(f), name


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dim,prompt", [(2, 80, 5), (3, 27, 2)])
def test_cache_both_ways(monkeypatch, heads, dim, prompt):
    g = torch.Generator(device="cuda").manual_seed(1)
    k, v = (torch.randn(1, heads, prompt, dim, generator=g, device="cuda") for _ in range(2))
    got = []
    for native in (None, _Python()):
        monkeypatch.setattr(_lib, "_native", native)
        c = ia.OIL4KVCache(1, prompt + 1, heads, dim, 32)
        c.append(0, k, v)
        c.append(0, k[:, :, :1].contiguous(), v[:, :, :1].contiguous())
        c.append(7, k, v)                                  # no such layer: ignored
        outs = [t.cpu() for r in ((0, prompt + 1), (1, prompt), (0, prompt + 9), (3, 3), (2, 1)) for t in c.get_range(0, *r)]
        with pytest.raises(AssertionError):
            c.append(0, k[0], v[0])
        got.append([(tuple(t.shape), t.numpy().tobytes()) for t in outs])
    assert got[0] == got[1]


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("heads,dim", [(2, 80), (3, 27)])
def test_cache_that_is_not_full(monkeypatch, native, heads, dim):
    """get_all() and a range past the tokens held: one decode, and outputs of the tokens held alone."""
    monkeypatch.setattr(_lib, "_native", None if native else _Python())
    c, held = ia.OIL4KVCache(2, 4096, heads, dim, 64), 6
    k, v = (torch.randn(1, heads, held, dim, device="cuda") for _ in range(2))
    c.append(1, k, v)
    wk, wv = c.get_range(1, 0, held)
    calls, lib = [], _lib.lib()
    if native:                                            # the whole call is the C function's
        monkeypatch.setattr(_lib, "lib", lambda: pytest.fail("the way through Python was taken"))
    else:
        class Counting:
            def __getattr__(self, name):
                calls.append(name)
                return getattr(lib, name)
        monkeypatch.setattr(_lib, "lib", Counting)
    for start, end in ((0, None), (2, 4096), (held - 1, held + 1)):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        calls.clear()
        gk, gv = c.get_all(1) if end is None else c.get_range(1, start, end)
        n = held - start
        assert torch.cuda.max_memory_allocated() - before <= 2 * (n * heads * dim * 4 + 512)
        assert native or calls.count("oilhip_kv_get_range") == 1
        assert gk.shape == gv.shape == (1, heads, n, dim)
        flat = lambda t: t.reshape(-1, heads * dim)  # noqa: E731
        assert torch.equal(flat(gk), flat(wk)[start:]) and torch.equal(flat(gv), flat(wv)[start:])
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    for empty in (c.get_all(0), c.get_all(2), c.get_range(1, held, held + 3), c.get_range(1, held + 2, 4096)):
        assert all(t.shape == (1, heads, 0, dim) for t in empty)
    for bad in ((-1, 0, 3), (1, -1, 3)):
        with pytest.raises(ia.OilHipError, match="negative layer or start"):
            c.get_range(*bad)


@pytest.mark.gpu
def test_function_modes_and_subclasses_go_through_python(monkeypatch):
    """A torch function mode sees the calls that it saw before, and so does a tensor subclass."""
    from torch.overrides import TorchFunctionMode
    f = _calls()["gemv4"]
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    want = f()
    with Mode():
        got = f()
    assert "new_empty" in seen and torch.equal(got, want)


def test_takes_only_the_ordinary_form():
    """Without a GPU every call is left to Python, whatever its arguments are."""
    n = _lib.native()
    x = torch.zeros(1, 256)
    assert n.gemv(0, x, None, 1, 256) is None and n.gemv(8, x, None, 1, 256) is None and n.gemv(8, np.zeros(256), None, 1, 256) is None
    assert n.gemv("a", x, None, 1, 256) is None and n.gemv(1 << 80, x, None, 1, 256) is None
    assert n.kv_append(8, 0, x, x, 256) is None and n.kv_get_range(8, 0, 4, 4, 9, 1, 1) is None
    with pytest.raises(TypeError):
        n.gemv(8, x)
