"""innova_amd._native under torch.func's transforms: their tensors are exact torch tensors without storage, whose data_ptr() raises.
A build of csrc/native_calls.cpp that takes host tensors, over a library that does nothing, shows on a machine without a GPU that the
interpreter keeps its lock and every call is left to Python."""
import os
import re
import subprocess
import sys
import sysconfig

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALLS = """
import sys, threading
import torch
sys.path.insert(0, sys.argv[1])
import _native as n
x = torch.randn(3, 2, 256)
cb = torch.zeros(256)
made = {"gemv": lambda x: n.gemv(8, x, None, 4, 256), "gemv out": lambda x: n.gemv(8, x, torch.empty(2, 4), 4, 256),
        "gemm": lambda x: n.gemm(8, x, None, 4, 256, 0), "norm": lambda x: n.gemv_rmsnorm(8, x, cb, None, 4, 256),
        "norm weights": lambda x: n.gemv_rmsnorm(8, torch.ones(2, 256), x, None, 4, 256),
        "mlp": lambda x: n.mlp_step(8, 8, x, None, None, 4, 256, 256), "mlp norm": lambda x: n.mlp_step(8, 8, torch.ones(1, 256), x, None, 4, 256, 256),
        "oil8": lambda x: n.oil8_gemm(x, cb, x, 1, 2, 256), "oil4": lambda x: n.oil4_gemm(cb, cb, x, 1, 2, 256),
        "spark": lambda x: n.prod(2, cb, None, 0.5, x, 2, 1, 256), "prod4": lambda x: n.prod(4, cb, x, 0.5, x, 2, 1, 256),
        "prod8": lambda x: n.prod(8, x, cb, 0.5, x, 2, 1, 256), "engine": lambda x: n.engine_quant_gemm(8, x, cb, cb, 1, 2, 256),
        "append": lambda x: n.kv_append(8, 0, x.reshape(1, 1, 2, 256), x.reshape(1, 1, 2, 256), 256)}
for name, f in made.items():
    print(name, flush=True)
    got = f(x[0].clone())
    assert got is True or isinstance(got, torch.Tensor), (name, got)          # the build does take host tensors
    seen = []
    def call(t):
        seen.append(f(t))
        return (t * 1.0).sum()
    torch.func.vmap(call)(x)
    torch.func.grad(call)(x[0].clone())
    torch.func.jvp(call, (x[0].clone(),), (x[0].clone(),))
    assert len(seen) == 3 and all(r is None for r in seen), (name, seen)
    t = threading.Thread(target=lambda: seen.append(sum(range(1000))))         # the lock can still be taken and given back
    t.start()
    t.join()
ids = torch.tensor([[0, 1], [1, 0]], dtype=torch.int32)
seen = []
def call(t):
    seen.append(n.embed_rows(8, t, 256))
    return t * 2
torch.func.vmap(call)(ids)
assert seen == [None] and isinstance(n.embed_rows(8, ids[0], 256), torch.Tensor)
print("all calls returned")
"""


@pytest.fixture(scope="module")
def host_build(tmp_path_factory):
    d = tmp_path_factory.mktemp("native_calls")
    src = open(os.path.join(ROOT, "innova_amd", "csrc", "native_calls.cpp")).read()
    used = sorted(set(re.findall(r"\boilhip_[a-z0-9_]+", src)))
    for was, now in (("t.is_cuda() && t.is_contiguous()", "t.is_contiguous()"),
                     ("return c10::hip::getCurrentHIPStream().stream();", "return nullptr;"),
                     ("void need_no_capture(void* s) {", "void need_no_capture(void* s) {\n    return;"),
                     ('"../../include/oilhip.h"', f'"{ROOT}/include/oilhip.h"')):
        assert src.count(was) == 1, was
        src = src.replace(was, now)
    (d / "native_calls.cpp").write_text(src)
    (d / "library.cpp").write_text("".join(f'extern "C" long {f}() {{ return 0; }}\n' for f in used))
    t = os.path.dirname(torch.__file__)
    subprocess.run(["g++", "-O0", "-std=c++20", "-fPIC", "-shared", "-w", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1", "-isystem", f"{t}/include", "-isystem",
                    f"{t}/include/torch/csrc/api/include", "-isystem", "/opt/rocm/include", "-isystem", sysconfig.get_paths()["include"], "-o", str(d / "_native.so"),
                    str(d / "native_calls.cpp"), str(d / "library.cpp"), f"-L{t}/lib", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"], check=True)
    return d


def test_transformed_tensors_are_left_to_python(host_build):
    r = subprocess.run([sys.executable, "-c", CALLS, str(host_build)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("all calls returned\n"), (r.returncode, r.stdout[-500:], r.stderr[-2000:])


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2])
def test_transformed_tensors_raise_what_torch_raises(M):
    """The package's own calls: the RuntimeError of data_ptr(), which a caller can catch, and the next call works."""
    import innova_amd as ia
    from innova_amd import layers
    w = ia.DeviceWeights.quantize(torch.randn(8 * 256).numpy(), torch.full((8,), int(ia.Format.OIL4), dtype=torch.uint8).numpy(), 8, 256)
    x, nw = torch.randn(3, M, 256, device="cuda"), torch.randn(256, device="cuda")
    cache = ia.OIL4KVCache(1, 8, 1, 256, 64)
    for f in (w.gemv, w.gemm_f32, lambda t: layers.gemv_rmsnorm(w, t, nw), lambda t: cache.append(0, t.reshape(1, 1, M, 256), t.reshape(1, 1, M, 256))):
        for transformed in (lambda: torch.func.vmap(f)(x), lambda: torch.func.grad(lambda t: (f(t), t.sum())[1])(x[0]), lambda: torch.func.jvp(f, (x[0],), (x[0],))):
            with pytest.raises(RuntimeError, match="data pointer of Tensor that doesn't have storage"):
                transformed()
    assert cache.context_len() == 0
    want = w.gemv(x[0], general=True)
    assert torch.allclose(w.gemv(x[0]), want, rtol=1e-4, atol=1e-4)
