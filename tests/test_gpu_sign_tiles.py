"""Tensors of SPARK_Q0 and OIL1 blocks stored as sign tiles (gemv_signs.hip): the edges of tiles of 16 rows, of the column blocks that a wavefront
holds, of chunks of tiles and parts of K, and activations that the INT8 digits do not hold."""
import numpy as np
import pytest
import torch

import innova_amd as ia
import oracle as O
from gpu_util import gaussian_weights, rel_l2, to_orc_blocks
from innova_amd import layers

pytestmark = pytest.mark.gpu


def tensor(rows, cols, share, seed):
    """rows x cols with that share of SPARK_Q0 blocks, drawn from a pool of 512 blocks of each format."""
    rng = np.random.default_rng(seed)
    pool = [ia.block_codec.quantize_tensor(gaussian_weights(512 * 256, seed + f, outlier_every=13), ia.Format(f)) for f in (0, 1)]
    n = rows * cols // 256
    fm = (rng.random(n) < share).astype(np.uint8)
    pick = rng.integers(0, 512, n)
    desc = np.zeros(n, ia._lib.BLOCK_DTYPE)
    for name in ("cb_off", "idx_off", "cb_bytes", "idx_bytes", "nw", "fmt"):
        desc[name] = np.where(fm == 0, pool[0][1][name][pick], pool[1][1][name][pick])
    spark = fm == 1
    desc["cb_off"][spark] += pool[0][0].size
    desc["idx_off"][spark] += pool[0][0].size
    return ia.DeviceWeights.from_blocks(np.concatenate([pool[0][0], pool[1][0]]), desc, rows, cols)


def reference(dw, x):
    return x.double() @ dw.dequant().view(dw.rows, dw.cols).double().t().contiguous()


# A run's sum is rounded to FP32 once, then meets a scale, its neighbour, up to four blocks, four lane groups and sixteen wavefronts (in four
# sums), and a part of K each: at most 4 + blocks / 16 + 2 + 6 + parts roundings of partial sums that are no larger than the whole's norm.
@pytest.mark.parametrize("share", [0.5, 1.0])
@pytest.mark.parametrize("rows,cols", [(1, 256), (15, 512), (16, 4096), (17, 4352), (33, 8192), (40, 8448), (40, 12288), (2600, 12544), (4111, 16640),
                                       (4096, 768), (66000, 256), (33500, 512), (50000, 4608)])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_sign_tiles(rows, cols, share, M):
    if rows * cols > 50e6 and (share != 0.5 or M in (2, 3)):
        pytest.skip("one mix and two batches of the largest tensors")
    with tensor(rows, cols, share, rows + cols) as dw:
        x = torch.randn(M, cols, generator=torch.Generator().manual_seed(M)).cuda()
        got, want = dw.gemv(x), reference(dw, x)
        assert float((got.double() - want).norm() / want.norm()) <= (12 + cols / 4096 + cols / 16384) * 2.0 ** -24
        assert torch.equal(got, dw.gemv(x))


@pytest.mark.parametrize("M", [1, 2, 4, 7])
def test_captured_without_workspace(M):
    """More rows than a pass, whichever kernel serves them eagerly, and rows past the part of K that a pass covers."""
    with tensor(100, 4608, 0.5, 3) as dw:
        x, y = torch.randn(M, 4608, device="cuda"), torch.empty(M, 100, device="cuda")
        side, g, L = torch.cuda.Stream(), torch.cuda.CUDAGraph(), ia._lib.lib()
        want = reference(dw, x)
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            ia._lib.check(L.oilhip_gemv_f32(dw.handle, x.data_ptr(), y.data_ptr(), M, ia._lib.current_stream()))
        for _ in range(3):
            y.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert rel_l2(y.cpu().numpy(), want.cpu().numpy()) <= 1e-6


def test_outputs_over_the_activations():
    """Several rows in place: a launch of its own packs the activations before any output is stored."""
    with tensor(512, 512, 0.5, 4) as dw:
        x = torch.randn(3, 512, generator=torch.Generator().manual_seed(1)).cuda()
        want = reference(dw, x)
        assert rel_l2(dw.gemv(x, out=x).cpu().numpy(), want.cpu().numpy()) <= 1e-6


def test_two_rows_of_outputs_over_the_activations():
    """More than 8192 rows, which are packed by a launch of their own (fewer never were: outputs may not lie over the activations there)."""
    with tensor(8448, 8448, 0.5, 4) as dw:
        x = torch.randn(2, 8448, generator=torch.Generator().manual_seed(1)).cuda()
        want = reference(dw, x)
        assert rel_l2(dw.gemv(x, out=x).cpu().numpy(), want.cpu().numpy()) <= 1e-6


def test_captured_outputs_over_the_activations():
    """The workspace that a captured call gets is what the activations are packed into; apart from them it stays unused."""
    L = ia._lib.lib()
    with tensor(512, 512, 0.5, 4) as dw:
        assert [L.oilhip_gemv_workspace_bytes(dw.handle, M) > 0 for M in (1, 2, 3, 4, 5)] == [False, False, True, True, True]
        x0 = torch.randn(3, 512, generator=torch.Generator().manual_seed(1)).cuda()
        x, want = x0.clone(), reference(dw, x0)
        dw.gemv(x.clone())
        side, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            dw.gemv(x, out=x)
        for _ in range(3):
            x.copy_(x0)
            g.replay()
            torch.cuda.synchronize()
            assert rel_l2(x.cpu().numpy(), want.cpu().numpy()) <= 1e-6


# outputs over the normalised rows (which are stored for the caller as well), over the norm's weights, over the step's scratch: calls of three and four rows,
# whose activations were always packed before any output was stored
@pytest.mark.parametrize("M", [3, 4])
def test_outputs_over_other_arrays_of_the_call(M):
    D, F, L, S = 1024, 2048, ia._lib.lib(), ia._lib.current_stream
    sq, gu, down = tensor(D, D, 0.5, 1), tensor(2 * F, D, 0.5, 2), tensor(D, F, 0.5, 3)
    x = torch.randn(M, D, generator=torch.Generator().manual_seed(M)).cuda()
    nw = torch.randn(D, generator=torch.Generator().manual_seed(9)).cuda() * 0.2
    xn = x.double() / (x.double().pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * (1.0 + nw.double())
    want = reference(sq, xn).cpu().numpy()
    for _ in range(8):                                     # stores in any order: several tries
        both = torch.empty(M, D, device="cuda")
        ia._lib.check(L.oilhip_gemv_rmsnorm_f32(sq.handle, x.data_ptr(), nw.data_ptr(), both.data_ptr(), M, both.data_ptr(), S()))
        assert rel_l2(both.cpu().numpy(), want) <= 1e-6
        over = torch.empty(M, D, device="cuda")
        over[M - 1] = nw
        spare = torch.empty(M, D, device="cuda")
        ia._lib.check(L.oilhip_gemv_rmsnorm_f32(sq.handle, x.data_ptr(), over[M - 1].data_ptr(), over.data_ptr(), M, spare.data_ptr(), S()))
        assert rel_l2(over.cpu().numpy(), want) <= 1e-6
    gate, up = reference(gu, xn)[:, :F], reference(gu, xn)[:, F:]
    want = reference(down, gate / (1.0 + (-gate).exp()) * up).cpu().numpy()
    for _ in range(8):
        scratch = torch.empty(M * (3 * F + D), device="cuda")
        ia._lib.check(L.oilhip_mlp_step_f32(gu.handle, down.handle, x.data_ptr(), nw.data_ptr(), scratch.data_ptr(), M, scratch.data_ptr(), S()))
        assert rel_l2(scratch[:M * D].cpu().numpy(), want) <= 3e-6
    for w in (sq, gu, down):
        w.close()


# infinities, NaN, a block of zeros, magnitudes whose power of two has no inverse among the floats, and the largest and smallest mantissas of a digit
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_unusual_activations(M):
    rows, cols, inf = 70, 1280, float("inf")
    rng = np.random.default_rng(M)
    with tensor(rows, cols, 0.5, 8) as dw:
        W = dw.dequant().view(rows, cols).cpu().numpy().astype(np.float64)
        for case in range(7):
            x = rng.standard_normal((M, cols)).astype(np.float32)
            m = M - 1
            if case == 0: x[m, 5] = inf
            if case == 1: x[m, [300, 1279]] = [inf, -inf]
            if case == 2: x[m, 700] = float("nan")
            if case == 3: x[:, 256:512] = 0.0
            if case == 4: x[:, 512:768] *= np.float32(1e-36)
            if case == 5: x *= np.float32(1e-41)
            if case == 6: x[m, 256:260] = np.array([0x407F7F7F, 0xC07F7F80, 0x407FFFFF, 0xC0000001], np.uint32).view(np.float32)
            got = dw.gemv(torch.from_numpy(x).cuda()).cpu().numpy()
            with np.errstate(invalid="ignore"):
                want = np.stack([(W * x[i].astype(np.float64)).sum(1) for i in range(M)])
            assert np.array_equal(np.isnan(got), np.isnan(want)), case
            assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0)), case
            ok = np.isfinite(want)
            # (subnormal sums carry 2^-150 per addition)
            assert rel_l2(np.where(ok, got, 0), np.where(ok, want, 0)) <= (1e-6 if case != 5 else 2e-3), case


# A run is held relative to its own largest magnitude: an outlier over a run of scale 0 (SPARK_Q0) or mean 0 (OIL1) must cost the others no bits.  The bound is
# test_sign_tiles'.
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("rows,cols", [(100, 4096), (8300, 1024), (40, 12288)])
@pytest.mark.parametrize("outlier", [1e3, 1e6, 1e10, 1e30])
def test_outliers_over_runs_of_scale_zero(rows, cols, outlier, M):
    if M > 2 and cols > 4096:
        pytest.skip("another kernel's call")
    rng = np.random.default_rng(rows)
    n = rows * cols // 256
    fm = (rng.random(n) < 0.5).astype(np.uint8)
    w = gaussian_weights(rows * cols, 3).reshape(n, 8, 32)
    w[:, 2] = np.where(np.arange(32) % 2, 0.02, -0.02)     # run 2: OIL1 blocks of mean 0 ...
    w[fm == 1, 2] = 0.0                                    # ... SPARK_Q0 blocks of scale 0
    payload, blocks = ia.block_codec.quantize_tensor(w.reshape(-1), fm)
    x = torch.randn(M, cols, generator=torch.Generator().manual_seed(M)).cuda()
    x.view(M, -1, 256)[:, ::2, 69] = outlier
    with ia.DeviceWeights.from_blocks(payload, blocks, rows, cols) as dw:
        got, want = dw.gemv(x), reference(dw, x)
    assert float((got.double() - want).norm() / want.norm()) <= (12 + cols / 4096) * 2.0 ** -24


# runs held as floats beside runs held as digits: the sums of the former may pass the largest float where the products with their scale do not
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_runs_that_are_not_finite_or_tiny(M):
    rows, cols = 70, 1024
    rng = np.random.default_rng(M)
    with tensor(rows, cols, 0.5, 8) as dw:
        W = dw.dequant().view(rows, cols).cpu().numpy().astype(np.float64)
        for case in range(3):
            x = rng.standard_normal((M, cols)).astype(np.float32)
            m = M - 1
            if case == 0: x[m, 64:96], x[m, 80] = 3e37, np.inf               # an infinity behind floats near the largest, in its run
            if case == 1: x[m, 64:96], x[m, 400] = 3e37, -np.inf             # ... in another block
            if case == 2: x[m, 32:64] *= np.float32(1e-30); x[m, 320:352] *= np.float32(1e-40); x[m, 352:384] = 1e37 * np.sign(x[m, 352:384])
            got = dw.gemv(torch.from_numpy(x).cuda()).cpu().numpy()
            with np.errstate(invalid="ignore"):
                want = np.stack([(W * x[i].astype(np.float64)).sum(1) for i in range(M)])
            assert np.array_equal(np.isnan(got), np.isnan(want)), case
            assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0)), case
            for i in range(M):
                ok = np.isfinite(want[i])
                assert rel_l2(got[i][ok].astype(np.float64) * 1e-20, want[i][ok] * 1e-20) <= 1e-6, (case, i)


def test_scales_that_are_not_finite_keep_window_streams():
    """+-inf times activations of both signs is NaN in FP32 sums: signs first would make it an infinity."""
    payload, blocks = ia.block_codec.quantize_tensor(gaussian_weights(64 * 512, 5), ia.Format.SPARK_Q0)
    payload = payload.copy()
    payload[int(blocks["idx_off"][7]):][:2] = [0x00, 0x7C]
    x = torch.randn(1, 512, generator=torch.Generator().manual_seed(1)).cuda()
    with ia.DeviceWeights.from_blocks(payload, blocks, 64, 512) as dw:
        got, plain = dw.gemv(x).cpu().numpy(), dw.gemv(x, general=True).cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(plain)) and np.isnan(got).sum() == 1


# one to four rows behind the norm and SwiGLU; blocks per wavefront 1 to 4, parts of K, activations at odd addresses, and the normalised rows
@pytest.mark.parametrize("M,D,F,shift", [(1, 512, 4352, 1), (1, 4352, 8448, 0), (1, 8448, 12544, 0), (2, 1024, 4352, 3), (3, 512, 4096, 0), (4, 4096, 768, 1), (4, 4352, 512, 0)])
def test_with_norm_and_swiglu(M, D, F, shift):
    rng = np.random.default_rng(D + F + M)
    gu, down = tensor(2 * F, D, 0.5, D), tensor(D, F, 0.5, F)
    x = torch.zeros(shift + M * D, device="cuda")[shift:].view(M, D)
    x.copy_(torch.from_numpy((rng.standard_normal((M, D)) * 2).astype(np.float32)))
    nw = torch.from_numpy((rng.standard_normal(D) * 0.2).astype(np.float32)).cuda()
    xn = x.double() / (x.double().pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * (1.0 + nw.double())
    want = reference(gu, xn)
    got, out, L = layers.gemv_rmsnorm(gu, x, nw), torch.full((M, D), float("nan"), device="cuda"), ia._lib.lib()
    assert rel_l2(got.cpu().numpy(), want.cpu().numpy()) <= 1e-6
    if M > 1:
        again = torch.empty_like(got)
        ia._lib.check(L.oilhip_gemv_rmsnorm_f32(gu.handle, x.data_ptr(), nw.data_ptr(), again.data_ptr(), M, out.data_ptr(), ia._lib.current_stream()))
        assert torch.equal(got, again) and rel_l2(out.cpu().numpy(), xn.cpu().numpy()) <= 3e-7
    g, u = want[:, :F], want[:, F:]
    want = reference(down, g / (1.0 + (-g).exp()) * u)
    assert rel_l2(layers.mlp_step(gu, down, x, norm_w=nw).cpu().numpy(), want.cpu().numpy()) <= 3e-6
    # a sum of squares past the largest float: the norm makes every x zero, an infinite one NaN
    if M > 1:
        x[0] = 3e38
        x[1, 3] = float("inf")
        y = layers.gemv_rmsnorm(gu, x, nw)
        assert bool((y[0] == 0).all()) and bool(y[1].isnan().all()) and bool(torch.isfinite(y[2:]).all())
    gu.close()
    down.close()


# x * r * (1 + w) in that order: a sum of squares past the largest float makes r and so every finite x zero, whatever x times a weight would be; an infinity
# stays NaN, and so does zero times an infinite weight of the norm
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("rows,cols", [(70, 768), (70, 4608), (9000, 512)])
def test_norm_of_the_largest_activations(rows, cols, M):
    with tensor(rows, cols, 0.5, rows + cols) as dw:
        for case in range(4):
            x = torch.randn(M, cols, generator=torch.Generator().manual_seed(M)).cuda()
            nw = torch.zeros(cols, device="cuda")
            x[M - 1] = 3e38 if case != 2 else 1e25
            if case == 1: x[M - 1, cols - 1] = float("inf")
            if case == 3: nw[5] = float("inf")
            y = layers.gemv_rmsnorm(dw, x, nw)
            assert bool((y[M - 1] == 0).all() if case in (0, 2) else y[M - 1].isnan().all()), case
            assert case == 3 or bool(torch.isfinite(y[:M - 1]).all() and (M == 1 or y[:M - 1].abs().max() > 0)), case


# prefill without a launch that decodes: K whole, in 2, 4 and 8 parts (uneven ones among them), and wavefronts of two row blocks; rows and tokens that end
# inside a tile.  Each operand is rounded to bf16 once, the weights here only: 2^-9 at most, a third of it in the mean.
@pytest.mark.parametrize("rows,cols,M", [(5001, 2816, 437), (11008, 4096, 40), (2600, 12544, 100), (4099, 11008, 64), (2600, 11008, 33), (11008, 4096, 2048)])
def test_prefill(rows, cols, M):
    with tensor(rows, cols, 0.5, rows + M) as dw:
        x = torch.randn(M, cols, generator=torch.Generator().manual_seed(M)).cuda()
        got = dw.gemm_f32(x)
        want = reference(dw, x.to(torch.bfloat16))
        assert float((got.double() - want).norm() / want.norm()) <= 2e-3
        assert torch.equal(got, dw.gemm_bf16(x.to(torch.bfloat16))) and torch.equal(got, dw.gemm_f32(x))


# K whole and in parts; activations that start inside 16 bytes (packed by loads that ask for 4 and 2 bytes), tokens with infinities and NaN, outputs over the activations (which
# are packed by a launch of their own)
@pytest.mark.parametrize("rows,cols,M", [(5001, 2816, 437), (11008, 4096, 40), (2600, 12544, 100)])
def test_prefill_of_unusual_activations(rows, cols, M):
    L, S = ia._lib.lib(), ia._lib.current_stream
    with tensor(rows, cols, 0.5, rows + M) as dw:
        x = torch.randn(M, cols, generator=torch.Generator().manual_seed(M)).cuda()
        x[3, 5], x[7, cols - 1], x[M - 1, 300] = float("inf"), float("-inf"), float("nan")
        x[9, [8, 700]] = torch.tensor([float("inf"), float("inf")], device="cuda")
        xb, plain = x.to(torch.bfloat16), dw.gemm_f32(x)
        want = reference(dw, xb)
        assert torch.equal(plain.isnan(), want.isnan()) and int(want.isnan().sum()) >= rows
        assert torch.equal(torch.where(plain.isinf(), plain.sign(), 0.0).double(), torch.where(want.isinf(), want.sign(), 0.0)) and int(want.isinf().sum()) >= 2 * rows
        ok = want.isfinite()
        assert float((plain.double() - want)[ok].norm() / want[ok].norm()) <= 2e-3
        bits = plain.view(torch.int32)
        same = lambda y: torch.equal(torch.where(plain.isnan(), 0, bits), torch.where(y.isnan(), 0, y.view(torch.int32)))
        for shift in (1, 2, 3):
            f = torch.zeros(shift + M * cols, device="cuda")[shift:].view(M, cols)
            f.copy_(x)
            assert same(dw.gemm_f32(f)), shift
        for shift in (1, 3, 7):
            b = torch.zeros(shift + M * cols, device="cuda", dtype=torch.bfloat16)[shift:].view(M, cols)
            b.copy_(xb)
            assert same(dw.gemm_bf16(b)), shift
        both = torch.zeros(M * max(rows, cols), device="cuda")
        both[:M * cols] = x.view(-1)
        ia._lib.check(L.oilhip_gemm_f32(dw.handle, both.data_ptr(), both.data_ptr(), M, S()))
        assert same(both[:M * rows].view(M, rows))
