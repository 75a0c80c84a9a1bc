"""tq_linear (linear layers over many rows) against float64, and the rule that sends calls to it.

Tolerance: the kernel adds, per 16 of K, six exact bf16 products' sums into an fp32 accumulator (each
addition off by at most 2^-24 of the running sum of |x w|) and drops products below 2^-24 |x w|, so an
output is within (6 K / 16 + 4) 2^-24 sum |x w| of the exact value, plus the bias addition's rounding.
GELU's slope is at most 1.13, its own evaluation good to a few 2^-24. That bound holds for every output but is
wide: over all outputs the roundings average out, to 3 x 2^-24 sqrt(K / 32) of the result's 2-norm with a
factor of two to spare (measured 7e-8 at K = 32, 4.2e-7 at 768, 8.7e-7 at 3,072), and that would show a lost limb product
(three products: 4e-6, test_the_norm_bound_tells_six_products_from_three). GELU: twice that."""

from __future__ import annotations

import os
import subprocess
import sys

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from tokquay_amd import _lib, ops

EPS = 2.0**-24


def _check(got, x, w, b, gelu=False, norm=False):
    x, w, got = x.double().cpu(), w.double().cpu(), got.double().cpu()
    ref = x @ w.t()
    bound = (6 * x.size(1) / 16 + 4) * EPS * (x.abs() @ w.abs().t())
    if b is not None:
        ref = ref + b.double().cpu()
        bound = bound + EPS * ref.abs()
    if gelu:
        bound = 1.13 * bound + 16 * EPS * (1 + ref.abs())
        ref = torch.nn.functional.gelu(ref, approximate="tanh")
    bound = bound + x.size(1) * 2.0**-149  # subnormal products
    assert ((got - ref).abs() <= bound).all(), float(((got - ref).abs() - bound).max())
    if norm:
        assert (got - ref).norm() <= (1 + gelu) * _norm_bound(x.size(1)) * ref.norm()


def _norm_bound(k):
    return 3 * EPS * max(1.0, (k / 32) ** 0.5)


def test_the_norm_bound_tells_six_products_from_three():
    """The limb products on the CPU, summed in float64: all six are far inside the norm bound of every K the model
    has, the three largest alone, or six with two limbs paired wrongly, outside."""

    def limbs(t):
        out = []
        for _ in range(3):
            out.append(t.bfloat16().float())
            t = t - out[-1]
        return [v.double() for v in out]

    for k in (32, 768, 3072):
        g = torch.Generator().manual_seed(k)
        x, w = torch.randn(64, k, generator=g), torch.randn(48, k, generator=g) * 0.02
        ref = x.double() @ w.double().t()
        xl, wl = limbs(x), limbs(w)
        error = lambda pairs: float((sum(xl[a] @ wl[b].t() for a, b in pairs) - ref).norm() / ref.norm())  # noqa: E731
        six = [(0, 0), (0, 1), (1, 0), (0, 2), (1, 1), (2, 0)]
        assert error(six) < _norm_bound(k) / 10
        assert error(six[:3]) > 1.5 * _norm_bound(k)
        assert error([(0, 0), (0, 1), (1, 0), (0, 2), (2, 0), (2, 0)]) > 1.2 * _norm_bound(k)


def _inputs(m, n, k, bias=True, seed=0):
    g = torch.Generator().manual_seed(1000 * m + n + k + seed)
    x, w = torch.randn(m, k, generator=g).cuda(), (torch.randn(n, k, generator=g) * 0.02).cuda()
    return x, w, (torch.randn(n, generator=g) * 0.02).cuda() if bias else None


# Rows around the 32-row waves and the 128- and 256-row tiles, columns around the 32-column blocks and
# not a multiple of four, K of one, two, three and many steps; every tile shape is among them.
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 32), (1, 33, 64), (31, 64, 96), (33, 50, 768), (127, 96, 32), (129, 127, 64), (255, 2304, 768),
    (257, 770, 96), (640, 2304, 768), (1000, 2304, 768), (1100, 3072, 64), (1987, 2304, 768), (2048, 3072, 96),
    (2100, 768, 3072), (4097, 1024, 32), (66, 50257, 768),
    # K in parts: 2, 3, 4, 6, 10 and 16 of them, ragged rows and columns
    (70, 100, 256), (129, 516, 384), (640, 768, 3072), (321, 768, 3072), (130, 1600, 1600), (100, 768, 3072),
])  # fmt: skip
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_matches_float64(m, n, k, gelu):
    x, w, b = _inputs(m, n, k, bias=(m + n) % 3 != 0)
    _check(ops._rows_linear(x, w, b, gelu), x, w, b, gelu, norm=m * n >= 1000)  # one output's rounding averages with nothing


@pytest.mark.gpu
def test_strided_rows_and_unaligned_outputs():
    x, w, b = _inputs(300, 129, 96)
    wide = torch.full((300, 132), 7.0, device="cuda")
    wide[:, 4:100] = x
    out = torch.full((300, 135), 5.0, device="cuda")
    torch.ops.tokquay_amd.linear(out[:, 3:132], wide[:, 4:100], w, b, False)
    _check(out[:, 3:132], x, w, b)
    assert (out[:, :3] == 5).all() and (out[:, 132:] == 5).all()


@pytest.mark.gpu
def test_wide_ranges_stay_fp32():
    """Rows from 1e-44 to 1e15 against weights from 1e-5 to 1e18 keep fp32's precision, those included whose limbs
    run out of exponents."""
    x, w, _ = _inputs(160, 96, 256, bias=False)
    x = x * torch.logspace(-44, 15, 160, dtype=torch.double).cuda()[:, None]
    w = w * torch.logspace(-5, 18, 96).cuda()[:, None]
    x = x.float()
    _check(ops._rows_linear(x, w, None, False), x, w, None)
    assert torch.equal(ops._rows_linear(x, torch.eye(256, device="cuda"), None, False), x)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(70, 100, 96), (1000, 2304, 768), (300, 768, 3072)])
def test_tiny_operands(m, n, k):
    """Tiny operands among ordinary ones, alone in their row, behind huge partners, and as weights; rows and
    columns of zeros give zeros."""
    x, w, _ = _inputs(m, n, k, bias=False)
    x[1], x[2], x[33], x[m - 1] = x[1] * 1e-36, x[2] * 1e-41, 0.0, 0.0
    x[3, ::2] *= 1e-38
    x[m - 1, k - 1], x[0, 1] = 3e-39, 2e-36
    w[n - 1], w[5], w[6] = 0.0, w[5] * 1e-37, 0.0
    w[7, k - 1], w[6, 1] = 1e30, 1e33  # one product each: x's tiny elements times these
    got = ops._rows_linear(x, w, None, False)
    _check(got, x, w, None)
    assert (got[33] == 0).all() and (got[:, n - 1] == 0).all()
    others = torch.ones(m, n, dtype=torch.bool, device="cuda")
    others[[1, 2, 3, 33, m - 1, 0]], others[:, [5, 6, 7, n - 1]] = False, False
    clean, weights, _ = _inputs(m, n, k, bias=False)
    assert torch.equal(got[others], ops._rows_linear(clean, weights, None, False)[others])


@pytest.mark.gpu
def test_non_finite_inputs_follow_fp32():
    x, w, b = _inputs(200, 160, 128)
    x[3, 5], x[40, 7], x[77, 0], x[150, 9] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[11, 5], w[12, 9] = 0.0, 1e10
    got = ops._rows_linear(x, w, b, False)
    ref = torch.addmm(b.double(), x.double(), w.double().t()).float()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    fin = ref.isfinite()
    assert torch.equal(got[~fin & ~ref.isnan()], ref[~fin & ~ref.isnan()])
    torch.testing.assert_close(got[fin], ref[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(200, 160, 128), (1000, 2304, 768), (1987, 2304, 96), (640, 768, 3072)])
def test_non_finite_rows_leave_the_others_alone(m, n, k):
    """The rows and columns without an infinity or NaN keep their bits; those with one follow fp32."""
    x, w, b = _inputs(m, n, k)
    clean = ops._rows_linear(x, w, b, True)
    rows, cols = [3, 34, 35, 130, m - 1], [0, 33, n - 1]
    for i, r in enumerate(rows):
        x[r, (7 * i) % k] = [float("inf"), float("nan"), float("-inf"), 3.4e38, float("nan")][i]
    for i, c in enumerate(cols):
        w[c, (11 * i + 5) % k] = [float("nan"), float("inf"), float("-inf")][i]
    got = ops._rows_linear(x, w, b, True)
    keep = torch.ones(m, n, dtype=torch.bool, device="cuda")
    keep[rows], keep[:, cols] = False, False
    assert torch.equal(got[keep], clean[keep])
    ref = torch.nn.functional.gelu(torch.addmm(b.double(), x.double(), w.double().t()).float(), approximate="tanh")
    assert torch.equal(got.isnan(), ref.isnan())
    fin = ref.isfinite()
    torch.testing.assert_close(got[fin], ref[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.gpu
def test_parts_of_k_follow_fp32_and_need_their_workspace():
    x, w, b = _inputs(130, 512, 1024)
    x[5, 700], w[9, 3] = float("inf"), float("nan")
    got = ops._rows_linear(x, w, b, True)
    ref = torch.nn.functional.gelu(torch.addmm(b.double(), x.double(), w.double().t()), approximate="tanh").float()
    assert torch.equal(got.isnan(), ref.isnan())
    fin = ref.isfinite()
    torch.testing.assert_close(got[fin], ref[fin], rtol=1e-4, atol=1e-4)
    L = _lib.lib()
    assert L.tq_linear_workspace_size(130, 512, 1024) == 8 * 130 * 512 * 4
    y = torch.empty(130, 512, device="cuda")
    args = (y.data_ptr(), 512, x.data_ptr(), 1024, 130, w.data_ptr(), b.data_ptr(), 512, 1024, 0)
    assert L.tq_linear(*args, None, 0, 0) == 3
    assert L.tq_linear(*args, y.data_ptr(), 8 * 130 * 512 * 4 - 1, 0) == 3


@pytest.mark.gpu
@pytest.mark.parametrize("gelu", [False, True])
def test_parts_of_k_take_any_bias(gelu):
    """A bias off a 16-byte boundary does not keep K from being split: same bits."""
    x, w, b = _inputs(130, 512, 1024)
    want = ops._rows_linear(x, w, b, gelu)
    for off in (1, 2, 3):
        flat = torch.zeros(520, device="cuda")
        flat[off : off + 512] = b
        assert torch.equal(ops._rows_linear(x, w, flat[off : off + 512], gelu), want)


def test_rule():
    """Few tiles, K not in whole steps: the library; many, or long K to split over the CUs: tq_linear."""
    assert ops.uses_rows_kernel(320, 768, 3072) and not ops.uses_rows_kernel(319, 768, 3072)
    assert not ops.uses_rows_kernel(640, 768, 768) and not ops.uses_rows_kernel(640, 766, 3072)
    assert not ops.uses_rows_kernel(1536, 768, 3072)  # 144 tiles: neither enough nor few enough for two parts
    assert _lib.lib().tq_linear_workspace_size(1536, 768, 3072) == 0
    assert _lib.lib().tq_linear_workspace_size(640, 766, 3072) == 0
    assert _lib.lib().tq_linear_workspace_size(640, 768, 3072) == 4 * 640 * 768 * 4
    assert not ops.uses_rows_kernel(256, 2304, 768) and not ops.uses_rows_kernel(0, 2304, 768)
    assert ops.uses_rows_kernel(640, 2304, 768) and ops.uses_rows_kernel(2048, 768, 3072)
    # K that cannot be split (97, 103 steps of 32), or into too few parts for the CUs: the library.
    for m, n, k in ((320, 768, 3104), (320, 768, 3296), (640, 768, 3136), (320, 1600, 6400), (320, 768, 8192)):
        assert not ops.uses_rows_kernel(m, n, k)
    assert ops.uses_rows_kernel(512, 1600, 6400) and ops.uses_rows_kernel(320, 768, 3136)
    assert ops.uses_rows_kernel(65, 50257, 768) and not ops.uses_rows_kernel(63, 50257, 768)
    assert not ops.uses_rows_kernel(400, 0, 3072)
    assert not ops.uses_rows_kernel(8192, 3072, 776) and not ops.uses_rows_kernel(8192, 3072, 0)


@pytest.mark.gpu
def test_calls_the_kernel_does_not_take_run_as_before(monkeypatch):
    """Gradients, transforms, other types and layouts go the library's way, with its results."""
    lin = torch.nn.Linear(64, 2304).cuda()
    x = torch.randn(1024, 64, device="cuda")
    taken = []
    monkeypatch.setattr(ops, "_rows_linear", lambda *a: taken.append(a) or torch.empty(0))
    y = ops.linear(x, lin)
    assert y.requires_grad and not taken  # grad mode with trainable weights
    with torch.no_grad():
        ref = torch.nn.functional.linear(x, lin.weight, lin.bias)
        for t in (x.t().contiguous().t(), torch.randn(1024, 66, device="cuda")[:, 1:65]):
            out = ops.linear(t, lin)
            torch.testing.assert_close(out, torch.nn.functional.linear(t, lin.weight, lin.bias), rtol=1e-4, atol=1e-4)
        torch.testing.assert_close(torch.vmap(lambda r: ops.linear(r, lin))(x.expand(2, -1, -1))[1], ref, rtol=1e-4,
                                   atol=1e-4)  # fmt: skip
        half = torch.nn.Linear(64, 2304).cuda().half()
        assert ops.linear(x.half(), half).dtype == torch.half
        for dtype in (torch.half, torch.bfloat16):
            with torch.autocast("cuda", dtype=dtype):
                assert ops.linear(x, lin).dtype == ops.lm_head(x, lin.weight).dtype == dtype
        assert not taken
        ops.linear(x, lin)
        assert len(taken) == 1


class _Names(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen = [*getattr(self, "seen", []), getattr(func, "__name__", "")]
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [100, 800])
def test_tracers_and_modes_see_torch_products(rows):
    """A traced or recorded layer holds torch's own product, and runs on other sizes and strides."""
    lin = torch.nn.Linear(3072, 768).cuda().requires_grad_(False)
    x = torch.randn(rows, 3072, device="cuda")
    f = lambda t: ops.linear(t, lin)  # noqa: E731
    assert ops._rows_kernel_takes(x, lin.weight, lin.bias)
    with torch.device("cuda"):
        assert ops._rows_kernel_takes(x, lin.weight, lin.bias)
    others = [x, x[: rows - 1], torch.randn(rows, 6144, device="cuda")[:, ::2], torch.randn(3072, 130, device="cuda").t()]
    same = lambda got, t: torch.testing.assert_close(got, torch.addmm(lin.bias, t, lin.weight.t()), rtol=1e-4, atol=1e-4)  # noqa: E731
    traced = torch.jit.trace(f, (x,), check_trace=False)
    recorded = make_fx(f)(x)
    assert [n.target for n in recorded.graph.nodes if "addmm" in str(n.target)] == [torch.ops.aten.addmm.default]
    compiled = torch.compile(f, backend="eager", fullgraph=True)
    for t in others:
        same(traced(t), t), same(recorded(t), t), same(compiled(t), t)
    torch._dynamo.reset()
    with FlopCounterMode(display=False) as flops:
        f(x)
    assert flops.get_total_flops() == 2 * rows * 3072 * 768
    with _Names() as names:
        f(x)
    assert "addmm" in names.seen


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 7, 16, 17, 100, 128, 129, 320, 321])
def test_few_rows_and_the_head(rows, monkeypatch):
    """Few rows: the wide layers on tq_linear, the same inside a capture as outside one, and on the library where
    a step is chosen by GPU time; the LM head on the library below 64 rows. All within fp32's bound."""
    x, w, b = _inputs(rows, 3072, 768)
    up, down, square = torch.nn.Linear(768, 3072).cuda(), torch.nn.Linear(3072, 768).cuda(), torch.nn.Linear(768, 768).cuda()
    for p in (*up.parameters(), *down.parameters(), *square.parameters()):
        p.requires_grad_(False)
    up.weight.copy_(w), up.bias.copy_(b)
    _check(ops.linear(x, up), x, w, b)
    _check(ops.linear(x, up, gelu=True), x, w, b, gelu=True)
    _check(ops.linear(x, square), x, square.weight, square.bias)
    h = torch.nn.functional.gelu(x @ w.t() + b, approximate="tanh")
    _check(ops.linear(h, down), h, down.weight, down.bias)
    wide = (torch.randn(50257, 768, generator=torch.Generator().manual_seed(rows)) * 0.02).cuda()
    _check(ops.lm_head(x, wide), x, wide, None)
    takes = lambda t, layer: ops._rows_kernel_takes(t, layer.weight, layer.bias)  # noqa: E731
    for capturing in (False, True):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        assert takes(x, up) == (rows <= 320) and takes(h, down) and takes(x, square) == (rows <= 128)
        assert ops._rows_kernel_takes(x, wide, None) == (rows >= 64)
        with ops.by_gpu_time():
            assert not takes(x, up) and takes(h, down) == (rows >= 320) and not takes(x, square)
            assert ops._rows_kernel_takes(x, wide, None) == (rows >= 64)


def test_few_rows_rule():
    """The cheaper call only where the GPU keeps up with it: not for an LM head's weights, nor where long K is left
    in few parts."""
    for m, n, k in ((1, 3072, 768), (128, 768, 768), (320, 768, 3072), (256, 1600, 6400), (128, 768, 3136)):
        assert ops._saves_host_time(m, n, k)
        with ops.by_gpu_time():
            assert not ops._saves_host_time(m, n, k)
        assert ops._saves_host_time(m, n, k)
    for m, n, k in ((0, 3072, 768), (100, 3072, 0), (100, 0, 3072), (8, 32000, 768), (129, 768, 768), (321, 768, 3072), (128, 766, 768), (128, 768, 776),
                    (128, 768, 3104), (320, 768, 3296), (320, 1600, 6400), (320, 768, 8192)):  # fmt: skip
        assert not ops._saves_host_time(m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [0, 1, 100, 400])
@pytest.mark.parametrize("k,n", [(0, 768), (0, 3072), (768, 0), (3072, 0), (768, 3072)])
def test_empty_layers_and_batches(rows, k, n):
    """No rows, no outputs, or an empty sum (the bias): torch's result."""
    layer = torch.nn.Linear(768, 3072).cuda().requires_grad_(False)
    layer.weight, layer.bias = (torch.nn.Parameter(torch.randn(s, device="cuda"), False) for s in ((n, k), (n,)))
    x = torch.randn(rows, k, device="cuda")
    want = torch.addmm(layer.bias, x, layer.weight.t())
    torch.testing.assert_close(ops.linear(x, layer), want, rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(ops.lm_head(x, layer.weight), x @ layer.weight.T, rtol=1e-4, atol=1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [100, 800])
def test_tensors_without_strided_storage(rows):
    """Sparse rows or weights and zero tensors: torch's result."""
    layer = torch.nn.Linear(768, 3072).cuda().requires_grad_(False)
    x = torch.randn(rows, 768, device="cuda")
    want = torch.addmm(layer.bias, x, layer.weight.t())
    for t in (x.to_sparse(), x.to_sparse_csr()):
        torch.testing.assert_close(ops.linear(t, layer), want, rtol=1e-4, atol=1e-4)
    zeros = torch._efficientzerotensor((rows, 768), device="cuda")
    torch.testing.assert_close(ops.linear(zeros, layer), layer.bias.expand(rows, -1))
    layer.weight = torch.nn.Parameter(layer.weight.to_sparse_csr(), False)
    torch.testing.assert_close(ops.linear(x, layer), want, rtol=1e-4, atol=1e-4)


CAPTURE = """
import torch
from tokquay_amd import ops
up, down = torch.nn.Linear(768, 3072).cuda(), torch.nn.Linear(3072, 768).cuda()
x = torch.randn({rows}, 768, device="cuda")
f = lambda: ops.linear(ops.linear(x, up, gelu=True), down)
with torch.no_grad():
    f()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = f()
    for _ in range(3):
        x.normal_()
        graph.replay()
        assert torch.equal(y, f())
        torch.cuda.synchronize()
print("captured")
"""


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [64, 100, 256, 400])
def test_one_eager_run_prepares_a_capture(rows):
    """In a process that has run nothing else, the MLP's layers are captured after one eager run, and every
    replay gives the eager call's bits."""
    run = subprocess.run([sys.executable, "-c", CAPTURE.format(rows=rows)], capture_output=True, text=True, timeout=100,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))  # fmt: skip
    assert run.returncode == 0 and "captured" in run.stdout, run.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_runs_on_its_tensors_device():
    """With another device current, the launch goes to the tensors' device and its stream."""
    x, w, b = _inputs(640, 2304, 768)
    want = ops._rows_linear(x, w, b, False)
    x, w, b = (t.to("cuda:1") for t in (x, w, b))
    with torch.cuda.device(0):
        x.mul_(2.0).mul_(0.5)  # queued on cuda:1's stream in front of the product
        assert torch.equal(ops._rows_linear(x, w, b, False).cpu(), want.cpu())
        assert torch.cuda.current_device() == 0
