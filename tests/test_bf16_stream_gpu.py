"""The weight-streaming bf16 projections of decode steps (csrc/bf16_stream.hip,
linear.py) against 64-bit products: plain with bias and residual, and gated, at
the edges of the kernel's tiles (1 to 16 rows, 16 weight rows a workgroup, eight
parts of K in steps of 32), rows of wider matrices, and the calls that stay on
the library (more rows, gradients, autocast).  Bound: one bf16 rounding per
rounded step (2^-9 of its value) and fp32 sums of at most 11264 terms in any
order (2^-16 of the sum of magnitudes)."""

import pytest
import torch

from evo2_flash_amd import _lib
from evo2_flash_amd.linear import gated, linear

pytestmark = pytest.mark.gpu
DEV = "cuda"
bf = torch.bfloat16


def _rand(*shape, seed, scale=1.0, pad=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rows, cols = shape
    return (torch.randn(rows, cols + pad, generator=g, device=DEV) * scale).to(bf)[:, :cols]


@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (7, 37, 224), (8, 4096, 4096), (16, 513, 1920),
                                   (3, 40, 288), (4, 4096, 11264)])
def test_linear_vs_fp64(M, N, K, monkeypatch):
    x, w = _rand(M, K, seed=1, pad=8), _rand(N, K, seed=2, scale=0.05, pad=8)
    b, r = _rand(1, N, seed=3)[0].contiguous(), _rand(M, N, seed=4, pad=(-N) % 8 + 8)
    calls = []
    call = _lib.call
    monkeypatch.setattr(_lib, "call", lambda n, *a: (calls.append(n), call(n, *a)))
    print(f"bf16 stream M={M} N={N} K={K}", flush=True)
    ref = x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t() * 2.0 ** -16
    got = linear(x, w).double()
    assert ((got - ref).abs() <= ref.abs() * 2.0 ** -8 + mag).all()
    out = torch.full((M + 1, N), 7.0, dtype=bf, device=DEV)
    assert linear(x, w, b, out=out[:M]).data_ptr() == out.data_ptr()
    ref = ref + b.double()
    assert ((out[:M].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag).all()
    assert (out[M] == 7).all()
    got = linear(x, w, b, residual=r).double()
    sum_ = ref + r.double()
    assert ((got - sum_).abs() <= (ref.abs() + sum_.abs()) * 2.0 ** -8 + mag).all()
    assert calls == ["evo2_bf16_stream_linear"] * 3


@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (16, 50, 1920), (8, 11264, 4096)])
@pytest.mark.parametrize("gelu", [False, True])
def test_gated_vs_fp64(M, N, K, gelu, monkeypatch):
    x = _rand(M, K, seed=5)
    w1, w2 = _rand(N, K, seed=6, scale=0.05), _rand(N, K, seed=7, scale=0.05)
    calls = []
    call = _lib.call
    monkeypatch.setattr(_lib, "call", lambda n, *a: (calls.append(n), call(n, *a)))
    print(f"bf16 stream gated M={M} N={N} K={K} gelu={gelu}", flush=True)
    got = gated(x, w1, w2, gelu).double()
    z1, z2 = x.double() @ w1.double().t(), x.double() @ w2.double().t()
    m1, m2 = ((x.double().abs() @ w.double().abs().t()) * 2.0 ** -16 + z.abs() * 2.0 ** -8
              for w, z in ((w1, z1), (w2, z2)))
    a = torch.nn.functional.gelu(z1) if gelu else z1
    m1 = 1.13 * m1 + a.abs() * 2.0 ** -8               # |gelu'| <= 1.13, and its rounding
    bound = m1 * (z2.abs() + m2) + a.abs() * m2 + (a * z2).abs() * 2.0 ** -8
    assert ((got - a * z2).abs() <= bound).all()
    assert calls == ["evo2_bf16_stream_gated"]


def test_calls_that_stay_on_the_library(monkeypatch):
    """More than 16 rows, a differentiated input, autocast, vmap and odd rows."""
    w = _rand(64, 64, seed=8)
    calls = []
    monkeypatch.setattr(_lib, "call", lambda n, *a: calls.append(n))
    F = torch.nn.functional.linear
    x = _rand(17, 64, seed=9)
    assert torch.equal(linear(x, w), F(x, w))
    x = _rand(4, 64, seed=10).requires_grad_()
    linear(x, w).float().sum().backward()
    assert x.grad is not None
    x = x.detach()
    with torch.autocast("cuda", dtype=torch.float16):
        assert linear(x, w).dtype == torch.float16
    xs = x.view(2, 2, 64)
    assert torch.equal(torch.vmap(lambda t: linear(t, w))(xs), F(xs, w))
    odd = _rand(4, 64, seed=11, pad=3)
    assert torch.equal(linear(odd, w), F(odd, w))
    assert linear(x.float(), w.float()).dtype == torch.float32
    assert calls == []


def test_operands_off_the_current_device_stay_on_the_library(monkeypatch):
    """x on a device that is not the current one (here by the current device's
    number): no launch of the package's own."""
    x, w = _rand(4, 64, seed=12), _rand(64, 64, seed=13)
    calls = []
    monkeypatch.setattr(_lib, "call", lambda n, *a: calls.append(n))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert torch.equal(linear(x, w), torch.nn.functional.linear(x, w))
    z = torch.nn.functional.linear(x, w)
    assert torch.equal(gated(x, w, w, False), z * z)
    assert calls == []
    monkeypatch.undo()
    with pytest.raises(RuntimeError):                  # the library's own refusal
        linear(x, w, bias=torch.zeros(64, dtype=bf))
    with pytest.raises(RuntimeError):
        linear(x, w, residual=torch.zeros(4, 64, dtype=bf))


def test_traced_calls_stay_in_the_graph():
    """torch.jit.trace and make_fx see a product, not a constant: the traced
    call follows new inputs."""
    from torch.fx.experimental.proxy_tensor import make_fx
    w, w2 = _rand(64, 64, seed=14), _rand(64, 64, seed=15)
    x, y = _rand(4, 64, seed=16), _rand(4, 64, seed=17)
    F = torch.nn.functional.linear
    for fn, want in ((lambda t: linear(t, w), F(y, w)),
                     (lambda t: gated(t, w, w2, False), F(y, w) * F(y, w2))):
        assert torch.equal(torch.jit.trace(fn, x, check_trace=False)(y), want)
        assert torch.equal(make_fx(fn)(x)(y), want)


def test_outputs_over_inputs(monkeypatch):
    """out over the residual: the library's product, which refuses a part of it;
    beside it: the kernel."""
    x, w, r = _rand(8, 64, seed=18), _rand(64, 64, seed=19), _rand(9, 64, seed=20)
    calls = []
    call = _lib.call
    monkeypatch.setattr(_lib, "call", lambda n, *a: (calls.append(n), call(n, *a)))
    want = torch.nn.functional.linear(x, w) + r[:8]
    buf = r.clone()
    assert torch.equal(linear(x, w, residual=buf[:8], out=buf[:8]), want)
    with pytest.raises(RuntimeError):
        linear(x, w, residual=buf[:8], out=buf[1:])
    assert calls == []
    linear(x, w, residual=r[:8], out=torch.empty_like(want))
    assert calls == ["evo2_bf16_stream_linear"]


def test_function_modes_see_the_product():
    """A function mode is called for the library's product; a default device,
    which is one too, leaves the kernel in place."""
    x, w = _rand(4, 64, seed=21), _rand(64, 64, seed=22)
    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    with Mode():
        y = linear(x, w)
        gated(x, w, w, False)
    assert seen.count("linear") == 3
    assert torch.equal(y, torch.nn.functional.linear(x, w))
    with torch.device(DEV), pytest.MonkeyPatch.context() as mp:
        calls, call = [], _lib.call
        mp.setattr(_lib, "call", lambda n, *a: (calls.append(n), call(n, *a)))
        linear(x, w)
        assert calls == ["evo2_bf16_stream_linear"]


def test_vmapped_bias():
    """A batch of biases or residuals over a plain product: torch's own."""
    x, w, b = _rand(4, 64, seed=23), _rand(64, 64, seed=24), _rand(3, 64, seed=25)
    F = torch.nn.functional.linear
    # (vmap's own form of F.linear rounds the product before it adds the bias)
    want = torch.vmap(lambda t: F(x, w, t))(b)
    assert torch.equal(torch.vmap(lambda t: linear(x, w, t))(b), want)
    r = torch.stack([_rand(4, 64, seed=s) for s in (26, 27)])
    got = torch.vmap(lambda t: linear(x, w, residual=t))(r)
    assert torch.equal(got, F(x, w) + r)


@pytest.mark.parametrize("M,N,K,streams", [(8, 64, 5120, True), (9, 64, 5120, False),
                                           (16, 64, 4096, True), (4, 4096, 8192, True),
                                           (5, 4096, 8192, False), (2, 512, 8192, False),
                                           (4, 64, 6144, False), (2, 64, 22528, False)])
def test_rows_that_stream(M, N, K, streams, monkeypatch):
    """Weights on which the library is the faster one stay there, at every width
    of the kernel's; both within the rounding of 64-bit products."""
    x, w = _rand(M, K, seed=28), _rand(N, K, seed=29, scale=K ** -0.5)
    calls, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda n, *a: (calls.append(n), call(n, *a)))
    got = linear(x, w)
    assert bool(calls) == streams
    ref = x.double() @ w.double().t()
    # bf16 of an fp32 sum of K products
    bound = ref.abs() * 2 ** -8 + K * 2 ** -23 * (x.double().abs() @ w.double().abs().t())
    assert ((got.double() - ref).abs() <= bound).all()
    calls.clear()
    gated(x, w, w, False)
    assert bool(calls) == (K <= 5120 or (M <= 8 and K <= 11264))
    r = _rand(M, N, seed=30)
    calls.clear()
    got = linear(x, w, residual=r)
    assert bool(calls) == (streams or (M, K) == (5, 8192))
    total = ref + r.double()                              # (rounded twice)
    assert ((got.double() - total).abs() <= bound + total.abs() * 2 ** -8).all()
