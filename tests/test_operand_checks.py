"""What the wrappers hand to the kernels by address, checked without a GPU: the
native call is replaced by one that reads its arguments on the host."""

import ctypes

import pytest
import torch

from evo2_flash_amd import _lib

bf = torch.bfloat16


@pytest.fixture
def native(monkeypatch):
    """CPU tensors pass the device check; calls are recorded, not made.  A
    recorded call is (name, arguments, what `native.look` returned inside it)."""
    class Native(list):
        look = staticmethod(lambda name, args: None)

    calls = Native()
    monkeypatch.setattr(_lib, "require_device", lambda *t: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t=None: None)
    monkeypatch.setattr(_lib, "call", lambda name, *a: calls.append((name, a, calls.look(name, a))))
    return calls


def _floats(address, n):
    return torch.tensor((ctypes.c_float * n).from_address(address))


def _rotary_case(hd=128, nh=2, rows=4):
    from evo2_flash_amd.attention import PagedKVCache
    cache = PagedKVCache(5, nh, hd, "cpu")
    qkv = torch.randn(rows, 3 * nh * hd).to(bf)
    table = torch.arange(1, 5, dtype=torch.int32).view(4, 1)
    inv_freq = 1.0 / 10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd)
    return qkv, cache, table, inv_freq


def _rotate(which, qkv, cache, table, inv_freq):
    from evo2_flash_amd.attention import rotary_decode, rotary_prefill
    if which == "prefill":
        return rotary_prefill(qkv, cache, table, inv_freq, 1.0, 1, qkv.shape[0])
    return rotary_decode(qkv, cache, table, torch.zeros(qkv.shape[0], dtype=torch.int64), inv_freq,
                         1.0)


@pytest.mark.parametrize("which", ["prefill", "decode"])
@pytest.mark.parametrize("form", ["bf16", "fp64", "strided"])
def test_rotary_frequencies_reach_the_kernel_as_fp32(which, form, native):
    """inv_freq of another type (a module cast with .to(torch.bfloat16)) or
    stride: the kernel reads head_dim / 2 contiguous fp32 of the same values."""
    qkv, cache, table, inv_freq = _rotary_case()
    f = {"bf16": inv_freq.to(bf), "fp64": inv_freq.double(),
         "strided": inv_freq.repeat_interleave(2)[::2]}[form]
    native.look = lambda name, a: _floats(a[2], 64)
    _rotate(which, qkv, cache, table, f)
    assert [c[0] for c in native] == ["evo2_rotary_" + which]
    assert torch.equal(native[0][2], f.float())


@pytest.mark.parametrize("which", ["prefill", "decode"])
@pytest.mark.parametrize("what", ["inv_freq", "qkv_dtype", "qkv_columns", "k_dtype", "v_dtype",
                                  "k_page", "v_pages", "v_strides"])
def test_rotary_refuses_what_the_kernel_cannot_address(which, what, native):
    qkv, cache, table, inv_freq = _rotary_case()
    if what == "inv_freq":
        inv_freq = inv_freq[:63]
    elif what == "qkv_dtype":
        qkv = qkv.float()
    elif what == "qkv_columns":
        qkv = qkv[:, :-8]
    elif what == "k_dtype":
        cache.k = cache.k.float()
    elif what == "v_dtype":
        cache.v = cache.v.to(torch.float16)
    elif what == "k_page":
        cache.k = cache.k[..., :8]
    elif what == "v_pages":
        cache.v = cache.v[:4]
    else:
        cache.v = cache.v.transpose(2, 3).contiguous().transpose(2, 3)
    with pytest.raises(ValueError):
        _rotate(which, qkv, cache, table, inv_freq)
    assert not native


def _rows_case(L=5, Lv=8, N=2, nh=3):
    z = lambda *s: torch.zeros(*s, dtype=bf)
    return z(N, nh, L, 128), z(N, nh, L, 128), z(N, nh, 128, Lv), z(N, nh, L, 128)


def test_prefill_attention_rows_takes_padded_values_and_any_rows(native):
    from evo2_flash_amd.attention import prefill_attention_rows
    q, k, vt, _ = _rows_case()
    out = torch.zeros(2, 5, 3, 128, dtype=bf).transpose(1, 2)
    prefill_attention_rows(q, k, vt, 1.0, out)
    assert [c[0] for c in native] == ["evo2_prefill_attention_rows"]


@pytest.mark.parametrize("what", ["dtype", "dims", "k_length", "k_heads", "out_length", "out_rows",
                                  "vt_planes", "vt_short", "vt_multiple", "q_strides",
                                  "vt_strides"])
def test_prefill_attention_rows_refuses_what_the_kernel_cannot_address(what, native):
    from evo2_flash_amd.attention import prefill_attention_rows
    q, k, vt, out = _rows_case()
    if what == "dtype":
        q = q.to(torch.float16)
    elif what == "dims":
        q = q[0]
    elif what == "k_length":
        k = k[:, :, :4].contiguous()
    elif what == "k_heads":
        k = k[:, :2].contiguous()
    elif what == "out_length":
        out = out[:, :, :4]
    elif what == "out_rows":
        out = torch.zeros(2, 3, 128, 5, dtype=bf).transpose(2, 3)
    elif what == "vt_planes":
        vt = vt[:1]
    elif what == "vt_short":
        q, k, _, out = _rows_case(L=9)
    elif what == "vt_multiple":
        vt = _rows_case(Lv=12)[2]
    elif what == "q_strides":
        q = torch.zeros(2, 5, 3, 128, dtype=bf).transpose(1, 2)
    else:
        vt = torch.zeros(2, 3, 8, 128, dtype=bf).transpose(2, 3)
    with pytest.raises(ValueError):
        prefill_attention_rows(q, k, vt, 1.0, out)
    assert not native


def _verify_case(columns, H=8, Q=3, n=2):
    state = torch.zeros(7, H, columns)
    t = torch.ones(n, Q, dtype=torch.int32)
    rows = torch.arange(n) * Q
    meta = (t, t + 1, rows, rows + Q, torch.ones(n, dtype=torch.int64))
    return torch.zeros(n * Q, 3 * H, dtype=bf), state, torch.zeros(H, dtype=bf), meta


@pytest.mark.parametrize("K", [7, 128])
@pytest.mark.parametrize("what", [None, "taps", "taps_dtype", "taps_rows", "columns", "state_dtype",
                                  "D"])
def test_gated_fir_operands(K, what, native):
    from evo2_flash_amd.verify import fir_verify_gated
    zf, state, D, meta = _verify_case(K - 1)
    w = torch.zeros(8, K, dtype=bf)
    if what == "taps":
        w = torch.zeros(8, 16, dtype=bf)
    elif what == "taps_dtype":
        w = w.float()
    elif what == "taps_rows":
        w = w[:7]
    elif what == "columns":
        state = state[..., :K - 2]
    elif what == "state_dtype":
        state = state.to(bf)
    elif what == "D":
        D = D[:7]
    if what is None:
        fir_verify_gated(zf, w, D, state, meta)
        fir_verify_gated(zf, w, None, state, meta)
        assert [c[0] for c in native] == ["evo2_fir_verify_gated"] * 2
    else:
        with pytest.raises(ValueError):
            fir_verify_gated(zf, w, D, state, meta)
        assert not native


@pytest.mark.parametrize("what", [None, "poles", "poles_dtype", "residues_dtype", "columns", "D"])
def test_gated_iir_operands(what, native):
    from evo2_flash_amd.verify import iir_verify_gated
    zf, state, D, meta = _verify_case(17)
    lp, res = torch.randn(8, 16), torch.zeros(8, 16)
    if what == "poles":
        lp = lp[:, :15]
    elif what == "poles_dtype":
        lp = lp.to(bf)
    elif what == "residues_dtype":
        res = res.double()
    elif what == "columns":
        state = state[..., :15]
    elif what == "D":
        D = D.repeat(2)
    if what is not None:
        with pytest.raises(ValueError):
            iir_verify_gated(zf, lp, res, D, state, meta)
        assert not native
        return
    # poles off 16-byte alignment or row-strided arrive as rows of float4
    wide = torch.zeros(8, 33)
    wide[:, 1::2] = lp
    native.look = lambda name, a: (a[2] % 16, a[3:5], _floats(a[2], 128).view(8, 16))
    for poles in (lp, wide[:, 1::2]):
        iir_verify_gated(zf, poles, res, D, state, meta)
    for name, _, (align, strides, seen) in native:
        assert name == "evo2_iir_verify_gated" and align == 0 and strides == (16, 1)
        assert torch.equal(seen, lp)


def test_one_row_fp8_linear_in_place_quantises_apart(native):
    """static_fp8_linear(x, out=x): x is read whole before any of it is
    overwritten, so the one-launch form is for outputs beside x only."""
    from evo2_flash_amd.fp8 import E4M3, static_fp8_linear
    K = 256
    buf = torch.zeros(4 * K, dtype=bf)
    x, one = buf[K:2 * K].view(1, K), torch.ones(1)
    w = torch.zeros(K, K).to(E4M3)
    apart, joint = ["evo2_fp8_quantize", "evo2_fp8_gemm"], ["evo2_fp8_quant_gemv"]
    for out, want in ((x, apart), (buf[K // 2:K // 2 + K].view(1, K), apart),
                      (buf[2 * K - 1:3 * K - 1].view(1, K), apart), (buf[:K].view(1, K), joint),
                      (buf[2 * K:3 * K].view(1, K), joint), (None, joint)):
        static_fp8_linear(x, w, one, one, out=out)
        assert [c[0] for c in native] == want
        native.clear()


@pytest.mark.parametrize("rows,N,reads", [(1, 64, True), (64, 60016, True), (256, 12288, True),
                                          (65, 25008, False), (320, 12000, False)])
def test_packed_copy_is_asked_for_where_it_is_read(rows, N, reads, native, monkeypatch):
    from evo2_flash_amd.fp8 import E4M3, Fp8StaticLinear
    lin = Fp8StaticLinear(128, N, bias=False)
    copy = torch.zeros(N, 128).to(E4M3)
    asked = []
    monkeypatch.setattr(lin, "decode_weight", lambda: (asked.append(1), copy)[1])
    lin(torch.zeros(rows, 128, dtype=bf))
    assert bool(asked) == reads
    assert (_lib.ptr(copy) in native[-1][1]) == reads


@pytest.mark.parametrize("M", [4, 33])
@pytest.mark.parametrize("bias", [False, True])
def test_linear_adds_a_residual_that_is_its_output(M, bias):
    """out = residual: product plus residual, not twice the product."""
    from evo2_flash_amd.linear import linear
    x, w, r = torch.randn(M, 64), torch.randn(32, 64), torch.randn(M, 32)
    b = torch.randn(32) if bias else None
    want = torch.nn.functional.linear(x, w, b) + r
    assert linear(x, w, b, out=r, residual=r).data_ptr() == r.data_ptr()
    assert torch.equal(r, want)


def test_overlap():
    t = torch.zeros(6, 8, dtype=bf)
    assert _lib.overlap(t, t[5:]) and _lib.overlap(t[:, :4], t[:, 4:])    # the ranges, not the elements
    assert not _lib.overlap(t[:3], t[3:]) and not _lib.overlap(t, t[:0])
    assert _lib.overlap(t[0], t.view(-1)[7:9]) and not _lib.overlap(t[0], t.view(-1)[8:9])


def _layer(H=8, inter=12):
    """A decoder layer whose norms and mixer are stand-ins that run on the CPU."""
    from evo2_flash_amd.config import HyenaConfig
    from evo2_flash_amd.model import Evo2DecoderLayer
    cfg = HyenaConfig(hidden_size=H, intermediate_size=inter, num_hidden_layers=1,
                      hcs_layer_idxs=[0])
    layer = Evo2DecoderLayer(cfg, 0, lambda x, token_ids: x)
    layer.pre_norm = torch.nn.Identity()
    layer.post_norm = type("Norm", (torch.nn.Module,), {"forward": lambda self, m, x: (m, x)})()
    for p in layer.mlp.parameters():
        p.data.copy_(torch.randn(p.shape))
    return layer


def _mlp_ref(mlp, x, gelu=True):
    F = torch.nn.functional
    z1 = F.linear(x, mlp.l1.weight)
    return F.linear((F.gelu(z1) if gelu else z1) * F.linear(x, mlp.l2.weight), mlp.l3.weight)


def test_mlp_hooks_see_the_module_outputs():
    """Hooks on l1, l2, l3 and the MLP run and see each module's own output, the
    layer's input not in it; the layer's result does not change."""
    layer = _layer()
    x = torch.randn(3, 8).to(bf)
    plain = layer(None, x, None, None)
    seen = {}
    for name in ("l1", "l2", "l3"):
        getattr(layer.mlp, name).register_forward_hook(
            lambda m, a, out, name=name: seen.__setitem__(name, out[0]))
    layer.mlp.register_forward_hook(lambda m, a, out: seen.__setitem__("mlp", out))
    assert torch.equal(layer(None, x, None, None), plain)
    mlp, F = layer.mlp, torch.nn.functional
    ref = _mlp_ref(mlp, x)
    assert torch.equal(seen["l1"], F.linear(x, mlp.l1.weight))
    assert torch.equal(seen["l2"], F.linear(x, mlp.l2.weight))
    assert torch.equal(seen["l3"], ref) and torch.equal(seen["mlp"], ref)
    assert torch.equal(plain, ref + x)


@pytest.mark.parametrize("what", ["module_bias", "replaced", "instance_forward", "global_hook",
                                  "mlp"])
def test_mlp_calls_what_stands_in_its_place(what):
    from evo2_flash_amd.mixers import Linear
    layer = _layer()
    mlp = layer.mlp
    x = torch.randn(3, 8).to(bf)
    ref = _mlp_ref(mlp, x)
    called = []
    if what == "module_bias":
        w = mlp.l2.weight
        mlp.l2 = Linear(8, 12, bias=True)
        mlp.l2.weight.data.copy_(w)
        mlp.l2.bias.data.fill_(2.0)
        F = torch.nn.functional
        z1 = F.gelu(F.linear(x, mlp.l1.weight))
        ref = F.linear(z1 * F.linear(x, w, mlp.l2.bias), mlp.l3.weight)
    elif what == "replaced":
        class Twice(torch.nn.Module):
            def forward(self, t):
                called.append("l")
                return torch.nn.functional.linear(t, self.inner.weight), None
        twice = Twice()
        twice.inner, mlp.l1 = mlp.l1, twice
        plain, mlp.l3 = mlp.l3, Twice()
        mlp.l3.inner = plain
    elif what == "instance_forward":
        inner = mlp.l2.forward
        mlp.l2.forward = lambda t: (called.append("l2"), inner(t))[1]
    elif what == "global_hook":
        handle = torch.nn.modules.module.register_module_forward_hook(
            lambda m, a, out: called.append(type(m).__name__))
    else:
        class Own(torch.nn.Module):
            def forward(self, t):
                return -t
        layer.mlp, ref = Own(), -x
    try:
        got = layer(None, x, None, None)
    finally:
        if what == "global_hook":
            handle.remove()
    assert torch.equal(got, ref + x)
    assert {"replaced": called == ["l", "l"], "instance_forward": called == ["l2"],
            "global_hook": called.count("Linear") == 3}.get(what, not called)


@pytest.mark.parametrize("which", ["prefill", "decode"])
@pytest.mark.parametrize("form", ["int64", "int16", "uint8", "columns", "transposed"])
def test_rotary_block_tables_of_any_integer_type_and_stride(which, form, native):
    """The kernel reads int32 entries at unit column stride; an int64 entry past
    32 bits does not wrap onto a page."""
    qkv, cache, _, inv_freq = _rotary_case()
    want = torch.tensor([[3, 1], [2, 4], [4, 2], [1, 3]])
    table = {"int64": want.clone(), "int16": want.short(), "uint8": want.byte(),
             "columns": want.int().repeat_interleave(2, 1)[:, ::2],
             "transposed": want.int().t().contiguous().t()}[form]
    if form == "int64":
        table[0, 1], table[1, 1], table[2, 1] = (1 << 32) + 1, -3, 5
        want[0, 1] = want[1, 1] = want[2, 1] = -1                # five pages: 0 .. 4
    n = 1 if which == "prefill" else 4

    def look(name, a):
        i = 17 if which == "prefill" else 14                     # table, row stride, columns
        assert a[i + 2] == 2
        flat = (ctypes.c_int32 * (a[i + 1] * (n - 1) + 2)).from_address(a[i])
        return [[flat[a[i + 1] * r + c] for c in (0, 1)] for r in range(n)]

    native.look = look
    _rotate(which, qkv, cache, table, inv_freq)
    assert native[0][2] == want[:n].tolist()


@pytest.mark.parametrize("which", ["prefill", "decode"])
def test_rotary_takes_rows_of_any_stride(which, native):
    qkv, cache, table, inv_freq = _rotary_case()
    wide = torch.zeros(qkv.shape[0], 2 * qkv.shape[1], dtype=bf)
    wide[:, ::2] = qkv

    def look(name, a):
        flat = (ctypes.c_int16 * qkv.numel()).from_address(a[0])
        return torch.tensor(flat, dtype=torch.int16).view(bf).view(qkv.shape), a[1]

    native.look = look
    _rotate(which, wide[:, ::2], cache, table, inv_freq)
    seen, stride = native[0][2]
    assert torch.equal(seen, qkv) and stride == qkv.shape[1]
    with pytest.raises(ValueError):
        _rotate(which, qkv, cache, table[:0], inv_freq)


def _mlp_or_linear(what):
    from evo2_flash_amd.mixers import Linear
    return Linear(8, 12) if what == "linear" else _layer().mlp


@pytest.mark.parametrize("what", ["linear", "mlp"])
def test_projections_trace_symbolically(what):
    """torch.fx and torch.export with any number of rows: no condition on the rows
    in front of the library's product, no argument beyond the module's own, and
    l1 .. l3 can be a tracer's leaves."""
    from torch import fx
    from evo2_flash_amd.mixers import Linear
    mod = _mlp_or_linear(what)
    with torch.no_grad():
        for p in mod.parameters():
            p.copy_(torch.randn(p.shape))
    x, y = torch.randn(3, 8).to(bf), torch.randn(40, 8).to(bf)
    want = mod(y)
    args = {"out": None} if what == "linear" else None
    traced = fx.symbolic_trace(mod, concrete_args=args)
    rows = torch.export.Dim("rows", min=2, max=4096)
    program = torch.export.export(mod, (x,), dynamic_shapes={"x": {0: rows}}).module()
    for form in (traced, program):
        got = form(y)
        assert torch.equal(*((got[0], want[0]) if what == "linear" else (got, want)))
    if what == "mlp":
        class Leaves(fx.Tracer):
            def is_leaf_module(self, m, name):
                return isinstance(m, Linear)
        nodes = Leaves().trace(mod).nodes
        assert [n.target for n in nodes if n.op == "call_module"] == ["l1", "l2", "l3"]


def test_linear_of_a_sparse_weight():
    """Sparse weights reach torch's own product."""
    from evo2_flash_amd.mixers import Linear
    mod = Linear(32, 12, dtype=torch.float32)
    w, x = torch.randn(12, 32), torch.randn(3, 32)
    for sparse in (w.to_sparse_csr(), w.to_sparse()):
        mod.weight = torch.nn.Parameter(sparse, requires_grad=False)
        torch.testing.assert_close(mod(x)[0], x @ w.t())


@pytest.mark.parametrize("bias", [False, True])
def test_linear_compiles_to_torchscript(bias):
    from evo2_flash_amd.mixers import Linear
    mod = Linear(8, 12, bias=bias)
    with torch.no_grad():
        for p in mod.parameters():
            p.copy_(torch.randn(p.shape))
    x, out = torch.randn(3, 8).to(bf), torch.empty(3, 12, dtype=bf)
    script = torch.jit.script(mod)
    assert script(x, out)[0].data_ptr() == out.data_ptr()
    assert torch.equal(out, mod(x)[0]) and torch.equal(script(x)[0], out)


def test_rows_that_stream_by_width():
    """The widths of the 1B, 7B and 40B models, and those between."""
    from evo2_flash_amd.linear import gated_rows, stream_rows
    for N, K, rows, added in ((1920, 1920, 16, 16), (5760, 1920, 16, 16), (1920, 5120, 8, 8),
                              (4096, 4096, 16, 16), (12288, 4096, 8, 8), (4096, 11264, 4, 8),
                              (8192, 8192, 4, 8), (24576, 8192, 4, 4), (512, 8192, 0, 0),
                              (8192, 22528, 0, 0), (6144, 6144, 0, 0)):
        assert stream_rows(N, K) == rows and stream_rows(N, K, residual=True) == added
    assert [gated_rows(K) for K in (1920, 4096, 5120, 8192, 11264, 16384)] == [16, 16, 16, 8, 8, 0]
