"""Decode attention of the whole-model harness (attention.py, csrc/attention.hip)
against plain fp32 attention on the CPU: out = softmax(scale q.k) v over cache
positions 0..positions[b].  Bar: max |out - ref| / max |ref| <= 1e-2 per case
(the kernel's output is bf16, ~4e-3 relative rounding).  Cases: head_dim 64 and
128; contexts of one and several 2048-position chunks; lengths ending inside a
chunk, at a chunk edge and at the cache end; a batch slice of a larger cache
(the harness's k_cache[:B]); the 7B attention shape (32 heads of 128) at the
benchmark's context; a prompt's pages shared by every sequence, with and
without the sharing declared (head_dim 64: bitwise the same; 128, the
matrix-core kernel: within a bf16 rounding step of the undeclared result,
nearly all elements the same bits), for one partial and two groups of 32
sequences.  Causal prefill attention (head_dim 128, the matrix-core kernel)
against fp32 attention on the CPU at several prompt lengths, and with
peaked scores.
"""

import pytest
import torch

from evo2_flash_amd.attention import (PAGE, PagedKVCache, decode_attention,
                                     paged_decode_attention, shared_prefix_pages, workspace)

from _cases import max_rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"
bf = torch.bfloat16


def _ref(q, k, v, pos, scale):
    B, nh, hd = q.shape
    out = torch.empty(B, nh, hd)
    for b in range(B):
        n = int(pos[b]) + 1
        s = torch.einsum("hd,hdl->hl", q[b].float(), k[b, :, :, :n].float()) * scale
        p = torch.softmax(s, dim=-1)
        out[b] = torch.einsum("hl,hld->hd", p, v[b, :, :n].float())
    return out


@pytest.mark.parametrize("hd,L,pos", [(64, 16, [15, 0, 7]), (128, 4104, [4103, 5, 2047, 2048]),
                                      (64, 2056, [2055, 1000])])
def test_decode_attention_vs_fp32(hd, L, pos):
    g = torch.Generator().manual_seed(hd + L)
    B, nh, maxb = len(pos), 4, len(pos) + 2
    q = torch.randn(B, nh, hd, generator=g).to(bf)
    kc = torch.randn(maxb, nh, hd, L, generator=g).to(bf)      # head_dim-major keys
    vc = torch.randn(maxb, nh, L, hd, generator=g).to(bf)
    positions = torch.tensor(pos, dtype=torch.int64)
    scale = hd ** -0.5
    ref = _ref(q, kc[:B], vc[:B], positions, scale)
    kd, vd = kc.to(DEV), vc.to(DEV)
    ws = workspace(maxb, nh, hd, L, DEV)
    print(f"decode_attention hd={hd} L={L} pos={pos}", flush=True)
    out = decode_attention(q.to(DEV), kd[:B], vd[:B], positions.to(DEV), scale, ws)
    assert out.dtype == bf and out.shape == (B, nh, hd)
    assert max_rel_err(out.cpu(), ref) <= 1e-2


def test_decode_attention_7b_shape():
    """32 heads of 128 at the 7B benchmark's context (8192 prompt + 512 steps)."""
    g = torch.Generator().manual_seed(7)
    B, nh, hd, L = 3, 32, 128, 8704
    q = torch.randn(B, nh, hd, generator=g).to(bf)
    kc = (torch.randn(B, nh, hd, L, generator=g) * 0.5).to(bf)
    vc = (torch.randn(B, nh, L, hd, generator=g) * 0.5).to(bf)
    positions = torch.tensor([8192, 8703, 3000], dtype=torch.int64)
    ref = _ref(q, kc, vc, positions, hd ** -0.5)
    print("decode_attention 7B shape", flush=True)
    out = decode_attention(q.to(DEV), kc.to(DEV), vc.to(DEV), positions.to(DEV), hd ** -0.5)
    assert max_rel_err(out.cpu(), ref) <= 1e-2


@pytest.mark.parametrize("hd,max_pages,pos", [(64, 3, [47, 0, 16, 15]),
                                              (128, 260, [4159, 2047, 2048, 100]),
                                              (128, 544, [8192, 8703, 17])])
def test_paged_decode_attention_vs_fp32(hd, max_pages, pos):
    """The cache in 16-position pages of a random block table (page 0 never
    used): the same attention as over the dense cache the pages hold."""
    g = torch.Generator().manual_seed(hd + max_pages)
    B, nh = len(pos), 4 if hd == 64 else 32
    num_pages = B * max_pages + 5
    table = (torch.randperm(num_pages - 1, generator=g)[:B * max_pages] + 1).to(torch.int32)
    table = table.view(B, max_pages)
    cache = PagedKVCache(num_pages, nh, hd, "cpu")
    cache.k.copy_((torch.randn(cache.k.shape, generator=g) * 0.5).to(bf))
    cache.v.copy_((torch.randn(cache.v.shape, generator=g) * 0.5).to(bf))
    q = torch.randn(B, nh, hd, generator=g).to(bf)
    positions = torch.tensor(pos, dtype=torch.int64)
    kd, vd = cache.dense(table, B, max_pages * PAGE)
    ref = _ref(q, kd, vd, positions, hd ** -0.5)
    print(f"paged decode_attention hd={hd} pages={max_pages} pos={pos}", flush=True)
    out = paged_decode_attention(q.to(DEV), cache.k.to(DEV), cache.v.to(DEV), table.to(DEV),
                                 positions.to(DEV), hd ** -0.5)
    assert out.shape == (B, nh, hd)
    assert max_rel_err(out.cpu(), ref) <= 1e-2


@pytest.mark.parametrize("hd", [64, 128])
def test_paged_decode_attention_masks_entries_outside_the_cache(hd):
    """Table entries outside [0, pages) (-1, pages, a large id) are never read
    through: their positions drop out of the softmax, and a sequence with no
    position left gets zeros (head_dim 64: the VALU kernel; 128: the
    matrix-core kernel)."""
    g = torch.Generator().manual_seed(3)
    nh, max_pages = 4, 140
    pos = [2239, 2239, 300, 40]
    B = len(pos)
    num_pages = B * max_pages + 1
    table = (torch.randperm(num_pages - 1, generator=g)[:B * max_pages] + 1).to(torch.int32)
    table = table.view(B, max_pages).clone()
    table[0, 5] = -1
    table[0, 130] = num_pages            # in the second 2048-position chunk
    table[1, :128] = 1 << 30             # the whole first chunk of sequence 1
    table[2, 3] = -7
    table[3, :3] = -1                    # every page sequence 3 uses
    cache = PagedKVCache(num_pages, nh, hd, "cpu")
    cache.k.copy_((torch.randn(cache.k.shape, generator=g) * 0.5).to(bf))
    cache.v.copy_((torch.randn(cache.v.shape, generator=g) * 0.5).to(bf))
    q = torch.randn(B, nh, hd, generator=g).to(bf)
    positions = torch.tensor(pos, dtype=torch.int64)
    ref = torch.zeros(B, nh, hd)
    for b in range(B):
        keep = [l for l in range(pos[b] + 1) if 0 <= int(table[b, l // PAGE]) < num_pages]
        if not keep:
            continue
        pg = table[b, [l // PAGE for l in keep]].long()
        off = torch.tensor([l % PAGE for l in keep])
        k = cache.k[pg, :, :, off].float()          # (n, heads, hd)
        v = cache.v[pg, :, off, :].float()          # (n, heads, hd)
        s = torch.einsum("hd,nhd->hn", q[b].float(), k) * hd ** -0.5
        ref[b] = torch.einsum("hn,nhd->hd", torch.softmax(s, dim=-1), v)
    print(f"paged decode_attention masked table entries hd={hd}", flush=True)
    out = paged_decode_attention(q.to(DEV), cache.k.to(DEV), cache.v.to(DEV), table.to(DEV),
                                 positions.to(DEV), hd ** -0.5).cpu()
    assert torch.isfinite(out.float()).all()
    assert torch.equal(out[3], torch.zeros(nh, hd, dtype=bf))
    assert max_rel_err(out[:3], ref[:3]) <= 1e-2


@pytest.mark.parametrize("B,hd", [(6, 128), (8, 128), (40, 128), (8, 64)])
def test_paged_decode_attention_shared_prompt(B, hd):
    """Rows sharing their first pages (one prompt behind every sequence), one
    shared entry masked, sequences shorter than the shared prompt.  With the
    sharing declared, the chunks inside the prompt read each page once for
    several sequences: at head_dim 64 four sequences per workgroup on the
    VALU, the same bits as without it; at 128 up to 32 per workgroup on the
    matrix cores (another order of the fp32 sums, the probabilities as bf16
    high and low parts), within a rounding step of the undeclared result.
    Both match fp32 attention over the pages."""
    g = torch.Generator().manual_seed(11 + B + hd)
    nh, sp, own = 4, 392, 24                   # 392 shared pages: three whole chunks and a part
    max_pages = sp + own
    num_pages = sp + B * own + 1
    perm = torch.randperm(num_pages - 1, generator=g) + 1
    table = torch.empty(B, max_pages, dtype=torch.int32)
    table[:, :sp] = perm[:sp].to(torch.int32)
    table[:, sp:] = perm[sp:].to(torch.int32).view(B, own)
    table[:, 70] = -1                           # masked for every sequence (inside chunk 0)
    pos = [sp * PAGE + 5, max_pages * PAGE - 1, 5000, sp * PAGE + 300, 4095, 2047, 6300, 6271]
    pos = (pos + torch.randint(0, max_pages * PAGE, (max(B - len(pos), 0),), generator=g).tolist())[:B]
    cache = PagedKVCache(num_pages, nh, hd, "cpu")
    cache.k.copy_((torch.randn(cache.k.shape, generator=g) * 0.5).to(bf))
    cache.v.copy_((torch.randn(cache.v.shape, generator=g) * 0.5).to(bf))
    q = torch.randn(B, nh, hd, generator=g).to(bf)
    positions = torch.tensor(pos, dtype=torch.int64)
    assert shared_prefix_pages(table, B) == sp
    ref = torch.zeros(B, nh, hd)
    for b in range(B):
        keep = [l for l in range(pos[b] + 1) if int(table[b, l // PAGE]) >= 0]
        pg = table[b, [l // PAGE for l in keep]].long()
        off = torch.tensor([l % PAGE for l in keep])
        k = cache.k[pg, :, :, off].float()
        v = cache.v[pg, :, off, :].float()
        s = torch.einsum("hd,nhd->hn", q[b].float(), k) * hd ** -0.5
        ref[b] = torch.einsum("hn,nhd->hd", torch.softmax(s, dim=-1), v)
    args = (q.to(DEV), cache.k.to(DEV), cache.v.to(DEV), table.to(DEV), positions.to(DEV), hd ** -0.5)
    print(f"paged decode_attention shared prompt B={B} hd={hd}", flush=True)
    plain = paged_decode_attention(*args).cpu()
    shared = paged_decode_attention(*args, shared_pages=sp).cpu()
    if hd == 64:
        assert torch.equal(plain.view(torch.int16), shared.view(torch.int16))
    else:
        pf, sf = plain.float(), shared.float()
        # one bf16 step is at most 2^-7 of the value
        assert ((sf - pf).abs() <= pf.abs() * 2.0 ** -7 + 1e-4 * pf.abs().max()).all()
        assert (plain.view(torch.int16) != shared.view(torch.int16)).float().mean() <= 0.01
    assert max_rel_err(shared, ref) <= 1e-2
    assert max_rel_err(plain, ref) <= 1e-2


def _causal_ref(q, k, v, scale):
    """fp32 causal attention on the CPU: (N, heads, L, hd)."""
    qf, kf, vf = q.float(), k.float(), v.float()
    L = q.shape[-2]
    s = torch.matmul(qf, kf.transpose(-1, -2).contiguous()) * scale
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    return torch.matmul(torch.softmax(s, dim=-1), vf)


@pytest.mark.parametrize("N,nh,L", [(1, 2, 8), (2, 3, 200), (1, 2, 392), (1, 4, 1024), (1, 2, 4104),
                                    (1, 8, 1032), (2, 16, 520)])
def test_prefill_attention_vs_fp32(N, nh, L):
    """Causal prefill attention on the matrix-core kernel against fp32
    attention on the CPU: one partial 256-query block, several, prompts
    ending inside a key block, a prompt past 4096 (the last query block
    partly outside it), and head counts that split over the eight XCDs (the
    head-per-XCD grid), with two sequences.  Bar 1e-2 (bf16 output and bf16
    softmax weights)."""
    from evo2_flash_amd.attention import prefill_attention
    g = torch.Generator().manual_seed(L + nh)
    hd = 128
    q = torch.randn(N, nh, L, hd, generator=g).to(bf)
    k = torch.randn(N, nh, L, hd, generator=g).to(bf)
    v = torch.randn(N, nh, L, hd, generator=g).to(bf)
    ref = _causal_ref(q, k, v, hd ** -0.5)
    print(f"prefill_attention N={N} heads={nh} L={L}", flush=True)
    out = prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), hd ** -0.5).cpu()
    assert out.shape == q.shape and out.dtype == bf
    assert torch.isfinite(out.float()).all()
    assert max_rel_err(out, ref) <= 1e-2


def test_prefill_attention_peaked_scores():
    """Large scores (a softmax close to one-hot, and rows whose running max
    jumps late in the sweep): the online rescaling keeps the sums exact
    enough."""
    from evo2_flash_amd.attention import prefill_attention
    g = torch.Generator().manual_seed(5)
    N, nh, L, hd = 1, 2, 640, 128
    q = (torch.randn(N, nh, L, hd, generator=g) * 4).to(bf)
    k = (torch.randn(N, nh, L, hd, generator=g) * 4).to(bf)
    k[:, :, 600] *= 3                  # a late key that dominates the rows after it
    v = torch.randn(N, nh, L, hd, generator=g).to(bf)
    ref = _causal_ref(q, k, v, hd ** -0.5)
    print("prefill_attention peaked scores", flush=True)
    out = prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), hd ** -0.5).cpu()
    assert max_rel_err(out, ref) <= 1e-2


def _rotary64(x, pos, inv_freq, factor):
    """Neox rotary in fp64: x (n, heads, hd) at positions pos (n,)."""
    ang = (pos.double() / factor)[:, None] * inv_freq.double()
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x.double().chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _near(got, ref):
    """One bf16 rounding (2^-9 of the value) of an fp32 rotation whose angles
    (below 100 rad here) carry 2^-23 relative errors: 2^-16 of |x| <= 8."""
    assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + 8 * 2.0 ** -16).all()


def _qkv_case(rows, nh, hd, seed):
    g = torch.Generator().manual_seed(seed)
    wide = torch.randn(rows, 3 * nh * hd + 8, generator=g).to(bf)   # rows of a wider matrix
    inv_freq = 1.0 / 10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd)
    return g, wide, inv_freq


@pytest.mark.parametrize("nseq,nh,L", [(1, 1, 1), (2, 3, 15), (1, 4, 64), (3, 5, 65), (2, 4, 79),
                                       (1, 8, 200)])
def test_rotary_prefill_vs_fp64(nseq, nh, L):
    """Rotary, page writes and the transposed values of prompts around the
    kernel's 64 positions, 16-position pages and four heads; one block-table
    entry outside the cache.  Then attention over them at any L."""
    from evo2_flash_amd.attention import prefill_attention_rows, rotary_prefill
    hd = 128
    g, wide, inv_freq = _qkv_case(nseq * L, nh, hd, nseq + L)
    npg = -(-L // PAGE)
    num_pages = nseq * npg + 2
    table = (torch.randperm(num_pages - 1, generator=g)[:nseq * npg] + 1).int().view(nseq, npg)
    bad = table[0, -1].item()
    table[0, -1] = num_pages                       # not written through
    cache = PagedKVCache(num_pages, nh, hd, DEV)
    cache.k.fill_(7.0)
    cache.v.fill_(7.0)
    wd = wide.to(DEV)
    print(f"rotary_prefill nseq={nseq} heads={nh} L={L}", flush=True)
    q, k, vt = rotary_prefill(wd[:, :3 * nh * hd], cache, table.to(DEV), inv_freq.to(DEV), 4.0,
                              nseq, L)
    pos = torch.arange(L).repeat(nseq)
    qr, kr, vr = wide[:, :3 * nh * hd].reshape(nseq * L, 3, nh, hd).unbind(1)
    qr, kr = (_rotary64(t, pos, inv_freq, 4.0) for t in (qr, kr))
    qr, kr, vr = (t.view(nseq, L, nh, hd).transpose(1, 2) for t in (qr, kr, vr))
    _near(q.cpu(), qr)
    _near(k.cpu(), kr)
    assert torch.equal(vt.cpu()[..., :L], vr.transpose(-1, -2))
    assert (vt.cpu()[..., L:] == 0).all()
    # the pages hold the same k and v, a zero tail, and nothing else
    want = PagedKVCache(num_pages, nh, hd, "cpu")
    want.k.fill_(7.0)
    want.v.fill_(7.0)
    table[0, -1] = bad
    want.write_prompt(k.cpu(), vr, table)
    want.k[bad] = want.v[bad] = 7.0
    assert torch.equal(cache.k.cpu(), want.k) and torch.equal(cache.v.cpu(), want.v)
    out = torch.empty(nseq, L, nh, hd, dtype=bf, device=DEV)
    prefill_attention_rows(q, k, vt, hd ** -0.5, out.transpose(1, 2))
    ref = _causal_ref(q.cpu(), k.cpu(), vr, hd ** -0.5)
    assert max_rel_err(out.cpu().transpose(1, 2), ref) <= 1e-2


@pytest.mark.parametrize("B,nh,hd", [(1, 1, 64), (3, 9, 128), (5, 8, 32)])
def test_rotary_decode_vs_fp64(B, nh, hd):
    """One token per sequence, positions at both ends of pages, one sequence
    whose page lies outside the cache, heads around the kernel's eight."""
    from evo2_flash_amd.attention import rotary_decode
    g, wide, inv_freq = _qkv_case(B, nh, hd, B + nh)
    table = (torch.randperm(B * 3, generator=g) + 1).int().view(B, 3)
    pos = torch.tensor([15, 16, 47, 0, 31][:B])
    if B > 2:
        table[2, 2] = -1
    cache = PagedKVCache(B * 3 + 1, nh, hd, DEV)
    wd = wide.to(DEV)
    print(f"rotary_decode B={B} heads={nh} hd={hd}", flush=True)
    q = rotary_decode(wd[:, :3 * nh * hd], cache, table.to(DEV), pos.to(DEV), inv_freq.to(DEV), 4.0)
    qr, kr, vr = wide[:, :3 * nh * hd].reshape(B, 3, nh, hd).unbind(1)
    _near(q.cpu(), _rotary64(qr, pos, inv_freq, 4.0))
    kr = _rotary64(kr, pos, inv_freq, 4.0)
    kc, vc = cache.k.cpu(), cache.v.cpu()
    for b in range(B):
        pg, off = int(table[b, pos[b] // PAGE]), int(pos[b] % PAGE)
        if pg >= 0:
            _near(kc[pg, :, :, off], kr[b])
            assert torch.equal(vc[pg, :, off], vr[b])
            kc[pg, :, :, off] = vc[pg, :, off] = 0
    assert (kc == 0).all() and (vc == 0).all()      # and nowhere else


@pytest.mark.parametrize("factor", [1.0, 4.0])
def test_rotary_bits_of_the_separate_operators(factor):
    """Both rotary launches round as the fp32 operators of rotary_neox do, one
    rounding per product and sum: the same bits, positions up to 2^20."""
    from evo2_flash_amd.attention import rotary_decode, rotary_prefill
    from evo2_flash_amd.model import rotary_neox
    hd, nh, L, B = 128, 4, 1000, 33
    g, wide, inv_freq = _qkv_case(L, nh, hd, 11)
    wd, fd = wide.to(DEV)[:, :3 * nh * hd], inv_freq.to(DEV)
    q0, k0 = (wd.reshape(L, 3, nh, hd)[:, i] for i in (0, 1))
    table = (torch.randperm(B * 64, generator=g)[:B * 64] + 1).int().view(B, 64).to(DEV)
    cache = PagedKVCache(B * 64 + 1, nh, hd, DEV)
    print(f"rotary bits factor={factor}", flush=True)
    q, k, _ = rotary_prefill(wd, cache, table, fd, factor, 1, L)
    pos = torch.arange(L, device=DEV)
    for got, x in ((q, q0), (k, k0)):
        assert torch.equal(got[0].transpose(0, 1), rotary_neox(x, pos, fd, factor))
    pos = torch.randint(0, 1 << 20, (B,), generator=g).to(DEV)
    q = rotary_decode(wd[:B], cache, table, pos, fd, factor)
    assert torch.equal(q, rotary_neox(q0[:B], pos, fd, factor))
    pos = torch.randint(0, 1024, (B,), generator=g).to(DEV)
    rotary_decode(wd[:B], cache, table, pos, fd, factor)
    page = table[torch.arange(B, device=DEV), pos // PAGE].long()
    assert torch.equal(cache.k[page, :, :, pos % PAGE], rotary_neox(k0[:B], pos, fd, factor))


@pytest.mark.parametrize("L", [40, 41])
def test_attention_layer_cast_to_bf16(L):
    """A layer after .to(torch.bfloat16), its inv_freq buffer with it: the
    prompt's and the next token's keys rotate by the cast frequencies."""
    from evo2_flash_amd.config import HyenaConfig
    from evo2_flash_amd.model import Evo2Attention, rotary_neox
    cfg = HyenaConfig(hidden_size=256, num_attention_heads=2, num_hidden_layers=1,
                      attn_layer_idxs=[0])
    layer = Evo2Attention(cfg, 9, 4, 1, rope_factor=4.0, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(L)
    for p in layer.parameters():
        p.data.copy_(torch.randn(p.shape, generator=g, device=DEV) * 0.05)
    layer = layer.to(bf)
    assert layer.inv_freq.dtype == bf
    table = torch.tensor([[5, 2, 7, 1]], dtype=torch.int32, device=DEV)
    x = torch.randn(L + 1, 256, generator=g, device=DEV).to(bf)
    print(f"attention layer cast to bf16 L={L}", flush=True)
    with torch.no_grad():
        layer.forward_prefill(x[:L], 1, L, table)
        layer.forward_decode(x[L:], torch.tensor([L], device=DEV), table)
        # the keys of either call, projected by the call's own GEMM
        for rows, pos in ((x[:L], torch.arange(L, device=DEV)),
                          (x[L:], torch.tensor([L], device=DEV))):
            k = layer.qkv_proj(rows)[0].view(-1, 3, 2, 128)[:, 1]
            want = rotary_neox(k, pos, layer.inv_freq, 4.0)
            page = table[0, pos // PAGE].long()
            assert torch.equal(layer.cache.k[page, :, :, pos % PAGE], want)


@pytest.mark.parametrize("trained", ["qkv_proj", "x"])
def test_attention_layer_gradient_at_odd_lengths(trained):
    """A prompt whose length is no multiple of 8 is differentiable, in the input
    and in a trained qkv_proj.weight: the gradient of an fp32 layer, the output
    of the layer without gradients."""
    from evo2_flash_amd.config import HyenaConfig
    from evo2_flash_amd.model import Evo2Attention, rotary_neox
    cfg = HyenaConfig(hidden_size=256, num_attention_heads=2, num_hidden_layers=1,
                      attn_layer_idxs=[0])
    L = 41
    layer = Evo2Attention(cfg, 9, 4, 1, rope_factor=4.0, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(3)
    for p in layer.parameters():
        p.data.copy_(torch.randn(p.shape, generator=g, device=DEV) * 0.05)
    table = torch.tensor([[5, 2, 7, 1]], dtype=torch.int32, device=DEV)
    x = torch.randn(L, 256, generator=g, device=DEV).to(bf)
    go = torch.randn(L, 256, generator=g, device=DEV).to(bf)
    print(f"attention layer gradient of {trained}", flush=True)
    plain = layer.forward_prefill(x, 1, L, table)
    leaf = (layer.qkv_proj.weight if trained == "qkv_proj" else x).requires_grad_()
    out = layer.forward_prefill(x, 1, L, table)
    out.backward(go)
    assert max_rel_err(out.detach(), plain) <= 1e-2
    # the same in fp32 on the CPU
    xr, wr = x.detach().cpu().float(), layer.qkv_proj.weight.detach().cpu().float()
    ref = (wr if trained == "qkv_proj" else xr).requires_grad_()
    q, k, v = (xr @ wr.t()).view(L, 3, 2, 128).unbind(1)
    pos, f = torch.arange(L), layer.inv_freq.cpu()
    q, k = rotary_neox(q, pos, f, 4.0), rotary_neox(k, pos, f, 4.0)
    s = torch.einsum("ihd,jhd->hij", q, k) * 128 ** -0.5
    s = s.masked_fill(torch.ones(L, L).triu(1).bool(), float("-inf"))
    o = torch.einsum("hij,jhd->ihd", s.softmax(-1), v).reshape(L, 256)
    o = o @ layer.o_proj.weight.detach().cpu().float().t()
    o.backward(go.cpu().float())
    assert max_rel_err(leaf.grad.cpu().float(), ref.grad) <= 2e-2   # some ten roundings of 2^-9


@pytest.mark.parametrize("form", ["int64", "cpu", "strided"])
def test_rotary_prefill_block_table_forms(form):
    """Tables that PagedKVCache.write_prompt takes: the pages an int32 table on
    the device gives."""
    from evo2_flash_amd.attention import rotary_prefill
    hd, nh, nseq, L = 128, 2, 2, 40
    g, wide, inv_freq = _qkv_case(nseq * L, nh, hd, 5)
    table = (torch.randperm(6, generator=g) + 1).view(nseq, 3)
    given = {"int64": table.to(DEV), "cpu": table,
             "strided": table.int().t().contiguous().to(DEV).t()}[form]
    caches = []
    print(f"rotary_prefill block table {form}", flush=True)
    for t in (table.int().to(DEV), given):
        caches.append(PagedKVCache(7, nh, hd, DEV))
        rotary_prefill(wide.to(DEV)[:, :3 * nh * hd], caches[-1], t, inv_freq.to(DEV), 1.0, nseq, L)
    assert torch.equal(caches[0].k, caches[1].k) and torch.equal(caches[0].v, caches[1].v)
    assert (caches[0].k[1:].abs().amax((1, 2, 3)) > 0).all()


@pytest.mark.parametrize("L", [1, 41, 129, 200])
def test_prefill_attention_infinite_value_stays_in_its_dim(L):
    """An infinite value of the first key makes that dim infinite for every
    query; the dim before it, whose row ends where that key's begins, is as
    without it.  The values' padding runs over whole key blocks, past the
    prompt's last 64 positions too."""
    from evo2_flash_amd.attention import prefill_attention_rows, rotary_prefill
    hd, nh, nseq = 128, 2, 2
    g, wide, inv_freq = _qkv_case(nseq * L, nh, hd, L)
    qkv = wide[:, :3 * nh * hd].contiguous()
    v = qkv.view(nseq, L, 3, nh, hd)[:, :, 2]
    v[:, 0, :, 60] = float("inf")
    npg = -(-L // PAGE)
    table = (torch.randperm(nseq * npg, generator=g) + 1).int().view(nseq, npg).to(DEV)
    cache = PagedKVCache(nseq * npg + 1, nh, hd, DEV)
    out = torch.empty(nseq, nh, L, hd, dtype=bf, device=DEV)
    print(f"prefill_attention infinite value L={L}", flush=True)
    q, k, vt = rotary_prefill(qkv.to(DEV), cache, table, inv_freq.to(DEV), 1.0, nseq, L)
    prefill_attention_rows(q, k, vt, 128 ** -0.5, out)
    assert (out[..., 60] == float("inf")).all()
    v[:, 0, :, 60] = 0
    out[..., 60] = 0
    ref = _causal_ref(q.cpu(), k.cpu(), v.transpose(1, 2), 128 ** -0.5)
    ref[..., 60] = 0
    assert max_rel_err(out.cpu(), ref) <= 1e-2
    assert vt.shape[3] == -(-L // 128) * 128 and (vt[..., L:] == 0).all()


@pytest.mark.parametrize("L", [203, 1001, 3001])
@pytest.mark.parametrize("spread", [0.3, 1.0, 3.0])
def test_prefill_rows_as_precise_as_fused_torch(L, spread):
    """Lengths off eights came to this kernel from torch's fused attention: its
    error against 64 bits is no larger (within 1% of that error, which the draw of
    the inputs moves)."""
    from evo2_flash_amd.attention import prefill_attention_rows
    g = torch.Generator(device=DEV).manual_seed(L)
    q, k, v = (torch.randn(1, 8, L, 128, generator=g, device=DEV).to(torch.bfloat16)
               for _ in range(3))
    q = (q.float() * spread).to(torch.bfloat16)
    vt = torch.zeros(1, 8, 128, -(-L // 128) * 128, dtype=torch.bfloat16, device=DEV)
    vt[..., :L] = v.transpose(-1, -2)
    out = torch.empty_like(q)
    print(f"prefill rows precision L={L} spread={spread}", flush=True)
    prefill_attention_rows(q, k, vt, 128 ** -0.5, out)
    fused = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True,
                                                             scale=128 ** -0.5)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * 128 ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
    ref = torch.matmul(torch.softmax(s, -1), v.double())
    own, torchs = (float((t.double() - ref).norm() / ref.norm()) for t in (out, fused))
    assert own <= 1.01 * torchs, (own, torchs)
