"""Attention over expanded key / value tiles (tq_prefill_attention, csrc/tq_dense.hip).

Many query rows per kv head take this path through compressed_attention and
TurboQuantCache.append_attend.  Reference: the float64 estimator on the device's own planes,
q_rot rounded to f16 and key centroids / S_eff at f16 as the estimator defines them.

Bars.  The kernel rounds V^ = C_v[c] vn to f16 (relative 2^-11 per element, independent signs)
and, at head_dim 64 / 128 with equal bits, the softmax weights too, so a row's relative error is
at most about sqrt(2) 2^-11 / sqrt(3) = 4e-4 (uniform rounding errors); q_rot's own f16 rounding
can fall either way between the f32 and the f64 rotation, which moves a score by 2^-11 of one
term in rare cases.  REL = 1e-3 covers both with a factor of two.
"""

import ctypes
import math

import pytest
import torch

from transformers_turboquant import TurboQuantCache
from turboquant_pytorch import _native, compressed_attention
from turboquant_pytorch.fused import attention_from_prepared
from turboquant_pytorch.kernels.attention import scores_from_prepared
from turboquant_pytorch.compressors import TurboQuantCompressorMSE, TurboQuantCompressorV2, _tables

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = 1e-3


def _unpack(p, b, d):
    bits = ((p.unsqueeze(-1) >> torch.arange(8, device=p.device, dtype=torch.uint8)) & 1)
    bits = bits.reshape(p.shape[0], -1)[:, : d * b].reshape(-1, d, b).long()
    return (bits << torch.arange(b, device=p.device)).sum(-1)


def _reference(q, kc, vc, ck, cv, mask=None, causal=False):
    B, Hq, Sq, D = q.shape
    _, Hkv, Sk, _ = ck["shape"]
    G, n = Hq // Hkv, B * Hkv * Sk
    pi, se = kc.Pi.double(), _tables(kc, q.device, True).s_eff16.double()
    codes = _unpack(ck["packed_key_indices"].reshape(n, -1), kc.mse_bits, D)
    sg = _unpack(ck["packed_qjl_signs"].reshape(n, -1), 1, D).double() * 2 - 1
    coeff = math.sqrt(math.pi / 2) / D
    kh = kc.centroids.half().double()[codes] * ck["vec_norms"].reshape(n, 1).double()
    kh += (sg @ se) * (coeff * ck["residual_norm"].reshape(n, 1).double())
    vh = vc.centroids.double()[_unpack(cv["packed_indices"].reshape(n, -1), vc.bits, D)]
    vh = vh * cv["vec_norms"].reshape(n, 1).double()
    kh, vh = (t.reshape(B, Hkv, Sk, D).repeat_interleave(G, dim=1) for t in (kh, vh))
    s = ((q.double() @ pi.T).half().double() @ kh.transpose(-2, -1).contiguous()) / math.sqrt(D)
    if mask is not None:
        s = s + mask.double().clamp(min=-3e38 / 1.4426950408889634)
    if causal:
        i = torch.arange(Sq, device=q.device)[:, None] + (Sk - Sq)
        s = s.masked_fill(torch.arange(Sk, device=q.device)[None] > i, -math.inf)
    return ((torch.softmax(s, -1) @ vh) @ vc.Pi.double()).transpose(1, 2)


def _make(d, bits, vbits, hq, hkv, sq, sk, dtype=torch.float32, B=2, scale=None, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + d + 7 * sk + sq)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    kc = TurboQuantCompressorV2(d, bits, seed=42, device=DEV)
    vc = TurboQuantCompressorMSE(d, vbits, seed=10042, device=DEV)
    k = r(B, hkv, sk, d)
    if scale is not None:
        k = k * scale(sk)
    return kc, vc, r(B, hq, sq, d).to(dtype), kc.compress(k.to(dtype)), vc.compress(r(B, hkv, sk, d).to(dtype))


def _err(got, ref):
    assert torch.isfinite(got).all()
    return ((got.double() - ref).norm() / ref.norm()).item()


_DT = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def _direct(q, kc, vc, ck, cv, mask=None, causal=False, out_dtype=torch.float32):
    """tq_prefill_attention through the C ABI: no choice of route, the mask as it lies in memory."""
    B, hq, sq, d = q.shape
    _, hkv, sk, _ = ck["shape"]
    tk, tv = _tables(kc, q.device, True), _tables(vc, q.device, False)
    lib, p = _native.lib(), _native.ptr
    m = mask.expand(B, hq, sq, sk) if mask is not None else None
    nb = lib.tq_prefill_workspace_size(B, hq, hkv, sq, sk, d, int(causal), int(m is not None))
    ws = torch.empty(nb, dtype=torch.uint8, device=DEV)
    out = torch.zeros(B, sq, hq, d, device=DEV, dtype=out_dtype)
    st = lib.tq_prefill_attention(
        p(q), _DT[q.dtype], q.stride(0), q.stride(1), q.stride(2), p(tk.pi_split), p(tk.s_eff16),
        p(ck["packed_key_indices"]), p(ck["packed_qjl_signs"]), p(ck["residual_norm"]), p(ck["vec_norms"]),
        p(tk.cent16), kc.mse_bits + 1, p(cv["packed_indices"]), p(cv["vec_norms"]), p(tv.cent32), vc.bits,
        p(tv.pit_split), B, hq, hkv, sq, sk, 0, d, math.sqrt(math.pi / 2) / d, 1 / math.sqrt(d), int(causal),
        p(m) if m is not None else None, _DT[m.dtype] if m is not None else 0,
        *(m.stride() if m is not None else (0, 0, 0, 0)), p(out), _DT[out_dtype], p(ws), ctypes.c_int64(nb),
        torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.tq_last_error()
    return out


@pytest.mark.parametrize("d,bits,vbits,hq,hkv,sq,sk,causal", [
    (128, 3, 3, 8, 2, 64, 64, True),       # one block of 256 columns, whole tiles
    (128, 2, 2, 8, 2, 65, 65, True),       # a second block and a second tile of one row / key
    (128, 4, 4, 7, 1, 73, 95, True),       # 36 rows of 7 heads per block, 4 columns idle
    (128, 3, 3, 4, 4, 300, 333, False),    # multi-head, ragged tail tile
    (128, 3, 3, 32, 8, 40, 3000, True),    # keys split over blocks, merged
    (128, 3, 2, 16, 2, 33, 1100, True),    # value bits below the key bits (hi + lo weights)
    (64, 3, 3, 12, 12, 129, 129, True),
    (64, 4, 4, 4, 2, 700, 1500, False),    # 4-wave blocks, split
    (64, 2, 1, 4, 2, 70, 31, False),       # fewer keys than a tile
    (32, 3, 3, 8, 2, 100, 257, False),
    (40, 2, 2, 4, 4, 130, 600, True),      # 5-byte sign rows: byte loads
    (48, 3, 4, 8, 2, 100, 900, True),      # 6-byte sign rows: 16-bit loads
    (80, 3, 3, 8, 2, 65, 530, True),
    (96, 4, 3, 6, 2, 90, 200, True),
    (112, 3, 3, 4, 1, 50, 90, False),
    (160, 3, 3, 4, 2, 66, 66, True),
    (192, 2, 2, 4, 4, 70, 700, True),
    (200, 3, 3, 4, 4, 64, 64, False),
    (224, 3, 3, 4, 4, 64, 100, True),
    (256, 4, 4, 4, 2, 100, 300, True),
])
def test_prefill_shapes(d, bits, vbits, hq, hkv, sq, sk, causal):
    print("case:", d, bits, vbits, hq, hkv, sq, sk, causal, flush=True)
    kc, vc, q, ck, cv = _make(d, bits, vbits, hq, hkv, sq, sk)
    got = compressed_attention(q, kc, vc, ck, cv, causal=causal)
    assert _err(got, _reference(q, kc, vc, ck, cv, causal=causal)) < REL


@pytest.mark.parametrize("d", [64, 80, 128, 256])
@pytest.mark.parametrize("mdt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sk,layout", [(160, "batch"), (161, "batch"), (200, "head"), (96, "strided")])
def test_prefill_masks(d, mdt, sk, layout):
    """Additive masks in their own type: broadcast over heads, per head, rows that start off a
    dword (odd key counts), and a layout that is not contiguous in keys.  Through the operator, whose
    rule keeps so few keys at head_dim 64 and 128 on the packed prefill kernel, and through the C entry,
    which has no rule and reads the mask where it lies."""
    print("case:", d, mdt, sk, layout, flush=True)
    sq, hq, hkv, B = 100, 8, 2, 2
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk)
    g = torch.Generator(device=DEV).manual_seed(sk)
    m = torch.randn(B, hq if layout == "head" else 1, sq, sk, device=DEV, generator=g).to(mdt)
    m[0, :, :, : sk // 3] = torch.finfo(mdt).min          # left padding
    m[1, :, 5:9, 40:] = -math.inf
    if layout == "strided":
        m = m.transpose(-1, -2).contiguous().transpose(-1, -2)
    ref = _reference(q, kc, vc, ck, cv, mask=m.expand(B, hq, sq, sk))
    assert _err(compressed_attention(q, kc, vc, ck, cv, attention_mask=m), ref) < REL
    assert _err(_direct(q, kc, vc, ck, cv, mask=m), ref) < REL


def _split(B, hq, hkv, sq, sk, d):
    """Whether a masked call's keys are split over blocks: its workspace then holds partial sums."""
    dp, tiles = (d + 31) // 32 * 32, (sk + 31) // 32
    q_part = 2 * dp * dp + (B * hq * sq * d * 2 + 255) // 256 * 256
    group = (_native.lib().tq_prefill_workspace_size(B, hq, hkv, sq, sk, d, 0, 1) - q_part) // (B * hkv)
    return group > (4 * tiles + 15) // 16 * 16 + tiles * (3 * dp * 64 + 256)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("mdt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,hq,hkv,sq,sk,split,causal", [
    (2, 8, 2, 40, 3000, True, False),     # keys split over blocks and merged
    (2, 8, 2, 40, 3000, True, True),
    (16, 16, 16, 130, 2304, False, False),  # a block of 72 tiles: the tile factors are loaded anew after 64
    (16, 16, 16, 130, 2304, False, True),
])
def test_prefill_masks_of_long_calls(d, mdt, B, hq, hkv, sq, sk, split, causal):
    """The masked kernels over many tiles, through the C entry: left padding by finfo.min, whole rows
    and whole key ranges of a split without a real key, -inf, with and without a causal limit."""
    print("case:", d, mdt, B, sq, sk, causal, flush=True)
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk, B=B)
    assert _split(B, hq, hkv, sq, sk, d) == split
    low = torch.finfo(mdt).min
    m = torch.randn(B, 1, sq, sk, device=DEV, generator=torch.Generator(device=DEV).manual_seed(d)).to(mdt)
    m[0, :, :, : sk // 2] = low
    if mdt != torch.float16:  # f16's lowest value leaves 2^-7 of a score in f32
        m[1, :, 3] = low
    m[1, :, 5:9, 40:] = -math.inf
    ref = _reference(q, kc, vc, ck, cv, mask=m.expand(B, hq, sq, sk), causal=causal)
    assert _err(_direct(q, kc, vc, ck, cv, mask=m, causal=causal), ref) < REL


@pytest.mark.parametrize("d", [64, 80, 128])
@pytest.mark.parametrize("mdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", ["query", "padding"])
def test_prefill_masks_sliced_to_an_odd_key_count(d, mdt, rows):
    """16-bit masks cut from a wider buffer: every row starts on a dword and ends inside one.  The last
    key, masked in half of the rows, counts as any other, and the buffer's values past it (they would
    raise a key's weight to 1) are never used.  1101 keys: the operator takes the expanded kernels at
    every head dim; the C entry takes the mask where it lies."""
    print("case:", d, mdt, rows, flush=True)
    sq, sk, hq, hkv, B = 100, 1101, 8, 2, 2
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk)
    g = torch.Generator(device=DEV).manual_seed(sk)
    n = sq if rows == "query" else 1
    wide = torch.full((B, 1, n, 1200), 60.0, device=DEV, dtype=mdt)
    m = wide[..., :sk]
    m.copy_(torch.randn(B, 1, n, sk, device=DEV, generator=g))
    m[..., sk - 1] = 30.0                       # the last key outweighs every other one ...
    m[0, ..., sk - 1] = torch.finfo(mdt).min    # ... or has no weight
    m[1, :, : n // 2, sk - 1] = torch.finfo(mdt).min
    ref = _reference(q, kc, vc, ck, cv, mask=m.expand(B, hq, sq, sk))
    assert _err(compressed_attention(q, kc, vc, ck, cv, attention_mask=m), ref) < REL
    assert _err(_direct(q, kc, vc, ck, cv, mask=m), ref) < REL


@pytest.mark.parametrize("mdt,dev", [(torch.float32, DEV), (torch.bfloat16, DEV), (torch.bool, DEV),
                                     (torch.bfloat16, "cpu")])
@pytest.mark.parametrize("sq", [1, 20])
def test_masks_are_converted_once(mdt, dev, sq):
    """Few-row and decode calls read float32 masks: what one `.to` to the device and that type does,
    and no more."""
    from torch.profiler import ProfilerActivity, profile

    def copies(f):
        f()
        with profile(activities=[ProfilerActivity.CPU]) as prof:
            f()
        return sum(e.name == "aten::_to_copy" for e in prof.events())

    kc, vc, q, ck, cv = _make(64, 3, 3, 4, 4, sq, 300)
    m = torch.zeros(2, 1, sq, 300, device=dev, dtype=mdt)
    assert (copies(lambda: compressed_attention(q, kc, vc, ck, cv, attention_mask=m))
            == copies(lambda: m.to(q.device, torch.float32)))


@pytest.mark.parametrize("mdt,sk", [(torch.float32, 1100), (torch.bfloat16, 1101)])
def test_broadcast_masks_are_laid_out_once(mdt, sk):
    """A mask that the caller has expanded over batch and heads, and that has to be laid out anew
    (not contiguous in keys; 16-bit rows of an odd key count), is copied without its repeats: the
    call's memory grows by one [Sq, Sk] float32 plane (a second one while a 16-bit copy is converted),
    not by B x Hq of them."""
    d, sq, hq, hkv, B = 64, 100, 16, 4, 2
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk)
    g = torch.Generator(device=DEV).manual_seed(sk)
    one = torch.randn(sk, sq, device=DEV, generator=g).to(mdt)
    plain = one.t().contiguous()

    def peak(m):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        out = compressed_attention(q, kc, vc, ck, cv, attention_mask=m)
        return torch.cuda.max_memory_allocated() - base, out

    bare, ref = peak(plain.float())
    for m in (one.t().expand(B, hq, sq, sk), plain.expand(B, hq, sq, sk)):
        used, out = peak(m)
        assert torch.equal(out, ref)
        assert used - bare <= 2 * 4 * sq * sk + 4096


@pytest.mark.parametrize("d,bits,vbits,hq,hkv,sq,sk", [
    (64, 3, 3, 4, 4, 65, 1100),    # the packed path splits these over keys on its tiled kernel, although
    (64, 4, 4, 12, 6, 64, 1100),   # it has a prefill kernel for the bit widths
    (64, 2, 2, 4, 4, 128, 5000),
    (128, 3, 2, 4, 2, 64, 700),    # no prefill kernel for the bit widths, or for the head dim
    (80, 3, 3, 4, 2, 64, 700),
])
def test_weights_keep_their_lo_parts(d, bits, vbits, hq, hkv, sq, sk):
    """Where the packed path keeps the softmax weights as f16 hi + lo, so does the expanded one.  Zero
    queries make the weights the softmax of the mask alone; against V^ = f16(C_v vn) what is left is
    the weights' own error (2^-22, one f16 would leave 2e-4), their f32 sums and exponents (a few 1e-7
    each) and the hi + lo output rotation: below 1e-5 by a factor of three."""
    print("case:", d, bits, vbits, hq, hkv, sq, sk, flush=True)
    kc, vc, q, ck, cv = _make(d, bits, vbits, hq, hkv, sq, sk)
    q = torch.zeros_like(q)
    m = 2 * torch.randn(2, 1, sq, sk, device=DEV, generator=torch.Generator(device=DEV).manual_seed(d))
    n = 2 * hkv * sk
    vh = vc.centroids.float()[_unpack(cv["packed_indices"].reshape(n, -1), vc.bits, d)]
    vh = (vh * cv["vec_norms"].float().reshape(n, 1)).half().double()
    vh = vh.reshape(2, hkv, sk, d).repeat_interleave(hq // hkv, dim=1)
    ref = ((torch.softmax(m.double(), -1).expand(2, hq, sq, sk) @ vh) @ vc.Pi.double()).transpose(1, 2)
    q_rot, q_proj = kc.prepare_queries(q)
    errs = [_err(x, ref) for x in (attention_from_prepared(q_rot, q_proj, kc, vc, ck, cv, attention_mask=m),
                                   compressed_attention(q, kc, vc, ck, cv, attention_mask=m),
                                   _direct(q, kc, vc, ck, cv, mask=m))]
    print("errors: packed %.2e, expanded %.2e, expanded through the C entry %.2e" % tuple(errs), flush=True)
    assert max(errs) < 1e-5


@pytest.mark.parametrize("d,hq,hkv,sq,sk,masked", [
    (128, 8, 2, 70, 140, False), (128, 8, 2, 70, 1100, True), (128, 8, 8, 300, 1200, False),
    (64, 8, 2, 70, 1100, True), (64, 4, 4, 200, 200, False), (80, 8, 2, 40, 700, False), (80, 8, 2, 40, 700, True),
    (200, 4, 4, 70, 90, False),
])
def test_norms_that_are_not_finite(d, hq, hkv, sq, sk, masked):
    """A key whose f16 norm overflowed has scores of +-inf: no weight in the rows where it is -inf, NaN
    in the rows where it is +inf.  Neither the rows that do not attend it nor the other keys of its tile
    see any of it.  Row for row as on the packed path, whose score terms carry the norms apart."""
    print("case:", d, hq, hkv, sq, sk, masked, flush=True)
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk)
    g = torch.Generator(device=DEV).manual_seed(d)
    mask = None
    if masked:
        mask = torch.randn(2, 1, sq, sk, device=DEV, generator=g)
        mask[0, :, :, : sk // 3] = torch.finfo(torch.float32).min
    inf, nan, last = math.inf, math.nan, sk - sq // 2  # a key that the first half of the causal rows misses
    q_rot, q_proj = kc.prepare_queries(q)
    vn, rn = ck["vec_norms"], ck["residual_norm"]
    for head, key, v, r in ((0, last, inf, 1.0), (0, 3, 1e-4, 1e-5), (1, last, inf, inf), (2, last, 1.0, inf),
                            (3, last, nan, 1.0), (2, 5, inf, 1.0)):
        at = (head % (2 * hkv)) * sk + key
        vn.view(-1)[at], rn.view(-1)[at] = v, r
    want = attention_from_prepared(q_rot, q_proj, kc, vc, ck, cv, attention_mask=mask, causal=True)
    bad = torch.isnan(want)
    assert 0.05 < bad.float().mean() < 0.95  # rows of both kinds
    for got in (compressed_attention(q, kc, vc, ck, cv, attention_mask=mask, causal=True),
                _direct(q, kc, vc, ck, cv, mask=mask, causal=True)):
        assert torch.equal(torch.isnan(got), bad)
        assert _err(got[~bad], want[~bad].double()) < REL


@pytest.mark.parametrize("B,d,sq,sk,expanded", [(1, 192, 130, 600, True), (64, 192, 130, 700, False),
                                                (64, 192, 170, 700, True), (64, 128, 130, 700, True),
                                                (1, 192, 128, 700, False)])
def test_scores_route(B, d, sq, sk, expanded):
    """As test_prefill_route, for materialised scores (12 heads)."""
    kc, _, q, ck, _ = _make(d, 3, 3, 12, 12, sq, sk, B=B)
    t = _tables(kc, q.device, True)
    packed = scores_from_prepared(*kc.prepare_queries(q), ck["packed_key_indices"], ck["packed_qjl_signs"],
                                  ck["residual_norm"], ck["vec_norms"], t.cent16, 3, math.sqrt(math.pi / 2) / d, 12,
                                  sk, sk)
    got = kc.asymmetric_attention_scores(q, ck)
    assert torch.equal(got, packed) != expanded
    assert ((got - packed).norm() / packed.norm()).item() < 4e-5


@pytest.mark.parametrize("d,group,masked,ok", [
    (128, 128, False, True), (128, 136, False, False), (128, 72, True, False), (128, 64, True, True),
    (64, 128, True, True), (64, 136, False, False), (80, 64, False, True), (80, 72, False, False),
])
def test_group_sizes(d, group, masked, ok):
    """The largest GQA group does not depend on the route: what the packed kernels refuse is refused."""
    kc, vc, q, ck, cv = _make(d, 3, 3, group, 1, 3, 70, B=1)
    m = torch.zeros(1, 1, 3, 70, device=DEV) if masked else None
    for split_k in (True, False):
        if ok:
            assert _err(compressed_attention(q, kc, vc, ck, cv, attention_mask=m, split_k=split_k),
                        _reference(q, kc, vc, ck, cv)) < REL
        else:
            with pytest.raises(RuntimeError, match="group size"):
                compressed_attention(q, kc, vc, ck, cv, attention_mask=m, split_k=split_k)


@pytest.mark.parametrize("d,group,ok", [(128, 128, True), (128, 136, False), (160, 64, True), (160, 72, False)])
def test_group_sizes_of_scores(d, group, ok):
    """As test_group_sizes, for materialised scores."""
    kc, _, q, ck, _ = _make(d, 3, 3, group, 1, 3, 70, B=1)
    if ok:
        assert kc.asymmetric_attention_scores(q, ck).shape == (1, group, 3, 70)
    else:
        with pytest.raises(RuntimeError, match="group size"):
            kc.asymmetric_attention_scores(q, ck)


@pytest.mark.parametrize("d,sq,sk", [(128, 64, 96), (64, 140, 75), (80, 140, 64), (256, 140, 96)])
def test_expanded_scores_over_all_norms(d, sq, sk):
    """Every key's scores at f32 grade whatever its neighbours' norms (f16's whole range in a tile), and
    the infinities and NaNs of the packed path.  Per key: a key's rounding flips of q_rot (see
    test_expanded_scores) are a sum over sq rows here, so the bar of 2e-5 is four times that of a matrix.
    The sign of an infinity is a dot product's: where that is within its rounding of 0 (one part in 2^12
    of its size: less than a thousandth of them) it can fall either way."""
    kc, _, q, ck, _ = _make(d, 3, 3, 8, 2, sq, sk, scale=lambda n: 10 ** torch.linspace(
        -4, 3, n, device=DEV)[torch.randperm(n, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n))][:, None])
    q_rot, q_proj = kc.prepare_queries(q)
    t = _tables(kc, q.device, True)
    args = (ck["packed_key_indices"], ck["packed_qjl_signs"], ck["residual_norm"], ck["vec_norms"], t.cent16, 3,
            math.sqrt(math.pi / 2) / d, 2, sk, sk)
    want = scores_from_prepared(q_rot, q_proj, *args).double()
    assert torch.isfinite(want).all()
    got = kc.asymmetric_attention_scores(q, ck)
    err = (got.double() - want).norm(dim=2) / want.norm(dim=2)  # per (batch, head, key)
    print("largest error of a key: %.2e" % err.max().item(), flush=True)
    assert err.max() < 8e-5
    for key, v, r in ((1, math.inf, 1.0), (34, 1.0, math.inf), (40, math.inf, math.inf), (sk - 1, math.nan, 1.0)):
        for plane, x in (("vec_norms", v), ("residual_norm", r)):
            ck[plane].view(-1, sk)[:, key] = x
    want, got = scores_from_prepared(q_rot, q_proj, *args), kc.asymmetric_attention_scores(q, ck)
    fin = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), fin)
    assert (got.nan_to_num(0, 1, -1) != want.nan_to_num(0, 1, -1))[~fin].float().mean() < 1e-3
    assert _err(got[fin], want[fin].double()) < 2e-5


@pytest.mark.parametrize("B,d,hq,hkv,sq,sk,masked,expanded", [
    (1, 128, 32, 8, 64, 600, False, True),      # few long query blocks
    (1, 128, 32, 8, 32, 600, False, False),     # 128 columns: the packed kernel splits the keys
    (24, 128, 12, 12, 132, 2000, False, False),  # many sequences fill the packed kernel's grid
    (2, 128, 12, 12, 132, 2000, False, True),
    (48, 64, 12, 12, 64, 500, False, False),
    (1, 64, 12, 12, 63, 200, False, False),     # below 64 columns
    (8, 64, 12, 12, 64, 1100, True, False),     # under a mask: 64 columns are one block
    (8, 64, 12, 12, 65, 1100, True, True),      # the tiled kernel's split
    (48, 64, 12, 12, 96, 1500, True, False),
    (1, 128, 32, 8, 40, 900, True, True),
    (1, 80, 32, 32, 64, 300, False, True),      # no prefill kernel
    (48, 192, 12, 12, 64, 500, True, False),    # many wide keys for 64 columns
    (48, 192, 12, 12, 100, 500, True, True),
])
def test_prefill_route(B, d, hq, hkv, sq, sk, masked, expanded):
    """Which kernels a call takes, on both sides of each line of the rule: bit for bit those of the path
    named here, and in agreement with the other path."""
    print("case:", B, d, hq, hkv, sq, sk, masked, expanded, flush=True)
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk, B=B)
    m = torch.randn(B, 1, sq, sk, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)) if masked else None
    got = compressed_attention(q, kc, vc, ck, cv, attention_mask=m, causal=not masked)
    q_rot, q_proj = kc.prepare_queries(q)
    packed = attention_from_prepared(q_rot, q_proj, kc, vc, ck, cv, attention_mask=m, causal=not masked)
    direct = _direct(q, kc, vc, ck, cv, mask=m, causal=not masked)
    assert torch.equal(got, direct if expanded else packed)
    assert not torch.equal(packed, direct) and _err(direct, packed.double()) < REL


@pytest.mark.parametrize("d", [64, 128])
def test_prefill_rows_without_a_real_key(d):
    """A row whose mask is finfo.min everywhere attends all keys equally, as softmax does."""
    kc, vc, q, ck, cv = _make(d, 3, 3, 8, 2, 70, 100)
    m = torch.zeros(2, 1, 70, 100, device=DEV)
    m[0, :, 3] = torch.finfo(torch.float32).min
    m[1, :, :, 50:] = torch.finfo(torch.float32).min
    ref = _reference(q, kc, vc, ck, cv, mask=m.expand(2, 8, 70, 100))
    for got in (compressed_attention(q, kc, vc, ck, cv, attention_mask=m), _direct(q, kc, vc, ck, cv, mask=m)):
        assert _err(got, ref) < REL


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [80, 128])
def test_prefill_dtypes_and_strides(d, dtype):
    """Queries of each type, as the transposed view a projection leaves, and with rows that are
    not 16-byte aligned."""
    kc, vc, q, ck, cv = _make(d, 3, 3, 8, 2, 70, 140, dtype)
    ref = _reference(q, kc, vc, ck, cv, causal=True)
    base = compressed_attention(q, kc, vc, ck, cv, causal=True, out_dtype=torch.float32)
    assert _err(base, ref) < REL
    view = q.transpose(1, 2).contiguous().transpose(1, 2)
    buf = torch.empty(q.numel() + 1, device=DEV, dtype=dtype)[1:]
    off = buf.copy_(q.reshape(-1)).view(q.shape)
    for x in (view, off):
        assert torch.equal(compressed_attention(x, kc, vc, ck, cv, causal=True, out_dtype=torch.float32), base)
    out = compressed_attention(q, kc, vc, ck, cv, causal=True)
    assert out.dtype == dtype and torch.equal(out, base.to(dtype))


@pytest.mark.parametrize("qs,ks", [(1.0, 1.0), (1e-3, 3e2), (300.0, 1e-2), (1.0, 1e-4)])
def test_prefill_norm_ranges(qs, ks):
    """Key norms over five decades inside every tile (the tile's power of two follows its largest)
    and query norms that keep the scores in softmax's range.  The norm planes are f16, so the
    largest norm stays below 65504: sqrt(128) * 1.4 (the widest of these rows) * 10 * 3e2 = 4.8e4."""
    kc, vc, q, ck, cv = _make(128, 3, 3, 8, 2, 64, 320, scale=lambda s: ks * 10 ** torch.linspace(
        -4, 1, 32, device=DEV).repeat(s // 32)[:, None])
    got = compressed_attention(q * qs, kc, vc, ck, cv, causal=True)
    assert _err(got, _reference(q * qs, kc, vc, ck, cv, causal=True)) < REL


def test_prefill_chunk_over_cache_planes():
    """A prompt chunk through TurboQuantCache.append_attend: capacity planes (kv_stride) against
    the compact planes of one compression, bit for bit, and against the reference."""
    d, hq, hkv, sk, sq = 128, 8, 2, 700, 150
    g = torch.Generator(device=DEV).manual_seed(3)
    k, v, q = (torch.randn(2, h, n, d, device=DEV, generator=g).bfloat16()
               for h, n in ((hkv, sk), (hkv, sk), (hq, sq)))
    kc = TurboQuantCompressorV2(d, 3, seed=42, device=DEV)
    vc = TurboQuantCompressorMSE(d, 3, seed=10042, device=DEV)
    cache = TurboQuantCache()
    cache.append(0, kc, vc, k[:, :, : sk - sq], v[:, :, : sk - sq])
    got = cache.append_attend(0, kc, vc, k[:, :, sk - sq:], v[:, :, sk - sq:], q, causal=True)
    ck, cv = kc.compress(k), vc.compress(v)
    assert torch.equal(got, compressed_attention(q, kc, vc, ck, cv, causal=True, out_dtype=torch.float32))
    assert _err(got, _reference(q, kc, vc, ck, cv, causal=True)) < REL


@pytest.mark.parametrize("sq,sk", [(100, 100), (40, 3000)])
def test_prefill_rounds_over_a_small_workspace(sq, sk):
    """A workspace of one (batch, kv head) runs them in rounds over the same memory: bit-identical
    to all at once; one byte less is refused."""
    d, hq, hkv, B = 128, 32, 8, 1
    kc, vc, q, ck, cv = _make(d, 3, 3, hq, hkv, sq, sk, B=B)
    tk, tv = _tables(kc, q.device, True), _tables(vc, q.device, False)
    lib = _native.lib()
    full = lib.tq_prefill_workspace_size(B, hq, hkv, sq, sk, d, 1, 0)
    q_part = 2 * d * d + (B * hq * sq * d * 2 + 255) // 256 * 256  # S_eff fragments and q_rot
    group = (full - q_part) // (B * hkv)
    assert (full - q_part) % (B * hkv) == 0

    def run(nbytes):
        out = torch.zeros(B, sq, hq, d, device=DEV)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        p = _native.ptr
        st = lib.tq_prefill_attention(
            p(q), 0, q.stride(0), q.stride(1), q.stride(2), p(tk.pi_split), p(tk.s_eff16),
            p(ck["packed_key_indices"]), p(ck["packed_qjl_signs"]), p(ck["residual_norm"]), p(ck["vec_norms"]),
            p(tk.cent16), 3, p(cv["packed_indices"]), p(cv["vec_norms"]), p(tv.cent32), 3, p(tv.pit_split), B, hq,
            hkv, sq, sk, 0, d, math.sqrt(math.pi / 2) / d, 1 / math.sqrt(d), 1, None, 0, 0, 0, 0, 0, p(out), 0,
            p(ws), ctypes.c_int64(nbytes), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return st, out

    st, whole = run(full)
    assert st == 0
    st, one = run(q_part + group)
    assert st == 0 and torch.equal(one, whole)
    assert run(q_part + group - 1)[0] == -1
    assert torch.equal(whole, compressed_attention(q, kc, vc, ck, cv, causal=True))


def test_prefill_under_graph_capture():
    kc, vc, q, ck, cv = _make(128, 3, 3, 8, 2, 200, 900)
    ref = compressed_attention(q, kc, vc, ck, cv, causal=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        compressed_attention(q, kc, vc, ck, cv, causal=True)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = compressed_attention(q, kc, vc, ck, cv, causal=True)
    for rep in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), rep
        compressed_attention(q * (rep + 2), kc, vc, ck, cv, causal=True)
        torch.cuda.synchronize()


@pytest.mark.parametrize("d,bits,hq,hkv,sq,sk,dtype", [
    (128, 3, 8, 2, 33, 64, torch.float32),       # a second row chunk of one row, whole key tiles
    (128, 2, 4, 4, 130, 1, torch.bfloat16),      # one key
    (128, 4, 7, 1, 50, 333, torch.float16),      # ragged tail, blocks over several heads
    (128, 3, 16, 2, 64, 3001, torch.float32),    # key ranges split over blocks
    (64, 3, 12, 12, 129, 129, torch.float32),
    (32, 2, 8, 2, 65, 100, torch.float32),
    (40, 3, 4, 2, 70, 95, torch.bfloat16),       # byte loads of the packed rows
    (80, 4, 4, 1, 40, 200, torch.float32),
    (160, 3, 4, 2, 70, 70, torch.float32),
    (192, 3, 4, 4, 130, 50, torch.float32),
    (256, 2, 4, 2, 66, 161, torch.float16),
])
def test_expanded_scores(d, bits, hq, hkv, sq, sk, dtype):
    """Materialised scores: f32 sums over q_rot (f16) and keys at f32 grade.  The reference rounds
    the f64 rotation to f16; an entry whose rounding falls the other way in the kernel's f32
    rotation (about 2^-11 of them) moves a score by 2^-11 of one of d terms, a relative error of
    about 2^-11 sqrt(2^-11) = 1e-5 over a matrix of scores; the bar is twice that.  Rows past a
    head's end or keys past Sk must not be written: the output is the whole buffer, filled with a
    marker by a larger allocation around it."""
    print("case:", d, bits, hq, hkv, sq, sk, dtype, flush=True)
    kc, _, q, ck, _ = _make(d, bits, bits, hq, hkv, sq, sk, dtype)
    got = kc.asymmetric_attention_scores(q, ck)
    B, G, n = 2, hq // hkv, 2 * hkv * sk
    pi, se = kc.Pi.double(), _tables(kc, q.device, True).s_eff16.double()
    sg = _unpack(ck["packed_qjl_signs"].reshape(n, -1), 1, d).double() * 2 - 1
    kh = kc.centroids.half().double()[_unpack(ck["packed_key_indices"].reshape(n, -1), kc.mse_bits, d)]
    kh = kh * ck["vec_norms"].reshape(n, 1).double()
    kh += (sg @ se) * (math.sqrt(math.pi / 2) / d * ck["residual_norm"].reshape(n, 1).double())
    kh = kh.reshape(B, hkv, sk, d).repeat_interleave(G, dim=1)
    ref = (q.double() @ pi.T).half().double() @ kh.transpose(-2, -1).contiguous()
    assert got.shape == ref.shape and got.dtype == torch.float32
    assert _err(got, ref) < 2e-5

    # the C entry point writes exactly [B, Hq, Sq, Sk]
    t = _tables(kc, q.device, True)
    guard, lib, p = 4096, _native.lib(), _native.ptr
    buf = torch.full((ref.numel() + 2 * guard,), 7.0, device=DEV)
    nb = lib.tq_prefill_scores_workspace_size(B, hq, hkv, sq, sk, d)
    ws = torch.empty(nb, dtype=torch.uint8, device=DEV)
    st = lib.tq_prefill_scores(
        p(q), {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype], q.stride(0), q.stride(1), q.stride(2),
        p(t.pi_split), p(t.s_eff16), p(ck["packed_key_indices"]), p(ck["packed_qjl_signs"]), p(ck["residual_norm"]),
        p(ck["vec_norms"]), p(t.cent16), bits, B, hq, hkv, sq, sk, 0, d, math.sqrt(math.pi / 2) / d,
        p(buf) + 4 * guard, p(ws), ctypes.c_int64(nb), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert st == 0 and (buf[:guard] == 7).all() and (buf[-guard:] == 7).all()
    assert torch.equal(buf[guard:-guard].view(ref.shape), got)


def test_expanded_scores_past_64_tiles():
    """Blocks of more than 64 key tiles load the tile factors anew: 96 (batch, kv head)s of 2048 rows are
    1536 blocks of 128 rows, and about eight blocks per compute unit leave 67 of the 90 tiles to one."""
    B, hkv, sq, sk, d = 8, 12, 2048, 2880, 32
    kc, _, q, ck, _ = _make(d, 3, 3, hkv, hkv, sq, sk, dtype=torch.bfloat16, B=B,
                            scale=lambda n: torch.linspace(0.5, 40, n, device=DEV)[:, None])
    got = kc.asymmetric_attention_scores(q, ck)
    t = _tables(kc, q.device, True)
    r, p = kc.prepare_queries(q[:, :, :64])
    want = scores_from_prepared(r, p, ck["packed_key_indices"], ck["packed_qjl_signs"], ck["residual_norm"],
                                ck["vec_norms"], t.cent16, 3, math.sqrt(math.pi / 2) / d, hkv, sk, sk)
    assert ((got[:, :, :64] - want).norm() / want.norm()).item() < 2e-5
    r, p = kc.prepare_queries(q[:, :, -33:])
    want = scores_from_prepared(r, p, ck["packed_key_indices"], ck["packed_qjl_signs"], ck["residual_norm"],
                                ck["vec_norms"], t.cent16, 3, math.sqrt(math.pi / 2) / d, hkv, sk, sk)
    assert ((got[:, :, -33:] - want).norm() / want.norm()).item() < 2e-5
