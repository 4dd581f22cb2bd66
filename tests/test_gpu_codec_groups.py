"""The 8-code-group stream kernels of the stand-alone codec against the general kernels.

Rows of a multiple of 8 codes that are contiguous take the stream kernels; a row stride takes the
general ones.  Both are exact, so every byte, code and f16 value must be equal: at block edges (256
groups), with a partial last dword, at every bit width, with ties and non-finite coordinates.
"""

import pytest
import torch

from turboquant_pytorch import _native

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(fn, *args):
    assert fn(*args, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("b", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("n,d", [(1, 8), (1, 40), (255, 8), (257, 8), (33, 128), (1000, 80), (4099, 64)])
def test_groups_equal_general(n, d, b):
    print("case:", n, d, b, flush=True)
    lib, p = _native.lib(), _native.ptr
    g = torch.Generator(device=DEV).manual_seed(n + d + b)
    oc, pad = d * b // 8, 4
    codes = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, d), device=DEV, dtype=torch.int32, generator=g)
    wide = torch.zeros(n, d + pad, device=DEV, dtype=torch.int32)
    wide[:, :d] = codes

    def out(cols, dtype, fill):
        return torch.full((n * cols + 64,), fill, device=DEV, dtype=dtype)

    # pack: codes wider than b bits are masked; nothing past the last byte is written
    a, c = out(oc, torch.uint8, 7), out(oc, torch.uint8, 7)
    _run(lib.tq_pack_bits, p(codes), n, d, d, b, p(a), oc)
    _run(lib.tq_pack_bits, p(wide), n, d, d + pad, b, p(c), oc)
    assert torch.equal(a, c) and (a[n * oc:] == 7).all()
    # unpack and dequantise of the same bytes; the padded output stride takes the general kernel
    u, gen = out(d, torch.int32, -1), torch.full((n, d + pad), -1, device=DEV, dtype=torch.int32)
    _run(lib.tq_unpack_bits, p(a), n, d, oc, b, p(u), d)
    _run(lib.tq_unpack_bits, p(a), n, d, oc, b, p(gen), d + pad)
    assert torch.equal(u[:n * d].view(n, d), gen[:, :d]) and torch.equal(gen[:, :d], codes & ((1 << b) - 1))
    assert (u[n * d:] == -1).all()
    cent = torch.randn(1 << b, device=DEV, generator=g).half()
    v, gen = out(d, torch.float16, 9.0), torch.full((n, d + pad), 9.0, device=DEV, dtype=torch.float16)
    _run(lib.tq_dequantize, p(a), n, d, oc, p(cent), b, p(v), d)
    _run(lib.tq_dequantize, p(a), n, d, oc, p(cent), b, p(gen), d + pad)
    assert torch.equal(v[:n * d].view(n, d), gen[:, :d]) and (v[n * d:] == 9.0).all()
    # quantise: coordinates on the boundaries, infinities and NaN among them
    bounds = torch.sort(torch.randn((1 << b) - 1, device=DEV, generator=g)).values.contiguous()
    y = torch.randn(n, d, device=DEV, generator=g)
    y[0, :5] = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -0.0], device=DEV)
    y[n // 2, 1] = bounds[0]
    y[n - 1, d - 1] = bounds[-1]
    yw = torch.zeros(n, d + pad, device=DEV)
    yw[:, :d] = y
    a, c = out(oc, torch.uint8, 7), out(oc, torch.uint8, 7)
    _run(lib.tq_quantize_pack, p(y), n, d, d, p(bounds), b, p(a), oc)
    _run(lib.tq_quantize_pack, p(yw), n, d, d + pad, p(bounds), b, p(c), oc)
    assert torch.equal(a, c) and (a[n * oc:] == 7).all()
