"""tq::attend (attention of raw queries) on meta tensors: its checks and output shape.

One set of checks serves both kernels behind the op, so what either refuses is refused before
any launch; driven here with meta tensors, as tests/test_op_checks_cpu.py does for the others.
"""

import pytest
import torch

from turboquant_pytorch._ops import ops

B, HQ, HKV, SQ, SK, D = 2, 8, 2, 100, 300, 128
F16, U8 = torch.float16, torch.uint8


def _e(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="meta")


def _args(**kw):
    n = B * HKV * SK
    a = dict(q=_e(B, HQ, SQ, D, dtype=torch.bfloat16), pi=_e(2, D, D, dtype=F16), se=_e(D, D, dtype=F16),
             codes=_e(n, 32, dtype=U8), signs=_e(n, 16, dtype=U8), rn=_e(n, dtype=F16), kn=_e(n, dtype=F16),
             kcent=_e(4, dtype=F16), bits=3, vcodes=_e(n, 48, dtype=U8), vn=_e(n, dtype=F16), vcent=_e(8), vbits=3,
             vpit=_e(2, D, D, dtype=F16), hkv=HKV, sk=SK, stride=0, coeff=0.01, scale=0.09, causal=True, mask=None,
             out=torch.float32, ws=1)
    a.update(kw)
    return ops().attend(*a.values())


@pytest.mark.parametrize("mask", [None, _e(SQ, SK), _e(B, 1, SQ, SK, dtype=torch.bfloat16), _e(1, 1, 1, SK)])
def test_attend_shape(mask):
    out = _args(mask=mask)
    assert out.shape == (B, SQ, HQ, D) and out.dtype == torch.float32


@pytest.mark.parametrize("bad,match", [
    (dict(q=_e(B, HQ, D)), "expected"),
    (dict(pi=_e(D, D, dtype=F16)), "split Pi"),
    (dict(se=_e(D, D)), "S_eff"),
    (dict(signs=_e(B * HKV * SK, 15, dtype=U8)), "packed_qjl_signs"),
    (dict(vn=_e(B * HKV * SK - 1, dtype=F16)), "vec_norms"),
    (dict(hkv=3), "multiple"),
    (dict(stride=SK - 1), "kv_stride"),
    (dict(stride=SK + 1), "holds"),
    (dict(mask=_e(B, 1, SQ, SK + 1)), "expand|size"),
    (dict(out=torch.int32), "out_dtype"),
    (dict(ws=3), "workspace"),
])
def test_attend_refuses(bad, match):
    with pytest.raises(RuntimeError, match=match):
        _args(**bad)


@pytest.mark.parametrize("mdt", [torch.bfloat16, torch.float16, torch.float64, torch.bool])
@pytest.mark.parametrize("few", [False, True])
def test_mask_checks_convert_nothing(mdt, few):
    """The checks look at a mask's shape only: a conversion belongs to the call that uses it, once
    (tests/test_gpu_prefill_expanded.py counts those)."""
    from torch.profiler import ProfilerActivity, profile

    sq = 1 if few else SQ
    m = _e(B, 1, sq, SK, dtype=mdt)
    k = dict(q=_e(B, HQ, sq, D, dtype=torch.bfloat16), mask=m)
    n = B * HKV * SK
    with profile(activities=[ProfilerActivity.CPU]) as prof:
        _args(**k)
        ops().attention(_e(B, HQ, sq, D, dtype=F16), _e(B, HQ, sq, D), _e(n, 32, dtype=U8), _e(n, 16, dtype=U8),
                        _e(n, dtype=F16), _e(n, dtype=F16), _e(4, dtype=F16), 3, _e(n, 48, dtype=U8), _e(n, dtype=F16),
                        _e(8), 3, _e(2, D, D, dtype=F16), HKV, SK, 0, 0.01, 0.09, False, m, torch.float32, 1)
    names = [e.name for e in prof.events()]
    assert any("tq::attend" in x for x in names) and any("tq::attention" in x for x in names)
    assert not [x for x in names if "_to_copy" in x or "contiguous" in x]
