"""dK/dV of a group of query heads (attn_kernels.hip, attn_bwd_reduce_kernel):
partials of up to two, of up to four, and of any number of heads in pieces of
eight, each with a remainder, with and without split dK/dV tiles, against the
oracle.  The gates are the library's: 1e-4 of the largest value in fp32 (sums of
at most 237 products of fp32 values), 2e-2 with bf16 tensors (a partial and a
gradient are rounded to within 2^-8 of themselves, P and dS likewise before their
sums).
"""
import numpy as np
import pytest

import glacier_attn as ga
import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GATE = {"float32": 1e-4, "bfloat16": 2e-2}


@pytest.fixture(scope="module")
def engines():
    assert torch.cuda.is_available(), "GPU tests need a ROCm GPU"
    made = {"float32": ga.GpuAttentionEngine(0, ga.PREC_FP32),
            "bfloat16": ga.GpuAttentionEngine(0, ga.PREC_BF16)}
    yield made
    for e in made.values():
        e.close()


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("ratio,hkv,d", [(1, 1, 96), (2, 2, 64), (3, 1, 96), (4, 1, 32), (5, 2, 96),
                                         (7, 4, 96), (8, 1, 128), (9, 1, 96), (16, 2, 64),
                                         (17, 1, 128), (24, 2, 32)])
def test_group_sums_match_oracle(engines, ratio, hkv, d, dtype):
    print(f"[group sums] ratio={ratio} kv heads={hkv} d={d} {dtype}", flush=True)
    lens, base = (200, 37), 1.0e6
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, hq = sum(lens), ratio * hkv
    x = [oracle.fill_normal((T, h, d), 90 + n, 0.0, s)
         for n, (h, s) in enumerate([(hq, 1.0), (hkv, 1.0), (hkv, 1.0), (hq, 0.01)])]
    if dtype == "bfloat16":
        x = [oracle.round_bf16(a) for a in x]
    ref = oracle.layer_fwd_bwd_varlen(*x, cu, base)
    q, k, v, do = (torch.from_numpy(a).to("cuda", getattr(torch, dtype)) for a in x)
    out, lse, q_rot, k_rot = engines[dtype].forward(q, k, v, base, cu_seqlens=cu)
    _, dk, dv = engines[dtype].backward(do, q_rot, k_rot, v, out, lse, base, cu_seqlens=cu)
    for got, name in ((dk, "dk"), (dv, "dv")):
        err = oracle.max_rel_err(got.float().cpu().numpy(), ref[name])
        assert err <= GATE[dtype], (name, err)
