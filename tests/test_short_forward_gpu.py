"""Short sequences: the bf16 forward that turns K itself (attn_fwd.hip,
attn_fwd_kernel_ks with RK: every sequence at most 128 tokens, 16- or 32-query
workgroups) against the same forward behind rope_k (64-query workgroups pinned,
which never take it).  Both round the same fp32 rotation once and walk the
same chunks, so every output is the same to the last bit.
"""
import os

import numpy as np
import pytest

import glacier_attn as ga

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engines():
    assert torch.cuda.is_available(), "GPU tests need a ROCm GPU"
    old = os.environ.get("GLACIER_ATTN_FWD_ROWS")
    try:
        os.environ["GLACIER_ATTN_FWD_ROWS"] = "64"
        pinned = ga.GpuAttentionEngine(0, ga.PREC_BF16)
        os.environ["GLACIER_ATTN_FWD_ROWS"] = "32"
        rows32 = ga.GpuAttentionEngine(0, ga.PREC_BF16)
    finally:
        if old is None:
            del os.environ["GLACIER_ATTN_FWD_ROWS"]
        else:
            os.environ["GLACIER_ATTN_FWD_ROWS"] = old
    made = {"pinned": pinned, "rows32": rows32, "auto": ga.GpuAttentionEngine(0, ga.PREC_BF16)}
    yield made
    for e in made.values():
        e.close()


LENGTHS = [(1,), (31,), (32,), (33,), (64,), (97,), (127,), (128,), (129,), (128, 1, 64, 17), (65, 128, 129)]


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (28, 4, 128), (3, 3, 128)])
def test_forward_turning_k_matches_rope_k(engines, hq, hkv, d, lengths):
    print(f"[short forward] lengths={lengths} heads={hq}/{hkv} d={d}", flush=True)
    T = sum(lengths)
    gen = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(T, h, d, device="cuda", generator=gen).bfloat16() for h in (hq, hkv, hkv))
    cu = None if len(lengths) == 1 else np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    want = engines["pinned"].forward(q, k, v, 1.0e6, cu_seqlens=cu)
    for name in ("auto", "rows32"):
        kept = k.clone()
        got = engines[name].forward(q, k, v, 1.0e6, cu_seqlens=cu)
        plain = engines[name].forward(q, k, v, 1.0e6, cu_seqlens=cu, save=False)[0]
        assert torch.equal(k, kept)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        assert torch.equal(plain, want[0])


@pytest.mark.parametrize("off", [2, 4])
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (28, 4, 128)])
def test_unaligned_k_stays_with_rope_k(engines, hq, hkv, d, off):
    """K in a view off 16 bytes is not for the DMA: rope_k turns it, and the
    results are those of an aligned K."""
    print(f"[short forward] K off by {2 * off} bytes heads={hq}/{hkv} d={d}", flush=True)
    T = 97
    gen = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(T, h, d, device="cuda", generator=gen).bfloat16() for h in (hq, hkv, hkv))
    moved = torch.empty(k.numel() + off, device="cuda", dtype=k.dtype)[off:].view(k.shape).copy_(k)
    assert moved.data_ptr() % 16 == 2 * off
    for a, b in zip(engines["auto"].forward(q, moved, v, 1.0e6), engines["auto"].forward(q, k, v, 1.0e6)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", ["out", "q_rot", "k_rot"])
@pytest.mark.parametrize("d", [64, 128])
def test_output_in_the_place_of_k(engines, name, d):
    """K is read before anything is written over it: the results of an output
    in K's memory are those of one beside it."""
    print(f"[short forward] {name} in K's place d={d}", flush=True)
    T, h = 97, 3
    gen = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(T, h, d, device="cuda", generator=gen).bfloat16() for _ in range(3))
    want = engines["auto"].forward(q, k, v, 1.0e6)
    for a, b in zip(engines["auto"].forward(q, k, v, 1.0e6, **{name: k}), want):
        assert torch.equal(a, b)
