"""Head sizes that run on padded rows (attn_pad.hip): rows copied in pieces of
up to 16 bytes (half a row is a whole number of them and every array is aligned
to them) against the same rows copied element by element (one array starts one
element off).  Both make the same padded rows, so every output is the same to
the last bit; the oracle covers the element-wise copy at the other sizes.
"""
import numpy as np
import pytest

import glacier_attn as ga

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    assert torch.cuda.is_available(), "GPU tests need a ROCm GPU"
    made = ga.GpuAttentionEngine(0, ga.PREC_BF16)
    yield made
    made.close()


def one_off(x):
    """The same values, the array's start one element past a 16-byte boundary."""
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    moved = flat[1:].view(x.shape)
    moved.copy_(x)
    assert moved.data_ptr() % 16 == x.element_size()
    return moved


# 8, 24 and 72: pieces for fp32 only; the others for both types, up to the
# widest row (240: one row of 30 or 60 pieces in 256).
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("d", [8, 16, 24, 48, 72, 80, 112, 144, 240])
@pytest.mark.parametrize("lengths,hq,hkv", [((1,), 1, 1), ((37, 5), 3, 1), ((130,), 4, 2)])
def test_pieces_match_elements(engine, lengths, hq, hkv, d, dtype):
    print(f"[padded heads] lengths={lengths} heads={hq}/{hkv} d={d} {dtype}", flush=True)
    T = sum(lengths)
    gen = torch.Generator(device="cuda").manual_seed(T + d)
    q, k, v, do = (torch.randn(T, h, d, device="cuda", generator=gen).to(getattr(torch, dtype))
                   for h in (hq, hkv, hkv, hq))
    cu = None if len(lengths) == 1 else np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    out, lse, q_rot, k_rot = engine.forward(q, k, v, 1.0e6, cu_seqlens=cu)
    moved = engine.forward(q, one_off(k), v, 1.0e6, cu_seqlens=cu, out=one_off(q))
    for a, b in zip(moved, (out, lse, q_rot, k_rot)):
        assert torch.equal(a, b)
    want = engine.backward(do, q_rot, k_rot, v, out, lse, 1.0e6, cu_seqlens=cu)
    got = engine.backward(do, q_rot, one_off(k_rot), v, out, lse, 1.0e6, cu_seqlens=cu,
                          dk=one_off(k))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


# halves of whole 8- and 4-byte pieces only, and the longest rows of each; more
# rows than one workgroup's, with a remainder
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("d", [4, 20, 100, 200, 248, 252])
def test_narrower_pieces_match_elements(engine, d, dtype):
    test_pieces_match_elements(engine, (130, 71), 6, 2, d, dtype)
