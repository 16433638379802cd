"""Address tables given as host arrays (pointer low bit set): the limit is checked on the
host before any launch; at the limit and one past it the wrappers give the same results."""

import ctypes

import pytest
import torch

from nexusquant_amd import _lib

DEV = "cuda:0"


def _tagged(n):
    arr = (ctypes.c_uint64 * n)(*([4096] * n))
    return arr, ctypes.c_void_p(ctypes.addressof(arr) | 1)


def test_too_many_host_addresses_are_refused():
    lib = _lib.load()
    n = _lib.MAX_HOST_ADDRESSES // 2 + 1
    keep, ptr = _tagged(n)
    d = _lib.QuantDesc(n_tensors=n, batch=1, heads=1, seq_in=4, seq_out=4, head_dim=64, dtype=0, levels=4, src=ptr,
                       recon=ptr, hadamard_scale=0.125)
    assert lib.nq_quantize(ctypes.byref(d), None) == -1
    assert b"at most 64 addresses" in lib.nq_last_error()
    assert lib.nq_gather_rows(ptr, ptr, n, 0, 1, 1, 4, 4, 64, None, None, None) == -1
    c = _lib.CodesDesc(n_tensors=n, batch=1, heads=1, seq=4, head_dim=64, levels=4, syms=ptr, cosets=ptr, scales=ptr, out=ptr)
    assert lib.nq_dequantize(ctypes.byref(c), None) == -1
    p = _lib.PageDesc(n_pages=n, heads=1, tokens=4, head_dim=64, levels=4, src=ptr, codes=ptr, scales=ptr, out=ptr)
    assert lib.nq_page_encode(ctypes.byref(p), None) == -1 and lib.nq_page_decode(ctypes.byref(p), None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 12, 13])
def test_quantizer_and_codes_at_the_limit(n):
    """5 addresses a tensor: 12 tensors travel in the arguments, 13 through the ring."""
    from nexusquant_amd.codec import codes_int8, dequantize
    from nexusquant_amd.ops import gather_rows, quantize_tensors
    print(f"[gpu] tables n={n}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(n)
    xs = [torch.randn(1, 2, 77, 128, device=DEV, generator=g).half() for _ in range(n)]
    rec, cd = quantize_tensors(xs, is_key=True, levels=8, codes=True)
    copies = [t for x in xs for t in (x,) * 3]  # 3n tensors: 2 addresses each
    for x, c in zip(copies, gather_rows(copies)):
        assert torch.equal(x, c)
    for x, r, c, d, q in zip(xs, rec, cd, dequantize(cd), codes_int8(cd)):
        r1, c1 = quantize_tensors([x], is_key=True, levels=8, codes=True)
        assert torch.equal(r, r1[0]) and torch.equal(r, d) and torch.equal(q, codes_int8(c1)[0])
        assert all(torch.equal(getattr(c, f), getattr(c1[0], f)) for f in ("syms", "cosets", "scales"))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [16, 17])
def test_pages_at_the_limit(n):
    """4 addresses a key page: 16 pages travel in the arguments, 17 through the ring."""
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor
    print(f"[gpu] page tables n={n}", flush=True)
    comp = NexusQuantKVCompressor(head_dim=64, bits=3)
    g = torch.Generator(device=DEV).manual_seed(n)
    work = [(torch.randn(2, 9, 64, device=DEV, generator=g).half(), torch.randn(2, 9, 64, device=DEV, generator=g).half(),
             torch.arange(9, dtype=torch.int32) + 9 * i) for i in range(n)]
    pages = comp.compress_pages(work)
    for p, w, back in zip(pages, work, comp.decompress_pages(pages)):
        one = comp.compress_page(*w)
        assert torch.equal(p.key_codes, one.key_codes) and torch.equal(p.value_scales, one.value_scales)
        k, v = comp.decompress_page(one)
        assert torch.equal(back[0], k) and torch.equal(back[1], v)
