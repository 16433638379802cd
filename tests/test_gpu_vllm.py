"""GPU parity of the vLLM page caller and the paged decode-attention consumer.

- nq_page_encode / nq_page_decode: bit for bit against the Tier-B spec
  (oracle/nq_spec.c), within tolerance of the reference's fixture.
- nq_page_logits and nq_paged_attention: within tolerance of the Tier-A
  restatement / the reference's fixture (fp32 sums in another order; the
  fused attention also skips the per-token fp16 rounding of decoded values).
- nibble packing: exact.
"""

import math

import numpy as np
import pytest
import torch

from oracle import spec as S
from oracle import torch_ref as T

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BASE = {"b2": 10000.0, "b3": 500000.0, "b4": 10000.0}


def _np16(t):
    return t.detach().cpu().numpy()


def _same_fp16(a, b):
    a = np.asarray(a)
    b = np.asarray(b)
    return bool(np.all((a.view(np.uint16) == b.view(np.uint16)) | ((a == 0) & (b == 0))))


def _tables(pos, d, base, h):
    c, s = T.rope_cos_sin(torch.as_tensor(pos).float(), d, base)
    return np.tile(c.numpy(), (h, 1)), np.tile(s.numpy(), (h, 1))


def _page(h, n, d, dtype, seed, pos_hi=200000):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn(h, n, d, generator=g) * 2
    k[:, :, :3] *= 6
    v = torch.randn(h, n, d, generator=g) * 0.5
    pos = torch.randint(0, pos_hi, (n,), generator=g, dtype=torch.int32)
    return k.to(dtype), v.to(dtype), pos


@pytest.mark.parametrize("bits,d,dtype", [(2, 128, torch.float16), (3, 128, torch.float32), (4, 64, torch.float16),
                                          (2, 256, torch.bfloat16), (3, 128, torch.float16), (4, 128, torch.float32)])
def test_page_encode_decode_bitexact_vs_spec(bits, d, dtype):
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor
    print(f"[gpu] page codec bits={bits} d={d} {dtype}", flush=True)
    h, n = 4, 40
    base = 500000.0
    comp = NexusQuantKVCompressor(head_dim=d, bits=bits, rope_base=base)
    k, v, pos = _page(h, n, d, dtype, seed=bits * 100 + d)
    page = comp.compress_page(k.to(DEV), v.to(DEV), pos.to(DEV))
    kd, vd = comp.decompress_page(page)
    torch.cuda.synchronize()
    c, s = _tables(pos, d, base, h)
    L = 2 ** bits
    for x, key, codes, scales, dec in ((k, True, page.key_codes, page.key_scales, kd),
                                       (v, False, page.value_codes, page.value_scales, vd)):
        rows = x.float().numpy().reshape(-1, d)
        want_c, want_s, _ = S.page_encode(rows, L, c if key else None, s if key else None)
        assert np.array_equal(_np16(codes).reshape(-1, d), want_c)
        assert np.array_equal(_np16(scales).reshape(-1).view(np.uint16), want_s.view(np.uint16))
        want_d = S.page_decode(want_c, want_s, key, c if key else None, s if key else None)
        assert _same_fp16(_np16(dec).reshape(-1, d), want_d)
    assert page.num_valid == n and page.positions.dtype == torch.int32


@pytest.mark.parametrize("tag,bits", [("b2", 2), ("b3", 3), ("b4", 4)])
def test_pages_within_tolerance_of_reference_fixture(golden, tag, bits):
    from nexusquant_amd.vllm_backend import CompressedPage, NexusQuantKVCompressor
    print(f"[gpu] page fixture {tag}", flush=True)
    g = golden("vllm_pages")
    base = BASE[tag]
    k, v, pos = (torch.from_numpy(g[f"{tag}_{n}"]) for n in ("k", "v", "pos"))
    h, n, d = k.shape
    comp = NexusQuantKVCompressor(head_dim=d, bits=bits, rope_base=base)
    page = comp.compress_page(k.to(DEV), v.to(DEV), pos.to(DEV))
    c, s = _tables(pos, d, base, h)
    for role, key, codes in (("k", True, page.key_codes), ("v", False, page.value_codes)):
        got = _np16(codes).reshape(-1, 8)
        ref = g[f"{tag}_{role}c"].reshape(-1, 8)
        _, _, margin = S.page_encode(g[f"{tag}_{role}"].astype(np.float32).reshape(-1, d), 2 ** bits,
                                     c if key else None, s if key else None)
        mism = (got != ref).any(1)
        assert mism.mean() <= 1e-2 and np.all(margin.reshape(-1)[mism] < 1e-5)
    # decode and logits of the reference's own page
    ref_page = CompressedPage(*(torch.from_numpy(g[f"{tag}_{n}"]).to(DEV) for n in ("kc", "vc", "ks", "vs", "pos")),
                              num_valid=n)
    kd, vd = comp.decompress_page(ref_page)
    for got, name in ((kd, "kdec"), (vd, "vdec")):
        a = _np16(got).astype(np.float32).reshape(-1, d)
        r = g[f"{tag}_{name}"].astype(np.float32).reshape(-1, d)
        tol = np.spacing(np.maximum(np.abs(a), np.abs(r)).astype(np.float16)).astype(np.float32)
        assert np.all(np.abs(a - r) <= tol + 1e-6 * np.abs(r).max(1, keepdims=True))
    q = torch.from_numpy(g[f"{tag}_q"])
    lg = comp.decompress_for_attention(ref_page, q.to(DEV)).cpu().numpy()
    ref = g[f"{tag}_logits"]
    keys32 = T.vllm_decompress_keys_fp32(*(torch.from_numpy(g[f"{tag}_{n}"]) for n in ("kc", "ks", "pos")), base)
    bound = (q.float().norm(dim=-1)[:, :, None] * keys32.norm(dim=-1)[:, None, :]).numpy() / math.sqrt(d)
    assert np.all(np.abs(lg - ref) <= 1e-5 * bound + 1e-6)


def test_decompress_for_attention_fp32_and_bf16_queries():
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor
    print("[gpu] page logits dtypes", flush=True)
    comp = NexusQuantKVCompressor(head_dim=128, bits=3, rope_base=10000.0)
    k, v, pos = _page(8, 33, 128, torch.float16, seed=4)
    page = comp.compress_page(k.to(DEV), v.to(DEV), pos.to(DEV))
    for qdt in (torch.float32, torch.bfloat16, torch.float16):
        q = torch.randn(8, 5, 128, generator=torch.Generator().manual_seed(5)).to(qdt)
        lg = comp.decompress_for_attention(page, q.to(DEV)).cpu()
        ref = T.vllm_decompress_for_attention(page.key_codes.cpu(), page.key_scales.cpu(), pos, q, 10000.0)
        assert torch.allclose(lg, ref, rtol=1e-4, atol=1e-4)


def test_nibble_pack_unpack_match_reference(golden):
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor as C
    print("[gpu] nibbles", flush=True)
    g = golden("vllm_pages")
    codes = torch.from_numpy(g["nib_codes"]).to(DEV)
    packed = C.pack_codes_nibble(codes)
    assert np.array_equal(packed.cpu().numpy(), g["nib_packed"])
    assert np.array_equal(C.unpack_codes_nibble(packed, 33).cpu().numpy(), g["nib_unpacked"])
    even = torch.randint(-4, 5, (7, 128), dtype=torch.int8).to(DEV)
    assert torch.equal(C.unpack_codes_nibble(C.pack_codes_nibble(even), 128), even)


def _fixture_cache(g):
    from nexusquant_amd.vllm_backend import CompressedPage
    cache = {}
    for i in range(6):
        cache[i] = CompressedPage(*(torch.from_numpy(g[n][i]).to(DEV)
                                    for n in ("fwd_kc", "fwd_vc", "fwd_ks", "fwd_vs", "fwd_pos")), num_valid=16)
    return cache


def _close_fp16(got, ref, rel_l2=1e-3, bf16=False):
    """Attended outputs: within 2^-9 of the row's largest entry (a few fp16 ulps
    of it), plus one bf16 ulp of the entry for bf16 outputs, which round the fp16
    result once more; and 1e-3 relative L2 overall -- 2^-9, bf16's rounding
    bound, for bf16 outputs: an fp16 result one ulp off the reference's moves
    the bf16 rounding by a whole bf16 ulp (2^-8) in about 8 % of the entries."""
    a = np.asarray(got, np.float32)
    r = np.asarray(ref, np.float32)
    if bf16:
        rel_l2 = max(rel_l2, 2.0 ** -9)
    assert np.linalg.norm(a - r) <= rel_l2 * max(np.linalg.norm(r), 1e-30)
    scale = np.abs(r).max(axis=-1, keepdims=True)
    tol = 2.0 ** -9 * scale + 1e-6 + (2.0 ** -7 * np.abs(r) if bf16 else 0.0)
    assert np.all(np.abs(a - r) <= tol)


def test_paged_forward_matches_reference_fixture(golden):
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print("[gpu] paged forward fixture", flush=True)
    g = golden("vllm_pages")
    attn = NexusQuantPagedAttention(NexusQuantKVCompressor(head_dim=128, bits=2, rope_base=10000.0))
    cache = _fixture_cache(g)
    query = torch.from_numpy(g["fwd_query"]).to(DEV)
    out = attn.forward(query, cache, cache, [[0, 1, 2], [3, 99, 4], [5], [2, 0]],
                       torch.from_numpy(g["fwd_ctx"]))
    torch.cuda.synchronize()
    ref = g["fwd_out"]
    got = out.cpu().numpy()
    assert np.all(got[2] == 0) and np.all(ref[2] == 0)  # empty row
    _close_fp16(got, ref)


def _oracle_forward(cache, query, tables, ctx, base, group):
    pages = {}
    for bid, p in cache.items():
        kc, vc, ks, vs, pos = (t.cpu() for t in (p.key_codes, p.value_codes, p.key_scales, p.value_scales,
                                                  p.positions))
        if group > 1:
            kc, vc, ks, vs = (t.repeat_interleave(group, dim=0) for t in (kc, vc, ks, vs))
        pages[bid] = (kc, vc, ks, vs, pos)
    return T.vllm_paged_forward(query.cpu(), pages, tables, ctx, base)


@pytest.mark.parametrize("group,qdt", [(1, torch.float16), (2, torch.float16), (4, torch.float16),
                                       (8, torch.float16), (1, torch.float32), (2, torch.bfloat16)])
def test_paged_forward_long_context_gqa_and_dtypes(group, qdt):
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print(f"[gpu] paged forward group={group} {qdt}", flush=True)
    kv, d, base = 2, 128, 500000.0
    comp = NexusQuantKVCompressor(head_dim=d, bits=3, rope_base=base)
    attn = NexusQuantPagedAttention(comp)
    gen = torch.Generator().manual_seed(group * 7 + 1)
    cache = {}
    work = []
    sizes = [16] * 70 + [5, 600, 16, 1]  # many 16-token pages, a partial page, one page larger than a chunk
    for bid, n in enumerate(sizes):
        k = (torch.randn(kv, n, d, generator=gen) * 2).to(torch.float16)
        v = (torch.randn(kv, n, d, generator=gen) * 0.5).to(torch.float16)
        pos = torch.arange(n, dtype=torch.int32) + 16 * bid
        work.append((k.to(DEV), v.to(DEV), pos))
    for bid, page in enumerate(comp.compress_pages(work)):
        cache[bid] = page
    tables = [list(range(74)), [71, 5, 3, 200, 72, 73], [9], [0, 1, 2]]
    ctx = [70 * 16 + 5 + 600 + 10, 10 ** 6, 0, -7]
    query = torch.randn(4, kv * group, d, generator=gen).to(qdt)
    out = attn.forward(query.to(DEV), cache, cache, tables, torch.tensor(ctx))
    torch.cuda.synchronize()
    assert out.dtype == qdt
    ref = _oracle_forward(cache, query, tables, ctx, base, group)
    _close_fp16(out.float().cpu().numpy(), ref.float().numpy(), bf16=qdt == torch.bfloat16)


@pytest.mark.parametrize("d,group,qdt,vmul", [(64, 8, torch.float16, 1.0), (256, 8, torch.float16, 1.0),
                                              (256, 4, torch.bfloat16, 1.0), (64, 2, torch.float32, 1.0),
                                              (128, 8, torch.float16, 1e-4), (128, 1, torch.float16, 2e3)])
def test_paged_forward_head_dims_and_value_ranges(d, group, qdt, vmul):
    """Every head_dim with 8 and fewer query heads per kv head; values scaled
    down (row scales near fp16's subnormals) and up (scales near 2^6) so the
    value weights' fp16 hi/lo split is exercised at both ends of its range."""
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print(f"[gpu] paged forward d={d} group={group} {qdt} vmul={vmul}", flush=True)
    kv, base = 2, 10000.0
    comp = NexusQuantKVCompressor(head_dim=d, bits=2, rope_base=base)
    attn = NexusQuantPagedAttention(comp)
    gen = torch.Generator().manual_seed(d + group)
    work = []
    sizes = [16] * 40 + [3, 40, 16]
    for bid, n in enumerate(sizes):
        k = (torch.randn(kv, n, d, generator=gen) * 2).to(torch.float16)
        v = (torch.randn(kv, n, d, generator=gen) * vmul).to(torch.float16)
        pos = torch.arange(n, dtype=torch.int32) + 16 * bid
        work.append((k.to(DEV), v.to(DEV), pos))
    cache = dict(enumerate(comp.compress_pages(work)))
    tables = [list(range(43)), [41, 7, 42], [40]]
    ctx = [40 * 16 + 3 + 40 + 16, 10 ** 6, 2]
    query = torch.randn(3, kv * group, d, generator=gen).to(qdt)
    out = attn.forward(query.to(DEV), cache, cache, tables, torch.tensor(ctx))
    torch.cuda.synchronize()
    ref = _oracle_forward(cache, query, tables, ctx, base, group)
    _close_fp16(out.float().cpu().numpy(), ref.float().numpy(), bf16=qdt == torch.bfloat16)


@pytest.mark.parametrize("d,group,qdt", [(128, 8, torch.float16), (64, 2, torch.bfloat16), (256, 4, torch.float32)])
def test_paged_forward_rows_of_many_chunks(d, group, qdt):
    """Rows of 66 chunks (33.6K tokens): each of the combine's 32 thread groups
    sums more than one chunk (rows of fewer than 32 chunks, the case of the
    tests above, give each group at most one)."""
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print(f"[gpu] paged forward, 66 chunks per row, d={d} group={group} {qdt}", flush=True)
    kv, base = 1, 500000.0
    comp = NexusQuantKVCompressor(head_dim=d, bits=2, rope_base=base)
    attn = NexusQuantPagedAttention(comp)
    gen = torch.Generator().manual_seed(3 * d + group)
    n_pages = 2100  # x 16 tokens = 33600 = 65.6 chunks of 512
    k = (torch.randn(n_pages, kv, 16, d, generator=gen) * 2).to(torch.float16)
    v = (torch.randn(n_pages, kv, 16, d, generator=gen) * 0.5).to(torch.float16)
    work = [(k[i].to(DEV), v[i].to(DEV), torch.arange(16, dtype=torch.int32) + 16 * i) for i in range(n_pages)]
    cache = dict(enumerate(comp.compress_pages(work)))
    tables = [list(range(n_pages)), list(range(n_pages))[::-1]]
    ctx = [16 * n_pages, 16 * n_pages - 9]
    query = torch.randn(2, kv * group, d, generator=gen).to(qdt)
    out = attn.forward(query.to(DEV), cache, cache, tables, torch.tensor(ctx))
    torch.cuda.synchronize()
    ref = _oracle_forward(cache, query, tables, ctx, base, group)
    _close_fp16(out.float().cpu().numpy(), ref.float().numpy(), bf16=qdt == torch.bfloat16)


def test_paged_forward_at_a_1m_token_context():
    """One row of 1,048,573 tokens in 1024-token pages (2048 chunks, pages larger
    than a chunk): the combine's groups each sum 64 chunks."""
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print("[gpu] paged forward, 1M-token context", flush=True)
    kv, d, base, group, size, n_pages = 1, 128, 500000.0, 8, 1024, 1024
    comp = NexusQuantKVCompressor(head_dim=d, bits=2, rope_base=base)
    attn = NexusQuantPagedAttention(comp)
    gen = torch.Generator().manual_seed(5)
    work = []
    for i in range(n_pages):
        k = (torch.randn(kv, size, d, generator=gen) * 2).to(torch.float16)
        v = (torch.randn(kv, size, d, generator=gen) * 0.5).to(torch.float16)
        work.append((k.to(DEV), v.to(DEV), torch.arange(size, dtype=torch.int32) + size * i))
    cache = dict(enumerate(comp.compress_pages(work)))
    del work
    tables = [list(range(n_pages))]
    ctx = [size * n_pages - 3]
    query = torch.randn(1, kv * group, d, generator=gen).half()
    out = attn.forward(query.to(DEV), cache, cache, tables, torch.tensor(ctx))
    torch.cuda.synchronize()
    ref = _oracle_forward(cache, query, tables, ctx, base, group)
    _close_fp16(out.float().cpu().numpy(), ref.float().numpy())


def test_paged_plan_reuse_across_queries():
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print("[gpu] paged plan reuse", flush=True)
    comp = NexusQuantKVCompressor(head_dim=64, bits=4, rope_base=10000.0)
    attn = NexusQuantPagedAttention(comp)
    gen = torch.Generator().manual_seed(3)
    work = [(torch.randn(4, 16, 64, generator=gen).half().to(DEV), torch.randn(4, 16, 64, generator=gen).half().to(DEV),
             torch.arange(16, dtype=torch.int32) + 16 * i) for i in range(40)]
    cache = dict(enumerate(comp.compress_pages(work)))
    tables = [list(range(40)), list(range(20, 40))]
    plan = attn.plan(cache, tables, [640, 300])
    for step in range(3):
        q = torch.randn(2, 4, 64, generator=gen).half()
        out = attn.run(plan, q.to(DEV))
        ref = _oracle_forward(cache, q, tables, [640, 300], 10000.0, 1)
        _close_fp16(out.cpu().numpy(), ref.numpy())


def test_compress_and_cache_follows_reference_semantics():
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print("[gpu] compress_and_cache", flush=True)
    comp = NexusQuantKVCompressor(head_dim=128, bits=2, rope_base=10000.0)
    attn = NexusQuantPagedAttention(comp)
    gen = torch.Generator().manual_seed(8)
    key = torch.randn(10, 4, 128, generator=gen).half()
    value = torch.randn(10, 4, 128, generator=gen).half()
    slots = torch.tensor([32, 33, 34, 35, 36, 37, 64, 65, 66, 9])
    kcache, vcache = {}, {}
    attn.compress_and_cache(key.to(DEV), value.to(DEV), kcache, vcache, slots.to(DEV))
    # the reference's block-size heuristic returns 4: blocks slot // 4, positions slot % 4
    assert attn._infer_block_size(slots) == 4
    assert sorted(kcache) == [2, 8, 9, 16] and kcache is not vcache and kcache[8] is vcache[8]
    for bid, page in kcache.items():
        idx = [i for i, sl in enumerate(slots.tolist()) if sl // 4 == bid]
        pos = torch.tensor([slots[i].item() % 4 for i in idx], dtype=torch.int32)
        kc, vc, ks, vs = T.vllm_compress_page(key[idx].permute(1, 0, 2), value[idx].permute(1, 0, 2), pos, 2, 10000.0)
        assert torch.equal(page.positions.cpu(), pos)
        mism = (page.key_codes.cpu().reshape(-1, 8) != kc.reshape(-1, 8)).any(1).float().mean().item()
        assert mism <= 2e-2


@pytest.mark.parametrize("d,group,qdt", [(64, 8, torch.float16), (128, 8, torch.float16), (128, 1, torch.bfloat16),
                                         (128, 4, torch.float32), (256, 2, torch.float32), (256, 4, torch.bfloat16)])
@pytest.mark.parametrize("ctx", [1, 15, 17, 63, 65, 128, 129, 1000])
def test_paged_forward_short_contexts_and_table_kinds(d, group, qdt, ctx):
    """Contexts around a unit (16 tokens) and the shortest chunk (64), where some of a
    workgroup's waves have no unit: against float64 attention over the decoded pages,
    and the same bits from cos / sin tables as from the merged ones."""
    from nexusquant_amd.vllm_backend import CompressedPage, NexusQuantKVCompressor, NexusQuantPagedAttention
    print(f"[gpu] short context d={d} group={group} {qdt} ctx={ctx}", flush=True)
    kv, block = 2, 16
    g = torch.Generator(device=DEV).manual_seed(d + group + ctx)
    comp = NexusQuantKVCompressor(head_dim=d, bits=3, rope_base=10000.0)
    attn = NexusQuantPagedAttention(comp)
    n_pages = -(-ctx // block)
    cache = {}
    for i in range(n_pages):
        k = torch.randn(kv, block, d, device=DEV, generator=g).half()
        v = (torch.randn(kv, block, d, device=DEV, generator=g) * 0.5).half()
        cache[i] = comp.compress_page(k, v, torch.arange(i * block, (i + 1) * block, dtype=torch.int32) + 70000)
    q = torch.randn(1, kv * group, d, device=DEV, generator=g).to(qdt)
    plan = attn.plan(cache, [list(range(n_pages))], [ctx])
    got = attn.run(plan, q)
    tables = comp._tables
    comp._tables = lambda m, dev: tables(m, dev)[:2] + (None, None)
    assert torch.equal(attn.run(plan, q), got)
    comp._tables = tables
    dec = comp.decompress_pages([cache[i] for i in range(n_pages)])
    k = torch.cat([p[0] for p in dec], 1)[:, :ctx].double()
    v = torch.cat([p[1] for p in dec], 1)[:, :ctx].double()
    want = torch.empty(1, kv * group, d, dtype=torch.float64, device=DEV)
    for h in range(kv * group):
        w = torch.softmax(k[h // group] @ q[0, h].double() / math.sqrt(d), 0)
        want[0, h] = w @ v[h // group]
    # _close_fp16's bounds are for a reference rounded as the op rounds: to fp16, then the
    # query's type (an unrounded one alone is up to 2^-8 from a bf16 output)
    want = want.half().to(qdt)
    _close_fp16(got.float().cpu().numpy(), want.float().cpu().numpy(), bf16=qdt == torch.bfloat16)


def test_compress_pages_takes_positions_of_any_kind():
    """Host positions of all pages travel in one copy: lists, int64 and float tensors and
    device tensors, mixed in one call, give the pages that single calls give."""
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor
    comp = NexusQuantKVCompressor(head_dim=64, bits=2)
    g = torch.Generator(device=DEV).manual_seed(3)
    kinds = [list(range(5, 12)), torch.arange(7), torch.arange(100, 107, dtype=torch.int32, device=DEV),
             torch.arange(7, dtype=torch.float32) + 30.5, torch.arange(9000, 9007, dtype=torch.int32)]
    work = [(torch.randn(3, 7, 64, device=DEV, generator=g).half(), torch.randn(3, 7, 64, device=DEV, generator=g).half(), p)
            for p in kinds]
    for many, w in zip(comp.compress_pages(work), work):
        one = comp.compress_page(*w)
        want = torch.as_tensor(w[2]).to(torch.int32)
        assert torch.equal(many.positions.cpu(), want.cpu()) and many.max_position == int(want.max())
        for name in ("key_codes", "value_codes", "key_scales", "value_scales", "positions"):
            assert torch.equal(getattr(many, name), getattr(one, name)), name
    with pytest.raises(ValueError, match="non-negative"):
        comp.compress_pages([(work[0][0], work[0][1], torch.arange(-1, 6))])


@pytest.mark.parametrize("d,group,qdt", [(64, 8, torch.float16), (128, 8, torch.float16), (128, 4, torch.float16),
                                         (256, 1, torch.float16), (64, 4, torch.bfloat16), (128, 4, torch.bfloat16),
                                         (256, 2, torch.bfloat16), (64, 1, torch.float32), (128, 2, torch.float32),
                                         (256, 4, torch.float32)])
def test_paged_forward_takes_the_page_decoders_keys(d, group, qdt):
    """The keys of decode attention are the fp16 keys that decompress_pages returns.

    Queries orthogonal to a row's keys and 2000 long per coordinate: the logits are what
    the keys' rounding leaves, times 2000 (a key rounded elsewhere moves a logit by 0.2)."""
    from nexusquant_amd.vllm_backend import CompressedPage, NexusQuantKVCompressor, NexusQuantPagedAttention
    print(f"[gpu] decoder's keys d={d} group={group} {qdt}", flush=True)
    kv, n = 2, 15
    g = torch.Generator(device=DEV).manual_seed(d + group)
    comp = NexusQuantKVCompressor(head_dim=d, bits=3, rope_base=10000.0)
    attn = NexusQuantPagedAttention(comp)
    page = comp.compress_page(torch.randn(kv, n, d, device=DEV, generator=g).half(),
                              torch.randn(kv, n, d, device=DEV, generator=g).half(),
                              torch.arange(n, dtype=torch.int32) + 5000)
    k, v = (t.double() for t in comp.decompress_pages([page])[0])
    q = torch.empty(1, kv * group, d, dtype=torch.float64, device=DEV)
    for h in range(kv * group):
        x = torch.randn(d, dtype=torch.float64, device=DEV, generator=g)
        basis = torch.linalg.qr(k[h // group].T.cpu())[0].to(DEV)
        q[0, h] = 2000 * (x - basis @ (basis.T @ x))
    q = q.to(qdt)
    got = attn.forward(q, {0: page}, {0: page}, [[0]], torch.tensor([n]))
    for h in range(kv * group):
        kh, qh = k[h // group], q[0, h].double()
        want = torch.softmax(kh @ qh / math.sqrt(d), 0) @ v[h // group]
        # fp32 sums of d exact products, rounded at random: 4 sqrt(d) 2^-24 of the products' sum
        # in a logit, as much relatively in a weight; the output rounded to fp16 and to the query's type
        logit = 4 * math.sqrt(d) * 2.0 ** -24 * float((kh.abs() @ qh.abs()).max()) / math.sqrt(d)
        tol = logit + (2.0 ** -8 if qdt == torch.bfloat16 else 2.0 ** -10)
        err = float((got[0, h].double() - want).norm() / want.norm())
        assert err <= tol, (h, err, tol)


@pytest.mark.parametrize("d,group,qdt", [(128, 4, torch.float16), (128, 4, torch.bfloat16), (64, 2, torch.float32)])
def test_paged_forward_row_alone_and_in_a_batch(d, group, qdt):
    """A row planned alone is cut at 64 tokens, among long rows at 512: the outputs agree to
    one rounding of the output."""
    from nexusquant_amd.vllm_backend import NexusQuantKVCompressor, NexusQuantPagedAttention
    print(f"[gpu] row alone and in a batch d={d} group={group} {qdt}", flush=True)
    kv, size = 2, 1024
    g = torch.Generator(device=DEV).manual_seed(d + group)
    comp = NexusQuantKVCompressor(head_dim=d, bits=3, rope_base=500000.0)
    attn = NexusQuantPagedAttention(comp)
    work = [(torch.randn(kv, size, d, device=DEV, generator=g).half(), torch.randn(kv, size, d, device=DEV, generator=g).half(),
             torch.arange(size, dtype=torch.int32) + size * i) for i in range(4)]
    cache = dict(enumerate(comp.compress_pages(work)))
    tables = [[0, 1]] + [[0, 1, 2, 3]] * 32
    ctx = [1500] + [4096] * 32
    q = torch.randn(33, kv * group, d, device=DEV, generator=g).to(qdt)
    alone, batch = attn.plan(cache, tables[:1], ctx[:1]), attn.plan(cache, tables, ctx)
    assert alone.n_chunks == -(-1500 // 64) and batch.n_chunks == 3 + 32 * 8
    a, b = attn.run(alone, q[:1])[0].double(), attn.run(batch, q)[0].double()
    # weights: x and the chunk's max are rounded to 2^-24 and differ by less than 2^4, exp to a
    # few ulp: 2^-18 of a weight; the output's rounding to fp16 (2^-11) and bf16 (2^-9) may fall
    # either way
    vmax = max(float(p[1].abs().max()) for p in comp.decompress_pages(list(cache.values())))
    ulp = 2.0 ** -8 + 2.0 ** -10 if qdt == torch.bfloat16 else 2.0 ** -10
    assert bool(((a - b).abs() <= ulp * a.abs() + 2.0 ** -17 * vmax).all())
