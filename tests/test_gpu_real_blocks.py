"""The real scorer's column sums per block of 128 queries: how they are added up
(one launch for few blocks, separate kernels, several rounds when the blocks'
sums exceed their workspace), against float64 and between the two entry points."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(b, hq, hkv, s, d, dt):
    g = torch.Generator(device=DEV).manual_seed(s + d)
    return [torch.randn(b, h, s, d, device=DEV, generator=g).to(dt) for h in (hq, hkv, hkv)]


def _both(q, k, v, **kw):
    from nexusquant_amd.scoring import attention_real, score_real_accumulate
    sc = q.shape[-1] ** -0.5
    a, b = (torch.zeros(q.shape[0], q.shape[2], device=DEV) for _ in range(2))
    out = attention_real(q, k, v, sc, a, **kw)
    assert torch.equal(out.isnan(), attention_real(q, k, v, sc, **kw).isnan())
    score_real_accumulate(q, k, b, sc, **kw)
    return a, b


@pytest.mark.parametrize("b,hq,hkv,s,d,dt,window", [
    (1, 8, 2, 31, 64, torch.float16, None), (2, 3, 3, 128, 128, torch.bfloat16, None),
    (1, 17, 1, 129, 64, torch.float16, None), (1, 8, 4, 2048, 128, torch.float16, None),
    (1, 8, 4, 2049, 128, torch.float16, None), (2, 4, 2, 3001, 64, torch.bfloat16, 1793),
    (2, 4, 2, 3001, 64, torch.bfloat16, 1791), (1, 4, 4, 1000, 128, torch.float16, 1),
    (1, 4, 4, 1000, 128, torch.bfloat16, 65),
])
def test_block_sums_match_float64(b, hq, hkv, s, d, dt, window):
    print(f"[gpu] block sums {(b, hq, hkv, s, d)} {dt} window={window}", flush=True)
    q, k, v = _inputs(b, hq, hkv, s, d, dt)
    imp, imp2 = _both(q, k, v, sliding_window=window)
    assert torch.equal(imp, imp2)
    i = torch.arange(s, device=DEV)
    hidden = (i[None, :] > i[:, None]) | (i[None, :] <= i[:, None] - (window or s))
    want = torch.zeros(b, s, dtype=torch.float64, device=DEV)
    for r in range(b):
        for h in range(hq):
            w = q[r, h].float() @ k[r, h * hkv // hq].float().t().contiguous()
            w = (w.to(dt).float() * d ** -0.5).to(dt).double().masked_fill(hidden, float("-inf"))
            want[r] += torch.softmax(w, -1).float().to(dt).double().sum(0) / hq
    # the probabilities agree but where an fp32 logit or probability lies at a rounding
    # boundary of the model dtype: 2^-11 (fp16) or 2^-8 (bf16) of single terms
    eps = 2.0 ** (-11 if dt == torch.float16 else -8)
    assert torch.all((imp.double() - want).abs() <= eps * want + 1e-6)


def test_rounds_of_blocks_equal_one_round():
    # 32 heads x 12289 keys: 97 blocks' sums are 153 MB, more than one round holds;
    # the heads' shares are the same when four heads fit at once
    from nexusquant_amd.scoring import score_real_accumulate
    q, k, v = _inputs(1, 32, 1, 12289, 64, torch.float16)
    imp, imp2 = _both(q, k, v)
    assert torch.equal(imp, imp2)
    parts = torch.zeros(1, 12289, dtype=torch.float64, device=DEV)
    for h in range(0, 32, 4):
        p = torch.zeros(1, 12289, device=DEV)
        score_real_accumulate(q[:, h:h + 4].contiguous(), k, p, 64 ** -0.5)
        parts += p.double() / 8
    # fp32 sums over 32 heads in another grouping: 64 roundings of at most 2^-24
    assert torch.all((imp.double() - parts).abs() <= 64 * 2.0 ** -24 * parts)


@pytest.mark.parametrize("s,at", [(300, 70), (300, 299), (2500, 130)])
def test_nan_query_reaches_only_its_block(s, at):
    q, k, v = _inputs(1, 2, 2, s, 128, torch.float16)
    q[0, 1, at] = float("nan")
    imp, imp2 = _both(q, k, v)
    assert torch.equal(imp.isnan(), imp2.isnan())
    assert imp[0, :at + 1].isnan().all() and imp[0, (at | 31) + 1:].isfinite().all()


@pytest.mark.parametrize("s,at,window", [(300, 70, None), (300, 299, None), (2500, 130, None), (300, 37, None),
                                         (300, 38, 20), (700, 390, 33), (700, 389, 100), (2500, 1999, 1000), (300, 5, 1)])
@pytest.mark.parametrize("d", [64, 128])
def test_nan_query_reaches_the_keys_it_sees_and_their_partners(s, at, window, d):
    """Exactly the keys that the query sees, and key ^ 16 of each: the two share a row of
    the MFMA that sums the columns."""
    q, k, v = _inputs(1, 2, 2, s, d, torch.float16)
    q[0, 1, at] = float("nan")
    imp, imp2 = _both(q, k, v, sliding_window=window)
    want = torch.zeros(s + 32, dtype=torch.bool, device=DEV)
    seen = torch.arange(max(0, at - (window or s) + 1), at + 1, device=DEV)
    want[seen] = True
    want[seen ^ 16] = True
    assert torch.equal(imp[0].isnan(), want[:s]) and torch.equal(imp2[0].isnan(), want[:s])


@pytest.mark.parametrize("hq,s,d,window", [(1, 40000, 64, None), (2, 33001, 64, 700), (1, 262209, 64, 300)])
def test_long_rows_share_blocks_and_take_turns(hq, s, d, window):
    """Few heads and many keys: a block's stages are shared by several workgroups (scores
    alone), sums of later launches are added, and past 262144 keys a causal output and its
    sums take passes of their own (with a window they do not)."""
    print(f"[gpu] long rows {hq} x {s} x {d} window={window}", flush=True)
    q, k, v = _inputs(1, hq, 1, s, d, torch.float16)
    imp, imp2 = _both(q, k, v, sliding_window=window)
    assert torch.equal(imp, imp2)
    # every row of P sums to 1: fp16 probabilities, each off by at most 2^-11 of itself or
    # half a subnormal step, 2^-25
    total, most = float(imp.double().sum()), window or s
    assert abs(total - s) <= s * (2.0 ** -11 + min(most, s) * 2.0 ** -25)


def test_calls_without_block_sums_hold_no_memory_for_them():
    """fp32 scores and attention without importance: 12 bytes per query row (and V transposed)."""
    from nexusquant_amd import ops
    from nexusquant_amd.scoring import attention_real, score_real_accumulate
    q, k, v = _inputs(1, 4, 2, 3000, 64, torch.float16)
    for call, most in ((lambda: score_real_accumulate(q.float(), k.float(), torch.zeros(1, 3000, device=DEV), 0.125),
                        12 * 4 * 3000 + 256),
                       (lambda: attention_real(q, k, v, 0.125), 12 * 4 * 3000 + 256 + 2 * 64 * 3008 * 2)):
        ops.release_workspaces()
        call()
        # the cached workspace is rounded up to 1 MiB; the blocks' sums would take 1.1 more
        assert sum(t.numel() for t in ops._workspaces.values()) == -(-most // (1 << 20)) << 20
    ops.release_workspaces()
