"""nq_score_keykey where its launch shape changes: tiles per wave, and the separate
combination of the splits' softmax statistics from 32 splits (16384 keys) on."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("b,h,s,d,dt,obs", [
    (1, 8, 31, 128, torch.float16, 32), (1, 2, 129, 64, torch.bfloat16, 32), (1, 8, 8160, 128, torch.bfloat16, 32),
    (1, 1, 8193, 96, torch.float16, 7), (1, 3, 15872, 128, torch.float16, 32), (1, 3, 15873, 128, torch.bfloat16, 40),
    (2, 2, 16385, 256, torch.float32, 64), (4, 1, 40001, 64, torch.float16, 32), (1, 9, 17000, 128, torch.bfloat16, 1),
])
def test_keykey_grid_edges_match_float64(b, h, s, d, dt, obs):
    from nexusquant_amd.ops import score_keykey
    print(f"[gpu] keykey {(b, h, s, d)} {dt} obs={obs}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(s)
    k = torch.randn(b, h, s, d, device=DEV, generator=g).to(dt)
    k[..., 3] *= 6
    got = score_keykey(k, obs).double()
    want = torch.zeros(b, s, dtype=torch.float64, device=DEV)
    n = min(obs, s)
    for i in range(b):
        for j in range(h):
            x = k[i, j].double()
            want[i] += torch.softmax(x[-n:] @ x.t().contiguous() * d ** -0.5, -1).sum(0) / h
    # logits are fp32 sums of d exact products (error a few 2^-24 of sum |q k| <= 40 here), so
    # exp(x) is within about 2e-5 of its value
    assert torch.all((got - want).abs() <= 2e-5 * want + 1e-9)
