"""Owner launches of one 16-column block that the split kernel does not take,
and so run on the partition kernel: more sequences than a grid dimension has
(4-wave workgroups), and, through the C entry point, a window call with fewer
slots than its window needs, which attends to the tiles it has (8-wave
workgroups for few pairs)."""

from __future__ import annotations

import math

import pytest
import torch

from flydsl_amd import pa_decode_ps_launch, prepare_pa_decode
from tests._cases import make_case
from tests.test_gpu_parity import assert_parity, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def fp8(gen, *shape):
    """Bytes of finite e4m3fn values up to 15 in magnitude."""
    x = torch.randint(0, 112, shape, generator=gen, device=DEV, dtype=torch.uint8)
    return (x | (torch.randint(0, 2, shape, generator=gen, device=DEV, dtype=torch.uint8) << 7)).view(torch.float8_e4m3fn)


def test_more_sequences_than_a_grid_dimension():
    B, gqa = 65536 + 37, 3
    gen = torch.Generator(device=DEV).manual_seed(2)
    kc, vc = fp8(gen, B, 1, 8, 16, 16), fp8(gen, B, 1, 1, 128, 16)
    q = torch.randn(B, gqa, 128, generator=gen, device=DEV).to(torch.bfloat16)
    table = torch.randperm(B, generator=gen, device=DEV).to(torch.int32).view(B, 1)
    lens = torch.randint(1, 17, (B,), generator=gen, device=DEV, dtype=torch.int32)
    one = torch.full((1,), 0.1, device=DEV)
    out = torch.empty_like(q)
    pa_decode_ps_launch(out, q, kc, vc, lens, None, None, 0.088, one, one, block_tables=table)
    for b0 in range(0, B, 16384):
        pages = table[b0:b0 + 16384, 0].long()
        k = kc[pages].float().permute(0, 3, 1, 2, 4).reshape(-1, 16, 128) * 0.1
        v = vc[pages].float().reshape(-1, 128, 16).transpose(1, 2) * 0.1
        qb = q[b0:b0 + 16384].float()
        hide = torch.arange(16, device=DEV)[None] >= lens[b0:b0 + 16384, None]
        ref = torch.empty_like(qb)
        for h in range(gqa):
            x = ((qb[:, h, None] * k).sum(-1) * 0.088).masked_fill(hide, -math.inf)
            ref[:, h] = (torch.softmax(x, -1)[..., None] * v).sum(1)
        assert_parity(out[b0:b0 + 16384], ref.cpu().to(torch.bfloat16), f"from sequence {b0}")


@pytest.mark.parametrize("batch", [3, 140])
def test_window_with_fewer_slots_than_it_needs(batch):
    window, slots = 400, 2  # needs three tiles of 256 tokens
    case = to_dev(make_case(batch=batch, ctx_range=(1, 1500), sliding_window=window, seed=batch))
    out = torch.empty_like(case["query"])
    call = prepare_pa_decode(out, case["query"], case["key_cache"], case["value_cache"], case["context_lengths"], None,
                             None, case["softmax_scale"], case["key_scale"], case["value_scale"],
                             sliding_window=window, block_tables=case["block_tables"])
    assert call._pa is not None and call._pa.num_partitions == 3
    call._pa.num_partitions = call._pa.slots_per_workgroup = slots
    call.launch()
    ref = torch.empty(case["query"].shape)
    for b, n in enumerate(case["context_lengths"].tolist()):
        lo = max(0, n - 1 - window)
        hi = min(n, (lo // 256 + slots) * 256)
        pages = case["block_tables"][b, :-(-n // 16)].long()
        k = case["key_cache"][pages].float().permute(1, 0, 3, 2, 4).reshape(2, -1, 128)[:, lo:hi].cpu()
        v = case["value_cache"][pages].float().permute(1, 0, 2, 4, 3).reshape(2, -1, 128)[:, lo:hi].cpu()
        k, v = k * float(case["key_scale"][0]), v * float(case["value_scale"][0])
        qb = case["query"][b].float().cpu().reshape(2, 4, 128)
        p = torch.softmax(torch.matmul(qb, k.transpose(1, 2)) * case["softmax_scale"], -1)
        ref[b] = torch.matmul(p, v).reshape(8, 128)
    assert_parity(out, ref.to(torch.bfloat16), f"{slots} of 3 slots")
