"""Decode attention at the edges of its launch rules (csrc/attention.hip): key splits and waves per block over the number of (sequence, kv head) groups."""
import numpy as np
import pytest
import torch

from tgis_amd import native
from oracle import ops_ref


@pytest.mark.parametrize("B,Hkv,ctx,splits", [
    (8, 32, 96, 1), (8, 32, 8192, 1), (255, 1, 8192, 1), (9, 32, 1504, 1), (9, 32, 1505, 2), (12, 32, 4096, 2), (13, 32, 4096, 1), (32, 12, 1505, 2), (16, 32, 4096, 1),
    (4, 32, 4096, 2), (64, 32, 4096, 1),
])
def test_splits(B, Hkv, ctx, splits):
    lib = native.load_library()
    assert lib.tgis_attn_num_splits(B, Hkv, Hkv, 1, ctx) == splits
    assert lib.tgis_attn_num_splits(B, Hkv, 8 * Hkv, 1, ctx) == splits  # up to 16 q heads of a kv head are one chunk


@pytest.mark.parametrize("B,Hkv,D,ctx,waves", [
    (255, 1, 128, 33, 8), (8, 32, 128, 33, 4), (8, 32, 64, 128, 4), (8, 32, 128, 129, 8), (128, 2, 64, 129, 8), (32, 4, 128, 4096, 8), (257, 1, 128, 4096, 4), (512, 1, 64, 224, 4), (512, 1, 64, 225, 8), (513, 1, 64, 4096, 4), (769, 1, 128, 4096, 4), (800, 1, 128, 4096, 4),
    (895, 1, 128, 4096, 4), (896, 1, 128, 352, 4), (896, 1, 128, 353, 8), (1023, 1, 128, 353, 8), (1023, 1, 128, 200, 4), (1024, 1, 128, 353, 2), (896, 1, 64, 4096, 4), (1536, 1, 128, 4096, 2),
    (1537, 1, 128, 352, 2), (1537, 1, 128, 353, 8), (2047, 1, 128, 353, 8), (2047, 1, 128, 130, 2), (2047, 1, 64, 353, 2), (2048, 1, 128, 353, 4),
])
def test_waves(B, Hkv, D, ctx, waves):
    assert native.load_library().tgis_attn_decode_waves(B, Hkv, Hkv, D, ctx) == waves


# B x Hkv groups: 8 waves up to 256 (256 of up to 4 pages: 4); 4 (D 64 from 8 pages on: 8) up to 511, two splits from 48 pages on up to 384; D 128 from 12 pages on 8 at 896 - 1023 and 1537 - 2047,
# between and D 64 2
@pytest.mark.gpu
@pytest.mark.parametrize("B,Hkv,G,D,longest", [
    (128, 2, 1, 128, 128), (128, 2, 4, 64, 129), (128, 2, 1, 128, 300), (257, 1, 2, 128, 300), (96, 4, 1, 128, 1505), (97, 4, 1, 128, 1505), (511, 1, 1, 64, 225), (512, 1, 1, 64, 225), (513, 1, 1, 64, 225), (511, 1, 1, 64, 224), (128, 3, 4, 64, 1504),
    (128, 3, 4, 64, 1505), (769, 1, 1, 128, 130), (1023, 1, 1, 128, 130), (1024, 1, 1, 128, 130), (1537, 1, 1, 128, 70), (1537, 1, 1, 64, 70), (2047, 1, 1, 128, 33),
    (896, 1, 1, 128, 353), (1023, 1, 1, 128, 353), (1537, 1, 1, 128, 353), (2047, 1, 1, 128, 353),
])
def test_groups(gpu_device, B, Hkv, G, D, longest):
    """Ragged sequences, among them one token, whole pages and one longest, against attention in float32."""
    dtype, H = torch.bfloat16 if D == 64 else torch.float16, Hkv * G
    lens = [1, 32, 31, longest] + [1 + (i * 37) % min(longest, 90) for i in range(B - 4)]
    g = torch.Generator().manual_seed(B + D)
    pages = [(n + 31) // 32 for n in lens]
    tables = torch.zeros((B, max(pages)), dtype=torch.int32)
    perm, at = torch.randperm(sum(pages), generator=g).int(), 0
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    T = sum(lens)
    kv = torch.randn(T, 2 * Hkv * D, generator=g).to(dtype)
    rows = torch.zeros((T, (H + 2 * Hkv) * D), dtype=dtype)
    rows[:, H * D:] = kv
    slots = torch.cat([tables[b, torch.arange(n) // 32].long() * 32 + torch.arange(n) % 32 for b, n in enumerate(lens)]).int()
    pools = [torch.zeros((sum(pages), Hkv, 32 * D), dtype=dtype, device=gpu_device) for _ in range(2)]
    native.rope_kv_write(rows.to(gpu_device), None, None, None, slots.to(gpu_device), *pools, H, Hkv, D, D)
    q = torch.randn(B, H * D, generator=g).to(dtype)
    want = ops_ref.attention_varlen(q.view(B, H, D), kv[:, :Hkv * D].view(T, Hkv, D), kv[:, Hkv * D:].view(T, Hkv, D), torch.arange(B + 1),
                                    [0] + list(np.cumsum(lens)), D ** -0.5)
    splits = native.attn_num_splits(B, Hkv, H, 1, longest)
    ws = native.Workspace(native.attn_workspace_bytes(B, H, Hkv, D, splits), gpu_device)
    out = torch.full((B, H * D), float("nan"), dtype=dtype, device=gpu_device)
    native.attn_paged(q.to(gpu_device), H * D, *pools, tables.to(gpu_device), torch.tensor(lens, dtype=torch.int32, device=gpu_device),
                      torch.arange(B + 1, dtype=torch.int32, device=gpu_device), out, B, H, Hkv, D, 1, longest, D ** -0.5, splits, ws)
    got, want = out.view(B, H, D).float().cpu(), want.float().cpu()
    # P and the output are rounded to the type once each: half an ulp of values of about 1, with room for both
    unit = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    assert (got - want).abs().max() <= 4 * unit * want.abs().max()
    assert (got - want).norm() <= 2 * unit * want.norm()
