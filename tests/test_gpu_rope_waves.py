"""The vector RoPE + paged K/V write at the edges of its waves of 64 chunks.

Bit-exact, as the other tests of the write: against the CPU oracle where a
token's chunks end inside a wave, fill it, or divide by one; and, for calls
large enough to take the non-temporal hint, against the same tokens in small
calls.
"""

from __future__ import annotations

import pytest
import torch

from attnarc_amd import ops
from test_gpu_rope import check_case, cos_sin_cache, packed_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("is_neox", [True, False])
@pytest.mark.parametrize("encoding", ["native", "per-head"])
@pytest.mark.parametrize("heads,head_size,rotary", [
    ((5, 3), 80, 80),     # 70 chunks of BF16: a wave and six lanes
    ((1, 1), 64, 16),     # one rotary chunk a head; 16 chunks a token
    ((4, 4), 64, 32),     # exactly one wave of BF16 chunks (interleaved)
    ((33, 1), 128, 128),
    ((2, 2), 256, 64),    # long unrotated tails
])
def test_chunks_of_a_token(dtype, is_neox, encoding, heads, head_size, rotary):
    for tokens in (1, 7):
        check_case(dtype, "HND", encoding, is_neox, T=tokens, Hq=heads[0], Hkv=heads[1], D=head_size, rd=rotary,
                   maxpos=64, NB=4, bs=4, seed=31)


@pytest.mark.parametrize("encoding", ["native", "per-head"])
@pytest.mark.parametrize("is_neox", [True, False])
@pytest.mark.parametrize("tokens", [279, 280, 341, 342, 390, 391])  # NeoX: 24 MiB from 280 (FP8: 342), a workgroup a token
def test_many_chunks_a_token(encoding, is_neox, tokens):
    check_case(torch.bfloat16, "HND", encoding, is_neox, T=tokens, Hq=32 if is_neox else 16, Hkv=32 if is_neox else 24,
               D=256, rd=128, maxpos=512, NB=30, bs=16, seed=41)


@pytest.mark.parametrize("tokens", [1732, 1733])  # 44 MiB from 1,733: a workgroup a token over native caches
def test_native_caches_of_448_chunks(tokens):
    check_case(torch.bfloat16, "NHD", "native", True, T=tokens, Hq=32, Hkv=8, D=128, rd=128, maxpos=512, NB=120, bs=16,
               seed=43)


@pytest.mark.parametrize("dtype,cache,tokens,is_neox", [
    (torch.bfloat16, torch.bfloat16, 8201, True), (torch.float16, torch.uint8, 9001, True),
    (torch.bfloat16, torch.uint8, 9001, False), (torch.float32, torch.float32, 4203, False)])
def test_large_calls_equal_small_ones(dtype, cache, tokens, is_neox):
    # over 192 MiB of rows and cache as one call, a few MiB in pieces of 501 tokens
    hq, hkv, d, bs = 32, 8, 128, 16
    gen = torch.Generator(device=DEV).manual_seed(3)
    packed = torch.randn((tokens, (hq + 2 * hkv) * d), generator=gen, device=DEV).to(dtype)
    pos = torch.randint(0, 512, (tokens,), generator=gen, device=DEV)
    pos[5] = 600  # outside the table: left untouched
    blocks = tokens // bs + 2
    slots = torch.randperm(blocks * bs, generator=gen, device=DEV)[:tokens].contiguous()
    slots[7] = -1
    cs = cos_sin_cache(512, d, dtype)
    ks, vs = (torch.rand(hkv, generator=gen, device=DEV) * 0.1 + 0.01 for _ in range(2))

    def write(pieces):
        rows = packed.clone()
        kv = packed_cache(blocks, bs, hkv, d, cache, "HND")
        q, k, v = (x.unflatten(1, (-1, d)) for x in rows.split((hq * d, hkv * d, hkv * d), dim=1))
        for part in torch.arange(tokens, device=DEV).split(tokens if pieces == 1 else 501):
            a, b = int(part[0]), int(part[-1]) + 1
            ops.rope_paged_kv_write_(q[a:b], k[a:b], v[a:b], pos[a:b].contiguous(), cs, kv, ks, vs,
                                     slots[a:b].contiguous(), is_neox)
        torch.cuda.synchronize()
        return rows, kv

    (rows, kv), (want_rows, want_kv) = write(1), write(0)
    assert torch.equal(rows, want_rows) and torch.equal(kv, want_kv)


@pytest.mark.parametrize("is_neox", [True, False])
@pytest.mark.parametrize("cache_tokens", [0, 1, 6])
def test_value_rows_end_with_the_slots(is_neox, cache_tokens):
    # V rows exist for the tokens that have a slot entry only
    tokens, hq, hkv, d, rd, bs = 9, 12, 2, 64, 32, 4
    gen = torch.Generator(device=DEV).manual_seed(11)
    q0, k0, v = (torch.randn((tokens, h, d), generator=gen, device=DEV).bfloat16() for h in (hq, hkv, hkv))
    pos = torch.randint(0, 64, (tokens,), generator=gen, device=DEV)
    cs = cos_sin_cache(64, rd, torch.bfloat16)
    slots = torch.randperm(6 * bs, generator=gen, device=DEV)[:tokens]

    def write(value, mapping):
        q, k = q0.clone(), k0.clone()
        kc, vc = (torch.full((6, bs, hkv, d), -3.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        ops.rope_paged_kv_write_strided(q, k, value, pos, cs, kc, vc, None, None, mapping, num_blocks=6, block_size=bs,
                                        key_cache_strides=kc.stride()[:3], value_cache_strides=vc.stride()[:3],
                                        is_neox=is_neox)
        torch.cuda.synchronize()
        return q, k, kc, vc

    padded = torch.where(torch.arange(tokens, device=DEV) < cache_tokens, slots, -1)
    want = write(v, padded)
    got = write(v[: max(cache_tokens, 1)].clone(), slots[:cache_tokens].clone() if cache_tokens else None)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
