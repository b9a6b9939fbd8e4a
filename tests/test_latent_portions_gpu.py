"""Attention through a latent for portions of prompts: the kernel of many tokens a workgroup against float64, and against the
kernel of a token a wave, whose arithmetic it repeats (hip only)."""
from types import SimpleNamespace

import pytest
import torch

from test_kirisun import _kernels


# latents below, at and above what the kernel is built for (128, 256, 384, 512 and rotated parts of 64 and 128 entries), fewer
# and more heads than a product's 16 columns, portions at the edges of the workgroups' halves and of the tiles, windows that
# end inside them
@pytest.mark.gpu
@pytest.mark.parametrize("rank,rot,heads,lens,behind,window", [
    (128, 64, 16, [2, 3, 4, 5, 31, 32, 33, 64, 65], [0, 1, 28, 31, 0, 32, 5, 0, 100], 0),
    (144, 24, 3, [70, 8], [0, 57], 0),
    (384, 64, 20, [200, 9], [0, 130], 0),
    (384, 72, 16, [97], [33], 40),
    (256, 128, 16, [130, 36], [0, 300], 200),
    (512, 64, 5, [67, 2], [3, 94], 0),
    (400, 128, 16, [40], [70], 17),
])
def test_portions_of_every_size(rank, rot, heads, lens, behind, window):
    k, dev = _kernels("hip", torch.bfloat16)
    g = torch.Generator().manual_seed(rank + rot)
    width, page, T = rank + rot, 64, sum(lens)
    kv = [a + b for a, b in zip(lens, behind)]
    per = max((n + page - 1) // page for n in kv)
    pages = torch.randperm(len(lens) * per, generator=g).int().reshape(len(lens), per)
    kc = torch.full((len(lens) * per, page, width), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((len(lens) * per, page // 32, rank, 32), float("nan"), dtype=torch.bfloat16)
    q = (torch.randn((T, heads, width), generator=g) * 2).bfloat16()
    sinks, scale = torch.randn(heads, generator=g), width ** -0.5
    want, t = [], 0
    for s, n in enumerate(kv):
        keys = torch.randn((n, width), generator=g).bfloat16()
        for i in range(n):
            kc[pages[s, i // page], i % page] = keys[i]
            vc[pages[s, i // page], i % page // 32, :, i % 32] = keys[i, :rank]
        x = torch.einsum("thc,kc->thk", q[t:t + lens[s]].double(), keys.double()) * scale
        at, of = torch.arange(behind[s], n)[:, None], torch.arange(n)[None, :]
        seen = (of <= at) & ((of > at - window) if window else True)
        x = torch.cat((x.masked_fill(~seen[:, None], float("-inf")), sinks.double()[None, :, None].expand(lens[s], heads, 1)), -1).softmax(-1)
        want.append(torch.einsum("thk,kc->thc", x[..., :-1], keys[:, :rank].double()))
        t += lens[s]
    want = torch.cat(want).reshape(T, -1)
    seq = [s for s, n in enumerate(lens) for _ in range(n)]
    batch = SimpleNamespace(
        num_seqs=len(lens), q_lens=list(lens), num_decode=0, max_kv_len=max(kv), max_q_len=max(lens), starts=list(behind), kv_lens_list=kv,
        groups=[SimpleNamespace(block_tables=pages.to(dev))], token_seq=torch.tensor(seq, dtype=torch.int32, device=dev),
        positions=torch.tensor([b + i for b, n in zip(behind, lens) for i in range(n)], dtype=torch.int32, device=dev),
        cu_seqlens_q=torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=dev),
        kv_lens=torch.tensor(kv, dtype=torch.int32, device=dev))
    args = (q.reshape(T, -1).to(dev), heads, rank, rot, kc.unsqueeze(1).to(dev), vc.unsqueeze(1).to(dev))
    got = k.latent_attention(*args, batch, 0, scale, sinks=sinks.to(dev), window=window or None)
    k.check_faults()
    # weights and outputs of 8 bits: 2^-9 of the largest value each, and as much for the weights' sum
    assert (got.cpu().double() - want).abs().max() <= 3 * 2.0 ** -9 * kc[kc == kc].abs().max().double()
    batch.num_decode = T                                   # every token by itself: one share where it has few keys
    batch.q_lens, k.latent_tiles_per_share = [1] * T, 1 << 20
    try:
        one = k.latent_attention(*args, batch, 0, scale, sinks=sinks.to(dev), window=window or None)
    finally:
        k.latent_tiles_per_share = 0
    assert torch.equal(got, one)
