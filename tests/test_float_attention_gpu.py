"""32-bit attention of prompts' portions with 64 or 128 channels a head, blocks of keys within pages (hip only)."""
import pytest
import torch


# portions at the edges of the tiles of 32 rows and of the blocks of 64 keys, alone and behind keys; scores so far apart that
# weights are zero within whole blocks (boost), sinks, a cap, gates; what unused slots hold is no number
@pytest.mark.gpu
@pytest.mark.parametrize("extras", [False, True])
@pytest.mark.parametrize("scale", [0.1, 30.0])
@pytest.mark.parametrize("hq,hkv,D,page,lens,q_lens", [
    (4, 2, 64, 64, [2, 31, 32, 33, 63, 64, 65, 129], [2, 31, 32, 33, 63, 64, 65, 129]),
    (3, 3, 128, 192, [64, 66, 128, 200, 500], [1, 2, 32, 33, 65]),
    (6, 1, 128, 256, [300, 97], [40, 97]),
    (128, 128, 64, 64, [250, 33], [250, 33]),                # two rows a wave, and (above 1024 tiles and heads) four
])
def test_portions_give_the_bits_of_one_wave_per_token(hq, hkv, D, page, lens, q_lens, scale, extras):
    from nano_vllm_amd.kernels import HipKernels
    from test_kernels_gpu import DEV, _paged_case, _plain_attention
    k = HipKernels(DEV, torch.float32, quiet=True)
    q, kc, vc, batch, parts = _paged_case(torch.float32, hq, hkv, D, page, lens, q_lens, seed=D + page, fill=float("nan"))
    more = {}
    if extras:
        g = torch.Generator().manual_seed(5)
        more = {"sinks": torch.randn(hq, generator=g).to(DEV), "softcap": 7.0, "head_gate": torch.rand((q.shape[0], hq), generator=g).to(DEV)}
    tiled = k.paged_attention(q, hq, hkv, D, kc, vc, batch, 0, scale, None, **more)
    k.tiled_general_attention = False
    per_token = k.paged_attention(q, hq, hkv, D, kc, vc, batch, 0, scale, None, **more)
    k.check_faults()
    assert torch.equal(tiled, per_token) and torch.isfinite(tiled).all()
    if not extras and scale < 1:
        want = _plain_attention(*parts, lens, q_lens, scale, None).to(DEV)
        # (sums of up to 512 terms of 24 bits)
        assert (tiled - want).abs().max() <= 512 * 2.0 ** -24 * want.abs().max()
