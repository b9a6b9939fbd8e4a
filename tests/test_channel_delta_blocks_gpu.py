"""The delta rule with a decay per key channel in blocks of 64 tokens on the matrix cores (bfloat16 models; hip_only)."""
import pytest
import torch

from test_kirisun import _delta_inputs, _delta_weights, _kernels, _new_states, _run_delta


def _states64(shape, w, inputs, S):
    """The states after a portion, in float64: S [heads, dim, vdim] before it; the convolution starts from zeros."""
    heads, kv_heads, dim, vdim, taps = shape
    proj, decay_in = inputs[0].double(), inputs[1].double()
    T, qk, vv = proj.shape[0], kv_heads * dim, heads * vdim
    raw = torch.cat((torch.zeros((taps - 1, 2 * qk + vv), dtype=torch.float64), proj[:, :2 * qk + vv]))
    c = sum(raw[j:j + T] * w["conv"][:, j].double() for j in range(taps))
    c = c * torch.sigmoid(c)
    k = c[:, qk:2 * qk].reshape(T, kv_heads, dim)
    k = (k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // kv_heads, 1)
    v, beta = c[:, 2 * qk:].reshape(T, heads, vdim), torch.sigmoid(proj[:, 2 * qk + vv:])
    step = torch.nn.functional.softplus(decay_in + w["dt_bias"].double(), threshold=1e9).reshape(T, heads, dim)
    a = torch.exp(-torch.exp(w["A_log"].double())[None, :, None] * step)
    for t in range(T):
        S = a[t][:, :, None] * S
        S = S + k[t][:, :, None] * (beta[t][:, None] * (v[t] - torch.einsum("hdv,hd->hv", S, k[t])))[:, None, :]
    return S


# what every third channel's decay input is moved by: nothing; to next to no decay beside decays of e^-12 a token; to decays
# whose logarithm is past float's exponents
@pytest.mark.gpu
@pytest.mark.parametrize("strong", [0.0, 12.0, 3e3, float("inf")])
@pytest.mark.parametrize("shape", [(4, 2, 12, 8, 3), (2, 2, 64, 64, 4), (3, 1, 30, 18, 1), (2, 1, 128, 128, 4), (1, 1, 98, 33, 2)])
def test_portions_at_the_edges_of_blocks_and_every_strength_of_decay(shape, strong):
    k, dev = _kernels("hip", torch.bfloat16)
    heads, kv_heads, dim, vdim, taps = shape
    w = _delta_weights(shape, 3, torch.bfloat16, slow=0)
    w["dt_bias"][:] = -2.0
    lens = [1, 63, 64, 65, 81, 130, 3]
    inputs = [_delta_inputs(shape, n, 60 + i, torch.bfloat16) for i, n in enumerate(lens)]
    for x in inputs:
        x[1][:, ::3] += strong
        x[1][1::2, 1::3] += min(strong, 40.0)
    part = tuple(torch.cat([x[i] for x in inputs]) for i in range(3))
    slots, found = [3, 0, 5, 1, 2, 6, 4], {}
    rule, k.channel_block_rule = k.channel_block_rule, (0, 100.0)
    try:
        for blocks in (True, False):
            k.delta_blocks = blocks
            states = _new_states(dev, 8, shape)
            found[blocks] = (_run_delta(k, dev, shape, w, part, 1e-5, states, lens, [0] * 7, slots), *states)
            # a second portion, from the states
            again = _run_delta(k, dev, shape, w, tuple(t[:70] for t in part), 1e-5, states, [70], [9], [6])
            found[blocks] += (again, states[1][6].clone())
            assert torch.isnan(states[1][7]).all()
    finally:
        k.delta_blocks, k.channel_block_rule = True, rule
    for i in (1,) if taps > 1 else ():
        assert torch.equal(found[True][i][:7], found[False][i][:7])
    # both ways' errors are some roundings of 2^-24 of a state's largest number a token; the blocks' is at most twice the
    # other's and one such rounding over the longest portion
    for s, (n, slot) in enumerate(zip(lens, slots)):
        if slot == 6:
            continue                    # (the second portion's)
        want = _states64(shape, w, inputs[s], torch.zeros((heads, dim, vdim), dtype=torch.float64))
        top = want.abs().max().item()
        errors = {b: (found[b][2][slot].cpu().double() - want).abs().max().item() / top for b in (True, False)}
        print(shape, strong, n, errors)
        assert errors[True] <= 2 * errors[False] + 16 * 2.0 ** -24, (n, errors)
    for i in (0, 3):
        got, one = found[True][i].float(), found[False][i].float()
        assert (got - one).abs().max() <= 2.0 ** -7 * one.abs().max()       # one rounding of bfloat16 each, at the largest
    top = found[False][4].abs().max()
    assert (found[True][4] - found[False][4]).abs().max() <= 2e-5 * top


def test_which_steps_run_in_blocks():
    from types import SimpleNamespace

    from nano_vllm_amd.kernels.ops import HipKernels
    k = SimpleNamespace(delta_blocks=True)
    for lens, first, want in (([256], 0, 0), ([300], 0, 5), ([257], 0, 0), ([1, 1, 300], 2, 5), ([1, 1, 300], 1, 0), ([512, 40, 40, 40], 0, 11),
                              ([300] + [80] * 3, 0, 0), ([1, 300, 2], 1, 0), ([1] * 9, 9, 0), ([640, 1], 0, 0 if 64 * 11 > 1.2 * 641 else 11)):
        batch = SimpleNamespace(q_lens=lens)
        got = HipKernels._delta_plan(k, batch, first, "cpu", lambda n: 8 * n, 256, 1.2)
        assert got[0] == want, lens
        if want:
            assert got[1] == len(lens) - first and got[4].numel() == 8 * want
    assert HipKernels._delta_plan(k, SimpleNamespace(q_lens=[300]), 0, "cpu", lambda n: 0, 256, 1.2)[0] == 0
