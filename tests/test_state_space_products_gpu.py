"""Portions of a bfloat16 state-space layer as products on the matrix cores: sub-blocks of 64 tokens, units of 128 and more,
at their edges and for every height of the state, against the plain recurrence in float64 on the same rounded inputs (the
convolution's output rounded once to bfloat16, as the layer rounds it) and against the token-by-token kernel."""
import pytest
import torch

import test_mafarax as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 64, 32, 1, 4, 1), (4, 64, 64, 2, 8, 2), (2, 128, 128, 1, 2, 1), (16, 64, 128, 8, 4, 1)])
def test_portions_at_the_edges_of_units_and_sub_blocks(shape):
    dtype = torch.bfloat16
    k, dev = M._kernels("hip", dtype)
    heads, vdim, n_state, groups, taps, norm_groups = shape
    width = 2 * heads * vdim + 2 * groups * n_state + heads
    g = torch.Generator().manual_seed(8)
    w = M._ssm_weights(*shape, 11, dtype, slow=0)
    lens = [1, 1, 127, 128, 129, 2, 64, 65, 300, 7]                     # two single tokens first
    starts = [3, 0, 0, 5, 0, 1, 0, 2, 9, 0]
    first = [torch.randn((s, width), generator=g).to(dtype) for s in starts]
    then = [torch.randn((n, width), generator=g).to(dtype) for n in lens]
    slots = list(range(len(lens)))

    def both(side_by_side):
        k.state_space_blocks_side_by_side = side_by_side
        try:
            states = M._new_states(dev, len(lens), shape, fill=float("nan"))
            for i, s in enumerate(starts):                              # what the requests had before, token by token
                for t in range(s):
                    M._run_ssm(k, dev, first[i][t:t + 1], w, shape, 1e-6, states, [1], [t], [slots[i]])
            return M._run_ssm(k, dev, torch.cat(then), w, shape, 1e-6, states, lens, starts, slots), states
        finally:
            k.state_space_blocks_side_by_side = True
    got, states = both(True)
    one, states_one = both(False)
    # both are float sums of the same numbers in another order, rounded once: half a unit of bfloat16 (2^-8) beside 1e-5
    M._close(got, one.cpu(), dtype, "token by token", tol=1e-2)
    for a, b in zip(states, states_one):
        M._close(a, b.cpu(), torch.float32, "the states left behind", tol=1e-4)
    # a portion's outputs do not depend on what else is in the step (units of one size)
    i, at = 8, sum(lens[:8])
    states = M._new_states(dev, 1, shape, fill=float("nan"))
    for t in range(starts[i]):
        M._run_ssm(k, dev, first[i][t:t + 1], w, shape, 1e-6, states, [1], [t], [0])
    alone = M._run_ssm(k, dev, then[i], w, shape, 1e-6, states, [lens[i]], [starts[i]], [0])
    assert torch.equal(alone, got[at:at + lens[i]])


def test_units_grow_with_the_step():
    from nano_vllm_amd.kernels.ops import state_space_units
    assert state_space_units([1, 129, 5], 1, 64, 256) == (128, [0, 0, 128, 2, 0, 128, 1, 2, 1, 0, 5, 1], [0, 2, 0, 1])
    size, units, chains = state_space_units([2000, 3], 0, 64, 256)          # 17 units of 128 are 4.25 workgroups a compute unit
    assert size == 256 and len(units) // 4 == 9 and chains == [0, 8, 0, 2000 - 7 * 256]
