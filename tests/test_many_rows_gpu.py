"""The row kernels for steps of many bfloat16 rows (a wave a row) against the ones for few rows, at the widths, strides and
options where their vectors, lanes and tails can go wrong.  Both sum in float, in other orders (a part in 2^20 at these
widths), and round once: their results differ by at most one unit of bfloat16 (2^-7 of the value, with the rounding)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def _k():
    from nano_vllm_amd.kernels import HipKernels
    return HipKernels(DEV, BF, quiet=True)


def _same(a, b, what):
    a, b = a.double(), b.double()
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6 * float(b.abs().max())).all()), (what, float((a - b).abs().max()))


def _parts(n, most):
    return [slice(i, min(i + most, n)) for i in range(0, n, most)]


@pytest.mark.parametrize("width", [8, 504, 512, 520, 2048, 2056, 4096])
def test_norms_of_the_float_stream(width):
    from nano_vllm_amd.parts.base import NormedAddend, ScaledPair, StreamAddend
    k, rows = _k(), 259
    g = torch.Generator(device=DEV).manual_seed(width)
    rand = lambda *s, dtype=BF: torch.randn(s, generator=g, device=DEV).to(dtype)
    a, b, r, x = rand(rows, width), rand(rows, width + 8)[:, 8:], rand(rows, width, dtype=torch.float32), rand(rows, width, dtype=torch.float32)
    w1, w2, s1, s2 = (1 + 0.1 * rand(width).float() for _ in range(4))

    def both(run):
        """run(rows slice) -> outputs, for all rows at once and in parts that the kernels for few rows take"""
        whole = run(slice(0, rows))
        parts = [run(p) for p in _parts(rows, 100)]
        for n, t in enumerate(whole):
            _same(t, torch.cat([p[n] for p in parts]), n)
    for w in (w1, w1.to(BF)):
        both(lambda p: k.stream_rms_norm((a[p], b[p]), r[p].clone(), w, 1e-6, 1.0))
        both(lambda p: k.stream_rms_norm((), r[p].clone(), w, 1e-6, 0.0, out=torch.empty_like(a[p])))
        both(lambda p: k.stream_rms_norm((a[p], b[p]), None, w, 1e-6))
        both(lambda p: k.stream_rms_norm((NormedAddend(a[p], w, 1e-5, 0.5, 1.0),), r[p].clone(), w, 1e-6))
        both(lambda p: k.stream_rms_norm((NormedAddend(ScaledPair(a[p], b[p], 0.75, 0.5, k), w, 1e-5), StreamAddend(x[p])), r[p].clone(), w, 1e-6))
        both(lambda p: k.stream_add((NormedAddend(a[p], w, 1e-5, 0.5),), r[p].clone()))
    both(lambda p: k.stream_scaled_norm([(a[p], s1), (b[p], s2)], r[p].clone(), w1, 1e-6, weight2=w2))
    both(lambda p: [t for t in k.stream_scaled_norm([(a[p], None)], None, w1, 1e-6) if t is not None])
    both(lambda p: (k.pair_norm_mean(a[p], w1, b[p], w2, 1e-6),))


@pytest.mark.parametrize("hq,hkv,D,DV,R,page", [(16, 8, 128, 128, 64, 256), (4, 2, 64, 64, 64, 32), (2, 1, 8, 16, 0, 8), (3, 1, 512, 256, 128, 16),
                                                (4, 4, 32, 64, 16, 20)])
@pytest.mark.parametrize("kind", ["whole", "head", "unit", "values first", "values mixed", "gates"])
def test_preparation_of_q_k_and_v(hq, hkv, D, DV, R, page, kind):
    from nano_vllm_amd.kernels import ops
    k, T = _k(), 133
    g = torch.Generator(device=DEV).manual_seed(D + R)
    rand = lambda *s: torch.randn(s, generator=g, device=DEV)
    gates = hq if kind == "gates" else 0
    width = (hq + hkv) * D + hkv * DV
    row = (2 * rand(T, width + 8 + (gates + 7) // 8 * 8)).to(BF)[:, 8:]
    row = row[:, :width + gates] if gates % 8 == 0 else row
    pos = torch.arange(T, dtype=torch.int32, device=DEV) * 7
    table = k.rotary_step_table((500.0 ** (-torch.arange(0, R, 2, device=DEV).float() / R)), pos) if R else None
    pages = (T + page - 1) // page + 2
    slots = torch.arange(T, dtype=torch.int32, device=DEV) + page            # runs of eight, whole and cut
    slots[40:60] = torch.randperm(20, generator=torch.Generator().manual_seed(1)).int().to(DEV) + page + 40
    slots[100] = -1
    first = rand(T, hkv * DV)
    weights = {"whole": (1 + 0.1 * rand(hq * D), 1 + 0.1 * rand(hkv * D)), "head": ((1 + 0.1 * rand(D)).to(BF), (1 + 0.1 * rand(D)).to(BF))}.get(kind, (None, None))

    def run(p):
        kc = torch.zeros((pages, hkv, page, D), dtype=BF, device=DEV)
        vc = torch.zeros(ops.v_cache_shape(pages, hkv, DV, page), dtype=BF, device=DEV)
        n = p.stop - p.start
        extra, out = {}, []
        if kind in ("head", "unit", "gates"):
            extra.update(norm_per_head=True, norm_unit=kind != "head")
        if kind.startswith("values"):
            extra.update(v_norm=True, rot_interleaved=True)
            if kind == "values first":
                out = [torch.zeros((n, hkv * DV), device=DEV)]
                extra["v_first_out"] = out[0]
            else:
                extra.update(v_first_in=first[p].contiguous(), v_mix=torch.tensor(0.3, device=DEV))
        if gates:
            out = [torch.zeros((n, gates), device=DEV)]
            extra["head_gate"] = out[0]
        q = k.qk_rownorm_store(row[p].clone() if kind != "whole" else row.clone()[p], hq, hkv, D, DV, *weights, 1e-6, pos[p].contiguous(),
                               0.1 if kind == "whole" else 0.0, 64, slots[p].contiguous(), kc, vc,
                               rot_table=None if table is None else table[p].contiguous(), **extra)
        return [q.reshape(n, -1)] + out, kc, vc
    whole, kc, vc = run(slice(0, T))
    parts = [run(p) for p in _parts(T, 50)]
    for n, t in enumerate(whole):
        _same(t, torch.cat([p[0][n] for p in parts]), n)
    _same(kc, sum(p[1].float() for p in parts), "keys")
    _same(vc, sum(p[2].float() for p in parts), "values")
