"""The 32-bit path's products on the matrix cores at the edges of their tiles, and their attention of few tokens at the edges
of its blocks of keys: against float64, and bit for bit against the same rows in another batch or kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _kernels(dtype=torch.float32):
    from nano_vllm_amd.kernels import HipKernels
    return HipKernels(DEV, dtype, quiet=True)


@pytest.mark.parametrize("n,k", [(16, 4), (17, 33), (100, 128), (1000, 260), (4096, 257), (20000, 64)])
def test_rows_give_the_same_bits_in_every_tile(n, k):
    kern = _kernels()
    g = torch.Generator().manual_seed(n + k)
    x, w, b = torch.randn((700, k), generator=g), torch.randn((n, k), generator=g), torch.randn(n, generator=g)
    want = x.double() @ w.double().T + b.double()
    xd, wd, bd = x.to(DEV), w.to(DEV), b.to(DEV)
    whole = kern.linear(xd, wd, bd)
    # a chain of k products and sums in float is off by at most k rounding units of the sum of magnitudes
    bound = (x.abs().double() @ w.abs().double().T + b.abs().double()) * (k + 1) * 2.0 ** -24
    assert bool(((whole.double().cpu() - want).abs() <= bound).all())
    for m in (1, 15, 16, 17, 31, 33, 64, 65, 127, 129, 300):
        assert torch.equal(kern.linear(xd[-m:], wd, bd), whole[-m:]), m
    wide = torch.zeros((40, k + 3), device=DEV)                     # rows that are no whole vectors, at an odd offset
    wide[:, 1:k + 1] = xd[:40]
    assert torch.equal(kern.linear(wide[:, 1:k + 1], wd, bd), whole[:40])


@pytest.mark.parametrize("dim,chunk,sink", [(128, 0, False), (64, 0, True), (8, 96, False), (128, 200, True)])
def test_attention_of_few_tokens(dim, chunk, sink):
    from nano_vllm_amd.kernels import ops
    from nano_vllm_amd.kernels import library
    kern = _kernels()
    heads, kv, page = 4, 2, 64
    lens = [1, 63, 64, 65, 128, 511, 512, 513, 577, 1100]
    g = torch.Generator().manual_seed(dim)
    pages = [(n + page - 1) // page for n in lens]
    table = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=g), 0
    for i, p in enumerate(pages):
        table[i, :p] = order[at:at + p]
        at += p
    kc = torch.randn((sum(pages), kv, page, dim), generator=g)
    vc = torch.randn(ops.v_cache_shape(sum(pages), kv, dim, page), generator=g)
    vplain = vc.permute(0, 1, 2, 4, 3).reshape(sum(pages), kv, page, dim)
    for i, n in enumerate(lens):                                    # slots past a request's keys must not be read as numbers
        if n % page:
            kc[table[i, pages[i] - 1], :, n % page:] = float("nan")
            vplain_last = vc[table[i, pages[i] - 1]]
            for key in range(n % page, page):
                vplain_last[:, key // 32, :, key % 32] = float("nan")
    q = torch.randn((len(lens), heads * dim), generator=g)
    sinks = torch.randn(heads, generator=g) if sink else None

    def run(rows):
        """The per-token entry with the given rows of q, repeated (many pairs take the kernel of one wave each)."""
        n = len(rows)
        out = torch.empty((n, heads * dim), device=DEV)
        d = [q[rows].to(DEV), kc.to(DEV), vc.to(DEV), table[rows].to(DEV), torch.arange(n, dtype=torch.int32, device=DEV),
             torch.tensor([lens[r] - 1 for r in rows], dtype=torch.int32, device=DEV), None if sinks is None else sinks.to(DEV)]
        p, i32, i64, f32 = ops._p, ops.c_i32, ops.c_i64, ops.c_f32
        library.call("attn_generic", "f32", "nva_paged_attention_generic", p(d[0]), i64(heads * dim), p(out), i64(heads * dim), p(d[1]), p(d[2]),
                     p(d[3]), i32(d[3].shape[1]), p(d[4]), p(d[5]), i64(n), i32(heads), i32(kv), i32(dim), i32(dim), i32(page), f32(dim ** -0.5),
                     i32(0), i32(chunk), i32(0), f32(0.0), p(d[6]), p(None), p(None), p(None), i32(1), p(kern.fault_flag), kern._stream())
        torch.cuda.synchronize()
        return out.cpu()
    rows = list(range(len(lens)))
    got = run(rows)
    assert torch.equal(got, run(rows * 410)[:len(lens)])             # 16400 pairs: one wave each, the same operations
    for i, n in enumerate(lens):
        lo = (n - 1) // chunk * chunk if chunk else 0
        slots = [(int(table[i, j // page]), j % page) for j in range(lo, n)]
        for h in range(heads):
            ks = torch.stack([kc[a, h // 2, b] for a, b in slots]).double()
            vs = torch.stack([vc[a, h // 2, b // 32, :, b % 32] for a, b in slots]).double()
            s = ks @ q[i, h * dim:(h + 1) * dim].double() * dim ** -0.5
            e = torch.exp(s - s.max())
            total = e.sum() + (torch.exp(sinks[h].double() - s.max()) if sink else 0.0)
            want = (e / total) @ vs
            assert float((got[i, h * dim:(h + 1) * dim].double() - want).abs().max()) < 1e-5 * float(vs.abs().max()), (i, h)
