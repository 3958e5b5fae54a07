"""The two ways of the 32-bit attention, rows of 16 on the matrix cores and tokens on their own: the same bits, in every mixture."""
import pytest
import torch

from reinfer_amd import kernels
from test_gpu_kernels import DEV, FakeBatch, kt, make_paged_case, vt

pytestmark = pytest.mark.gpu


def attend(q, kc, vc, q_lens, starts, tables, Hq, Hkv, d, **how):
    T = sum(q_lens)
    out = torch.full((T, Hq * d), float("nan"), device=DEV)
    kernels.current().attention(q.reshape(T, Hq * d), Hq * d, out, kt(kc), vt(vc), FakeBatch(q_lens, starts, tables), Hq, Hkv, d,
                                d ** -0.5, **{"window": 0, "group": 0, **how})
    return out


def exact(q, kc, vc, n, start, table, Hq, Hkv, d, window, keep, aligned):
    """In 64 bits, one request."""
    ctx = start + n
    flat = lambda c: c[table.long()].transpose(1, 2).reshape(-1, Hkv, d)[:ctx].double().cpu().nan_to_num()
    K, V = flat(kc).repeat_interleave(Hq // Hkv, 1), flat(vc).repeat_interleave(Hq // Hkv, 1)
    s = torch.einsum("thd,khd->htk", q.double().cpu(), K) * d ** -0.5
    p, k = torch.arange(start, ctx)[:, None], torch.arange(ctx)[None]
    lo = p * 0 if not window else p - p % window if aligned else p - window + 1
    s = s.masked_fill(~((k <= p) & ((k >= lo) | (k < keep))), float("-inf"))
    return torch.einsum("htk,khd->thd", torch.softmax(s, -1), V).reshape(n, -1)


# groups of 1 (16 tokens a workgroup), 3 (five), 4, 8 and 16 (one); blocks of one tile and three
@pytest.mark.parametrize("Hq,Hkv,d,bs", [(6, 6, 64, 16), (24, 8, 128, 48), (16, 4, 128, 16), (16, 2, 256, 16), (32, 2, 64, 48)])
@pytest.mark.parametrize("how", [{}, {"window": 37}, {"window": 100, "keep": 21}, {"window": 64, "aligned": True},
                                 {"softcap": 5.0}])
def test_rows_and_tokens_alone(Hq, Hkv, d, bs, how):
    """A step of portions of many lengths, at the edges of tiles and of workgroups, against every one of its tokens in a step of its own,
    and against 64 bits: a sum of n terms of chains that are each rounded, below n 2^-24 of the terms' sizes."""
    q_lens = [1, 16, 33, 1, 1, 90, 47, 15, 130]
    starts = [0, 16, 300, 511, 31, 0, 129, 240, 5]
    q, kc, vc, tables = make_paged_case("float32", Hq, Hkv, d, q_lens, starts, bs=bs, seed=d + Hq,
                                       window=0 if "keep" in how else how.get("window", 0))
    whole = attend(q, kc, vc, q_lens, starts, tables, Hq, Hkv, d, **how)
    assert torch.isfinite(whole).all()
    at = 0
    for i, (n, s) in enumerate(zip(q_lens, starts)):
        for lo, hi in {(0, 1), (n - 1, n), (n // 2, n // 2 + 1)}:
            one = attend(q[at + lo:at + hi].contiguous(), kc, vc, [hi - lo], [s + lo], tables[i:i + 1], Hq, Hkv, d, **how)
            assert torch.equal(one, whole[at + lo:at + hi]), (i, lo)
        if "softcap" not in how:
            want = exact(q[at:at + n], kc, vc, n, s, tables[i], Hq, Hkv, d, how.get("window", 0), how.get("keep", 0),
                         how.get("aligned", False))
            # scores of size 1 to within their chains' rounding, weights and sums after them: 4 (d + n) 2^-24 of values up to 5
            assert (whole[at:at + n].double().cpu() - want).abs().max() < 4 * (d + s + n) * 2 ** -24 * 5
        at += n


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 3e38])
def test_a_value_that_is_no_finite_number_reaches_those_alone_that_see_it(bad):
    Hq, Hkv, d, n = 32, 8, 128, 70
    q, kc, vc, tables = make_paged_case("float32", Hq, Hkv, d, [n], [0], seed=3)
    plain = attend(q, kc, vc, [n], [0], tables, Hq, Hkv, d)
    vc[tables[0, 50 // 16], 5, 50 % 16, 7] = bad
    out = attend(q, kc, vc, [n], [0], tables, Hq, Hkv, d).view(n, Hkv, -1, d)
    plain = plain.view(n, Hkv, -1, d)
    assert torch.equal(out[:50], plain[:50])
    rest = [h for h in range(Hkv) if h != 5]
    assert torch.equal(out[:, rest], plain[:, rest])
    assert torch.equal(out[50:, 5, :, :7], plain[50:, 5, :, :7]) and torch.equal(out[50:, 5, :, 8:], plain[50:, 5, :, 8:])
    for t in (50, n - 1):
        one = attend(q[t:t + 1].contiguous(), kc, vc, [1], [t], tables, Hq, Hkv, d).view(Hkv, -1, d)
        assert torch.equal(out[t].nan_to_num(), one.nan_to_num()) and torch.equal(out[t].isnan(), one.isnan())


# groups of 5, 7 and 14 (all heads a workgroup), 6 (two tokens), 24 (12 heads) and 11 (a head each); more requests than a wave has lanes
@pytest.mark.parametrize("Hq,Hkv,d", [(40, 8, 128), (14, 2, 64), (28, 2, 64), (12, 2, 256), (24, 1, 128), (22, 2, 64)])
def test_steps_of_many_requests(Hq, Hkv, d):
    """Single tokens beside portions, a few tokens of many requests: tiles of each request's own, of which a step's first and last count."""
    for q_lens in ([1] * 9 + [100] + [1] * 3, [1 + i % 5 for i in range(70)], [3] * 64 + [40], [1] * 130):
        starts = [(37 * i) % 210 for i in range(len(q_lens))]
        q, kc, vc, tables = make_paged_case("float32", Hq, Hkv, d, q_lens, starts, seed=len(q_lens))
        whole = attend(q, kc, vc, q_lens, starts, tables, Hq, Hkv, d)
        assert torch.isfinite(whole).all()
        at = 0
        for i, (n, s) in enumerate(zip(q_lens, starts)):
            if i % 11 == 0 or n > 30 or i == len(q_lens) - 1:
                for t in {0, n - 1}:
                    one = attend(q[at + t:at + t + 1].contiguous(), kc, vc, [1], [s + t], tables[i:i + 1], Hq, Hkv, d)
                    assert torch.equal(one, whole[at + t:at + t + 1]), (len(q_lens), i, t)
            at += n


def test_many_requests_beside_a_portion_take_what_their_workgroups_take():
    """Eight single tokens and a portion of 100, 40 heads on 8 KV heads: a workgroup that took 16 tokens of nine requests one request after
    the other made this four times the portion alone."""
    Hq, Hkv, d = 40, 8, 128

    def time(q_lens, starts):
        q, kc, vc, tables = make_paged_case("float32", Hq, Hkv, d, q_lens, starts, seed=1)
        out, batch, best = torch.empty(sum(q_lens), Hq * d, device=DEV), FakeBatch(q_lens, starts, tables), float("inf")
        rows, k, v = q.reshape(sum(q_lens), Hq * d), kt(kc), vt(vc)
        for _ in range(8):
            first, last = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda._sleep(200000)
            first.record()
            for _ in range(4):
                kernels.current().attention(rows, Hq * d, out, k, v, batch, Hq, Hkv, d, d ** -0.5, window=0, group=0)
            last.record()
            torch.cuda.synchronize()
            best = min(best, first.elapsed_time(last))
        return best
    # as workgroups of their own the single ones add 64 to 56: 1.5 times (measured), with room for twice that
    assert time([1] * 8 + [100], [300] * 8 + [0]) < 3 * time([100], [0])


def test_first_tokens_that_the_kernel_cannot_read_are_refused():
    q, kc, vc, tables = make_paged_case("float32", 4, 2, 64, [3, 2], [0, 5], seed=0)
    batch, out = FakeBatch([3, 2], [0, 5], tables), torch.empty(5, 256, device=DEV)
    cu = batch.cu_tokens
    for wrong, error in ((cu.long(), TypeError), (cu[:2], ValueError), (torch.stack([cu, cu], 1)[:, 0], TypeError)):
        batch.cu_tokens = wrong
        with pytest.raises(error):
            kernels.current().attention(q.reshape(5, -1), 256, out, kt(kc), vt(vc), batch, 4, 2, 64, 0.125, window=0, group=0)
