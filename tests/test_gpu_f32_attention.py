"""The 32-bit attention over the paged cache: the order of a token's sums, and scores that are no finite numbers."""
import pytest
import torch

from reinfer_amd import kernels
from test_gpu_kernels import DEV, FakeBatch, kt, make_paged_case, vt

pytestmark = pytest.mark.gpu


def attend(q, kc, vc, q_lens, starts, tables, Hq, Hkv, d, window=0, keep=0):
    T = sum(q_lens)
    out = torch.full((T, Hq * d), float("nan"), device=DEV)
    kernels.current().attention_plain(q.reshape(T, Hq * d), Hq * d, out, kt(kc), vt(vc), FakeBatch(q_lens, starts, tables), Hq, Hkv,
                                      d, d ** -0.5, window, 0, keep=keep)
    return out


# one and two heads a workgroup; fewer tiles than shares, some more, many; windows and kept keys off the tiles. The long portion
# is taken by workgroups of two waves, the short ones by workgroups of eight
@pytest.mark.parametrize("Hq,Hkv,d", [(32, 8, 128), (32, 32, 64), (64, 16, 64), (24, 8, 256)])
@pytest.mark.parametrize("start,window,keep", [(0, 0, 0), (700, 0, 0), (150, 77, 0), (400, 100, 21)])
def test_a_token_has_the_same_bits_whatever_stands_beside_it(Hq, Hkv, d, start, window, keep):
    n = 330
    q, kc, vc, tables = make_paged_case("float32", Hq, Hkv, d, [n], [start], seed=start + d)
    whole = attend(q, kc, vc, [n], [start], tables, Hq, Hkv, d, window, keep)
    assert torch.isfinite(whole).all()
    for lo, hi in ((0, 1), (1, 18), (127, 129), (300, 330), (329, 330)):
        part = attend(q[lo:hi].contiguous(), kc, vc, [hi - lo], [start + lo], tables, Hq, Hkv, d, window, keep)
        assert torch.equal(part, whole[lo:hi]), (lo, hi)


@pytest.mark.parametrize("n", [1, 300])
def test_scores_that_are_no_finite_numbers(n):
    """A whole tile of keys whose scores overflow to minus infinity weighs nothing, and a key that is no number reaches every
    result that sees it."""
    Hq, Hkv, d, start = 32, 8, 128, 400
    q, kc, vc, tables = make_paged_case("float32", Hq, Hkv, d, [n], [start], seed=n, poison=False)
    q[..., 0] = 10.0
    blocks = tables[0].long()
    assert kc.shape[2] == 16
    for tile in (0, 3, 8, 11):               # a share's first tile, others in its middle, the first of its second round
        kc[blocks[tile], :, :, 0] = -3e38
    out = attend(q, kc, vc, [n], [start], tables, Hq, Hkv, d)
    gone = torch.isin(torch.arange(start + n) // 16, torch.tensor([0, 3, 8, 11]))
    flat = lambda c: c[blocks].transpose(1, 2).reshape(-1, Hkv, d)[:start + n].double().cpu()
    K, V = flat(kc).repeat_interleave(Hq // Hkv, 1), flat(vc).repeat_interleave(Hq // Hkv, 1)
    for t in (0, n - 1):
        s = (K * q[t].double().cpu()[None]).sum(-1) * d ** -0.5
        s[gone | (torch.arange(start + n) > start + t)] = float("-inf")
        want = (torch.softmax(s, 0)[..., None] * V).sum(0).reshape(-1)
        assert (out[t].double().cpu() - want).abs().max() < 1e-5
    kc[blocks[2], 0, 5, 7] = float("nan")
    out = attend(q, kc, vc, [n], [start], tables, Hq, Hkv, d).view(n, Hkv, -1)
    assert torch.isnan(out[:, 0]).all() and torch.isfinite(out[:, 1:]).all()
