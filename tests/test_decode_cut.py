"""How a decode step's keys are cut, by the numbers of workgroups that an MI355X holds at once (256 CUs)."""
import pytest

from reinfer_amd.kernels.ops import HipKernels


class Chip(HipKernels):
    def __init__(self):
        pass

    def _slots_of_decode(self, num_heads, num_kv_heads, head_dim, waves):
        lds = waves * (num_heads // num_kv_heads) * (head_dim + 2) * 4
        if waves == 12:
            return 256 if lds <= 64 << 10 else 0
        return 256 * (5 if head_dim <= 64 else 3 if head_dim <= 128 else 1)


# 11 query heads a KV head and more at 128, 6 and more at 256: the large workgroups' sums do not fit
NO_LARGE_FORM = [(64, 4, 128), (24, 2, 128), (16, 1, 256), (12, 2, 256)]
# above 128 elements the large form spills its registers, and is not used
WIDE_HEADS = [(16, 8, 256), (16, 4, 256), (4, 1, 256), (5, 1, 144), (8, 2, 192)]


@pytest.mark.parametrize("Hq,Hkv,d", NO_LARGE_FORM + WIDE_HEADS)
def test_few_pairs_without_the_large_form_are_cut(Hq, Hkv, d):
    chip = Chip()
    slots = chip._slots_of_decode(Hq, Hkv, d, 4)
    assert (chip._slots_of_decode(Hq, Hkv, d, 12) == 0) == ((Hq, Hkv, d) in NO_LARGE_FORM)
    for n in (1, 2, 3, 8, 16, 32, 64, 200):
        pairs = n * Hkv
        for ctx in (1, 256, 512, 1024, 2048, 4096, 16384, 65536):
            least, most, waves = chip.decode_chunk(n, Hq, Hkv, d, ctx)
            assert waves == 4 and least in (128, 256) and 1 <= most <= max(1, -(-ctx // least))
            if pairs <= 256:                                   # the chunks run side by side
                assert pairs * most <= max(slots, pairs)
            if pairs <= 64 and ctx * d >= 1024 * 128:          # one chunk a pair would leave three quarters of the CUs idle
                assert most >= 4 or most == slots // pairs
            if pairs <= 8 and ctx * d >= 16384 * 128:          # no more than 1,024 keys of 128 elements one after the other
                assert most * 1024 >= ctx * d // 128 or most == slots // pairs


def test_pairs_that_fill_half_of_the_chip():
    """Pairs that the chip holds twice as large workgroups are two such chunks each above 1,024 keys; a few more, which it holds
    once, are one up to 4,096 keys and small chunks above."""
    def cut(n, ctx):
        return Chip().decode_chunk(n, 32, 8, 128, ctx)[1:]
    assert cut(16, 1024) == (1, 12) and cut(16, 1025) == (2, 12) and cut(16, 16384) == (2, 12)
    assert cut(17, 4095) == (1, 12) and cut(17, 4096) == (768 // 136, 4)
    assert cut(20, 4096) == (1, 12) and cut(32, 16384) == (1, 12)


@pytest.mark.parametrize("Hq,Hkv", [(20, 2), (28, 4), (64, 8)])
def test_few_pairs_of_four_thousand_keys(Hq, Hkv):
    """A captured step's bucket of 2,049 to 4,096 keys: small chunks for up to 8 pairs, large ones from there and from the next bucket on."""
    chip = Chip()
    assert chip.decode_chunk(1, Hq, Hkv, 128, 4096)[1:] == (16, 4)
    assert chip.decode_chunk(1, Hq, Hkv, 128, 8192)[2] == 12
    assert chip.decode_chunk(16 // Hkv, Hq, Hkv, 128, 4096)[2] == 12
