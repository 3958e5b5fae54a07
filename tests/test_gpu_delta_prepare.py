"""The delta rule's inputs for prompts, made in runs of eight tokens, against the plain form and the kernel of one token a wave."""
import pytest
import torch

from kernel_double import KernelDouble
from reinfer_amd import kernels
from test_gpu_kobolix_kernels import DEV, make_batch

pytestmark = pytest.mark.gpu


# heads of 16, 32 and 64 lanes a group, that fill and do not fill them, key and value heads of unlike width, fewer taps than the
# kernel holds; requests of one to three tokens and ones that end inside a run, a padding row, requests that go on
@pytest.mark.parametrize("H,G,dk,dv,taps,rows", [(64, 32, 16, 20, 4, 600), (16, 8, 128, 96, 4, 1100), (16, 8, 128, 128, 2, 1028),
                                                 (8, 4, 132, 256, 3, 1201), (32, 16, 64, 64, 1, 1500)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_delta_rule_prepare_in_runs(H, G, dk, dv, taps, rows, dtype):
    ops, ref = kernels.current(), KernelDouble()
    g = torch.Generator().manual_seed(rows + taps)
    C = 2 * G * dk + H * dv
    filt = torch.randn(C, taps, generator=g) * 0.6
    state = torch.randn(6, 8 + (taps - 1) * C, generator=g)
    q_lens, slots, fresh = [1, 2, 3, rows - 17, 1, 10], [0, 3, 1, 5, -1, 2], [0, 1, 0, 0, 0, 1]
    proj = torch.randn(rows, C + 4, generator=g).to(dtype)
    st_ref, want = state.clone(), torch.empty(rows, C)
    ref.delta_rule_prepare(proj, filt, st_ref, 8, make_batch(q_lens, slots, fresh, "cpu"), G, dk, H, dv, taps, 1e-6, 0.25, want)
    st, got = state.to(DEV), torch.full((rows, C), float("nan"), device=DEV)
    args = (G, dk, H, dv, taps, 1e-6, 0.25)
    ops.delta_rule_prepare(proj.to(DEV), filt.to(DEV), st, 8, make_batch(q_lens, slots, fresh, DEV), *args, got)
    # taps products and a sum of a head's squares in float: a few roundings of the largest values
    assert ((got.cpu() - want).abs() <= 1e-5 * want.abs().max()).all()
    assert torch.equal(st.cpu(), st_ref)
    # rows that four-channel accesses cannot read: the kernel of one token a wave
    odd = torch.empty(rows, C + 3, device=DEV, dtype=dtype)
    odd[:, :C] = proj[:, :C].to(DEV)
    st, other = state.to(DEV), torch.full((rows, C), float("nan"), device=DEV)
    ops.delta_rule_prepare(odd, filt.to(DEV), st, 8, make_batch(q_lens, slots, fresh, DEV), *args, other)
    assert ((got - other).abs() <= 1e-5 * other.abs().max()).all()


@pytest.mark.parametrize("H,G,dk,dv", [(64, 32, 16, 20), (16, 8, 64, 48), (16, 8, 68, 96), (16, 8, 128, 128), (16, 8, 132, 256), (8, 8, 256, 40)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_token_alone_and_in_a_prompt_has_the_same_inputs(H, G, dk, dv, dtype):
    """Tokens one a step, which a wave a head takes, against the same tokens as one portion in runs: the same bits."""
    ops = kernels.current()
    g = torch.Generator().manual_seed(dk)
    C, rows, taps, last = 2 * G * dk + H * dv, 1203, 4, 6
    filt = (torch.randn(C, taps, generator=g) * 0.6).to(DEV)
    proj = torch.randn(rows, C + 4, generator=g).to(dtype).to(DEV)
    args = (G, dk, H, dv, taps, 1e-6, 0.25)
    st, whole = torch.zeros(1, (taps - 1) * C, device=DEV), torch.empty(rows, C, device=DEV)
    ops.delta_rule_prepare(proj, filt, st, 0, make_batch([rows], [0], [1], DEV), *args, whole)
    one = torch.zeros(1, (taps - 1) * C, device=DEV)
    first = torch.empty(rows - last, C, device=DEV)
    ops.delta_rule_prepare(proj[:-last], filt, one, 0, make_batch([rows - last], [0], [1], DEV), *args, first)
    assert torch.equal(first, whole[:-last])
    for t in range(rows - last, rows):
        got = torch.empty(1, C, device=DEV)
        ops.delta_rule_prepare(proj[t:t + 1], filt, one, 0, make_batch([1], [0], [0], DEV), *args, got)
        assert torch.equal(got[0], whole[t]), t
    assert torch.equal(one, st)
    few = torch.empty(5, C, device=DEV)
    ops.delta_rule_prepare(proj[:5], filt, torch.zeros_like(st), 0, make_batch([5], [0], [1], DEV), *args, few)
    assert torch.equal(few, whole[:5])
