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
