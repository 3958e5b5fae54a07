"""Experts' choice and activation on both sides of the number of rows up to which they are one kernel: which kernels run, and the same bits."""
import pytest
import torch

from reinfer_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def places():
    return 8 * torch.cuda.get_device_properties(DEV).multi_processor_count


@pytest.mark.parametrize("E,top,ff,shared,groups,kept", [(16, 4, 1024, 2048, 4, 2), (64, 8, 512, 512, 8, 4), (8, 3, 256, 8, 1, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gated(library_calls, E, top, ff, shared, groups, kept, dtype):
    ops = kernels.current()
    n = E * ff + shared
    line = places() // -(-(n // 8) // 256)
    for T in (line, line + 1, 2 * line + 5):
        g = torch.Generator(device=DEV).manual_seed(T + E)
        up, logits = torch.randn(T, 2 * n, generator=g, device=DEV).to(dtype), torch.randn(T, E, generator=g, device=DEV)
        act, want = torch.full((T, n), 7.0, device=DEV, dtype=dtype), torch.empty(T, n, device=DEV, dtype=dtype)
        names = library_calls(lambda: ops.moe_choose_scale(up, act, logits, top, E, ff, shared=shared, scoring="sigmoid", scale=2.5,
                                                           groups=groups, groups_kept=kept, group_top=2))
        assert names == (["ra_moe_choose_scale"] if T <= line else ["ra_moe_route_sigmoid", "ra_moe_silu_gate_scale_shared"])
        ids, weights = torch.empty(T, top, device=DEV, dtype=torch.int32), torch.empty(T, top, device=DEV)
        kernels.library.call("ra_moe_route_sigmoid", logits.data_ptr(), logits.stride(0), E, top, groups, kept, 2, 2.5, ids.data_ptr(),
                             weights.data_ptr(), T, torch.cuda.current_stream().cuda_stream)
        ops.moe_silu_gate_scale(up, want, ids, weights, E, ff, shared)
        assert torch.equal(act, want)


@pytest.mark.parametrize("E,top,ff", [(16, 4, 1536), (64, 6, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_squared(library_calls, E, top, ff, dtype):
    ops = kernels.current()
    n = E * ff
    line = places() // -(-(n // 8) // 256)
    for T in (line, line + 1, 2 * line + 5):
        g = torch.Generator(device=DEV).manual_seed(T + E)
        up, logits = torch.randn(T, n, generator=g, device=DEV).to(dtype), torch.randn(T, E, generator=g, device=DEV)
        act, want = torch.full((T, n), 7.0, device=DEV, dtype=dtype), torch.empty(T, n, device=DEV, dtype=dtype)
        names = library_calls(lambda: ops.moe_choose_scale(up, act, logits, top, E, ff))
        assert names == (["ra_moe_choose_scale"] if T <= line or dtype == torch.float32 else ["ra_moe_topk", "ra_moe_relu2_scale"])
        ids, weights = torch.empty(T, top, device=DEV, dtype=torch.int32), torch.empty(T, top, device=DEV)
        kernels.library.call("ra_moe_topk", logits.data_ptr(), E, E, top, ids.data_ptr(), weights.data_ptr(), T, torch.cuda.current_stream().cuda_stream)
        ops.moe_relu2_scale(up, want, ids, weights, E, ff)
        assert torch.equal(act, want)
