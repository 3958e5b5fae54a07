"""A step in which every request brings one token runs kernels of its own for the matrix memory and the delta rule: its results and
what it leaves in the states are, bit for bit, those of the same tokens in a step with a longer portion beside them."""
import pytest
import torch

from reinfer_amd import kernels
from test_gpu_kobolix_kernels import DEV, make_batch

pytestmark = pytest.mark.gpu

# a prompt in slots 2 and 0 first, then single tokens: a padding row among them, a request that starts with its first token
LIVE = [([2, 0], [0, 0]), ([2, -1, 0, 3], [0, 0, 0, 1]), ([3, 2, 0], [0, 0, 0])]


def batch_of(q_lens, slots, fresh):
    batch = make_batch(q_lens, slots, fresh, DEV)
    batch.max_q_len = max(q_lens)
    return batch


def beside(rows, extra):
    return torch.cat([rows, extra[:, :rows.shape[1]].to(rows.dtype)])


# lanes of 8, 16, 32 and 64 a column; runs of 2, 4 and 8, whole and part full; keys and rows that 16-byte accesses cannot read
@pytest.mark.parametrize("H,dk,dv", [(16, 128, 256), (2, 64, 20), (3, 20, 28), (1, 8, 3), (2, 256, 17), (1, 512, 6), (2, 300, 10), (4, 12, 70)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", [0, 3])
def test_matrix_memory(H, dk, dv, dtype, pad):
    ops = kernels.current()
    g = torch.Generator(device=DEV).manual_seed(H * 100 + dk + dv)
    width = 2 * H * dk + H * dv + pad
    bias = torch.randn(2 * H, generator=g, device=DEV)
    st = torch.full((5, ops.scan_state_floats("matrix_memory", H, dk, dv)), float("nan"), device=DEV)

    def run(q_lens, slots, fresh, proj, gates, state):
        out = torch.empty(proj.shape[0], H * dv, device=DEV)
        ops.matrix_memory_scan(proj, pad, pad + H * dk, pad + 2 * H * dk, gates, bias, state, batch_of(q_lens, slots, fresh), H,
                               dk, dv, 6.0, dk ** -0.5, 1e-6, out)
        return out
    rows = lambda n: (torch.randn(n, width, generator=g, device=DEV).to(dtype), torch.randn(n, 2 * H, generator=g, device=DEV) * 3)
    run([5, 9], [2, 0], [1, 1], *rows(14), st)
    other = st.clone()
    for slots, fresh in LIVE:
        (proj, gates), (p2, g2) = rows(len(slots)), rows(2)
        a = run([1] * len(slots), slots, fresh, proj, gates, st)
        b = run([1] * len(slots) + [2], slots + [4], fresh + [1], beside(proj, p2), beside(gates, g2), other)
        assert torch.isfinite(a).all() and torch.equal(a, b[:len(slots)])
        kept = [s for s in slots if s >= 0]
        assert torch.equal(st[kept].view(torch.int32), other[kept].view(torch.int32))


@pytest.mark.parametrize("H,G,dk,dv,taps", [(32, 16, 128, 128, 4), (4, 1, 20, 12, 3), (2, 2, 136, 8, 1), (1, 1, 64, 70, 2), (6, 3, 130, 9, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_delta_rule(H, G, dk, dv, taps, dtype):
    ops = kernels.current()
    g = torch.Generator(device=DEV).manual_seed(H * 100 + dk + taps)
    C = 2 * G * dk + H * dv
    filt = torch.randn(C, taps, generator=g, device=DEV) * 0.6
    a_log, dt_bias = torch.randn(H, generator=g, device=DEV) - 1.0, torch.randn(H, generator=g, device=DEV) * 0.5
    off = ops.scan_state_floats("delta_rule", H, dk, dv)
    st = torch.full((5, off + (taps - 1) * C), float("nan"), device=DEV)

    def run(q_lens, slots, fresh, proj, ba, state):
        batch = batch_of(q_lens, slots, fresh)
        qkv, out = torch.empty(proj.shape[0], C, device=DEV), torch.empty(proj.shape[0], H * dv, device=DEV)
        ops.delta_rule_prepare(proj, filt, state, off, batch, G, dk, H, dv, taps, 1e-6, dk ** -0.5, qkv)
        ops.delta_rule_scan(qkv, ba.clone(), a_log, dt_bias, state, batch, H, G, dk, dv, out)
        return torch.cat([qkv, out], 1)
    rows = lambda n: (torch.randn(n, C + 3, generator=g, device=DEV).to(dtype), torch.randn(n, 2 * H, generator=g, device=DEV) * 2)
    run([5, 2], [2, 0], [1, 1], *rows(7), st)
    other = st.clone()
    for slots, fresh in LIVE:
        (proj, ba), (p2, b2) = rows(len(slots)), rows(2)
        a = run([1] * len(slots), slots, fresh, proj, ba, st)
        b = run([1] * len(slots) + [2], slots + [4], fresh + [1], beside(proj, p2), beside(ba, b2), other)
        assert torch.isfinite(a).all() and torch.equal(a, b[:len(slots)])
        kept = [s for s in slots if s >= 0]
        assert torch.equal(st[kept].view(torch.int32), other[kept].view(torch.int32))


# rows of whole runs of eight, part of a wave's, one and two a thread; rows that are none, or too long; operands off 16 bytes
@pytest.mark.parametrize("h", [3, 8, 248, 512, 4095, 4096, 8192, 8200])
@pytest.mark.parametrize("n", [1, 2, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mean_of_normed_rows(h, n, dtype):
    g = torch.Generator(device=DEV).manual_seed(h + n)
    xs = [torch.randn(3 * h + 1, generator=g, device=DEV).to(dtype)[h % 16 == 0 and n == 4:][:3 * h].view(3, h) for _ in range(n)]
    ws = [torch.rand(h, generator=g, device=DEV) + 0.5 for _ in range(n)]
    base = torch.randn(3, h, generator=g, device=DEV)
    want = sum(x.double() / (x.double().pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w.double() for x, w in zip(xs, ws)) / n
    resid, out = base.clone(), torch.empty(3, h, dtype=dtype, device=DEV)
    kernels.current().normed_mean(xs, ws, 1e-6, resid=resid, scale=0.5)
    kernels.current().normed_mean(xs, ws, 1e-6, out=out)
    # sums of h squares: their relative error is below h 2^-24 at worst, half of it reaches the result; products of a few roundings
    assert (resid.double() - (base.double() + 0.5 * want)).abs().max() <= (h / 2 + 8) * 2.0 ** -24 * 8
    assert (out.double() - want).abs().max() <= ((h / 2 + 8) * 2.0 ** -24 + (2.0 ** -9 if dtype == torch.bfloat16 else 0.0)) * 8


# whole runs of eight for each thread and for some; one row fewer, as many rows as CUs, and one more, where rows are read twice again
@pytest.mark.parametrize("h", [520, 4096])
@pytest.mark.parametrize("n", [2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mean_of_as_many_rows_as_cus(h, n, dtype):
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    g = torch.Generator(device=DEV).manual_seed(h + n)
    xs = [torch.randn(cus + 1, h, generator=g, device=DEV).to(dtype) for _ in range(n)]
    ws = [torch.rand(h, generator=g, device=DEV) + 0.5 for _ in range(n)]
    want = sum(x.double() / (x.double().pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w.double() for x, w in zip(xs, ws)) / n
    outs = []
    for rows in (1, cus - 1, cus, cus + 1):
        resid = torch.ones(rows, h, device=DEV)
        kernels.current().normed_mean([x[:rows] for x in xs], ws, 1e-6, resid=resid, scale=0.5)
        assert (resid.double() - 1 - 0.5 * want[:rows]).abs().max() <= (h / 2 + 8) * 2.0 ** -24 * 8
        outs.append(resid)
    for a in outs[:-1]:
        assert torch.equal(a, outs[-1][:len(a)])
