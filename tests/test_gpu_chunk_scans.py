"""The matrix memory and the delta rule in chunks of 16 tokens, against a plain PyTorch form token by token: keys and values
that end inside a tile or a group of columns, portions around a chunk's length, requests side by side, a padding row, and
calls that take turns with the token-by-token kernels on one state."""
import pytest
import torch

from kernel_double import KernelDouble
from reinfer_amd import kernels
from test_gpu_kobolix_kernels import DEV, close, make_batch

pytestmark = pytest.mark.gpu

# (lengths, state slots, first steps, in chunks): the second call goes on token by token, the third in chunks again
CALLS = [([17, 33], [2, 0], [1, 1], True), ([3, 1, 20], [2, -1, 0], [0, 0, 0], False),
         ([16, 1, 150, 15], [0, -1, 2, 3], [0, 0, 0, 1], True), ([65, 100], [2, 0], [1, 0], True), ([2, 1], [0, 3], [0, 0], False)]


def matrix_memory(proj, q_off, k_off, v_off, z, bias, state, batch, H, dk, dv, cap, eps):
    """Token by token in 64 bits -> (read-out, how far roundings may move it for one of 2^-24 a term): beside the memory and
    its normaliser, those of the entries' sizes."""
    out, size = (torch.zeros(proj.shape[0], H, dv, dtype=torch.float64) for _ in range(2))
    p = proj.double()
    g = z.double() + bias.double()
    g = cap * torch.tanh(g / cap)
    for i, slot in enumerate(batch.state_slots.tolist()):
        if slot < 0:
            continue
        if batch.fresh[i]:
            state[slot] = [torch.zeros(H, dk, dv + 1, dtype=torch.float64) for _ in range(2)] + [torch.zeros(H, dtype=torch.float64)]
        S, A, m = state[slot]
        for t in range(int(batch.cu_tokens[i]), int(batch.cu_tokens[i + 1])):
            q, k = (p[t, o:o + H * dk].view(H, dk) for o in (q_off, k_off))
            q = q * dk ** -0.5
            v = torch.cat([p[t, v_off:v_off + H * dv].view(H, dv), torch.ones(H, 1, dtype=torch.float64)], 1)
            a, b = g[t, :H], torch.nn.functional.logsigmoid(g[t, H:])
            new = torch.maximum(b + m, a)
            keep, take = torch.exp(b + m - new)[:, None, None], torch.exp(a - new)[:, None, None]
            m = new
            S = keep * S + take * k[:, :, None] * v[:, None]
            A = keep * A + take * k.abs()[:, :, None] * v.abs()[:, None]
            o, mag = (S * q[..., None]).sum(1), (A * q.abs()[..., None]).sum(1)
            den = torch.maximum(o[:, -1:].abs(), torch.exp(-m)[:, None]) + eps
            out[t] = o[:, :-1] / den
            size[t] = mag[:, :-1] / den + out[t].abs() * mag[:, -1:] / den
        state[slot] = [S, A, m]
    return out.view(-1, H * dv), size.view(-1, H * dv)


@pytest.mark.parametrize("H,dk,dv", [(2, 128, 40), (3, 20, 28), (1, 136, 9), (1, 8, 17), (2, 256, 12), (5, 64, 24), (2, 100, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("spread", [3.0, 30.0])          # gates far apart: factors that vanish in float inside a chunk
def test_matrix_memory_in_chunks(H, dk, dv, dtype, spread):
    ops = kernels.current()
    g = torch.Generator().manual_seed(H * 1000 + dk)
    width = 2 * H * dk + H * dv + 8
    q_off, k_off, v_off = 8, 8 + H * dk, 8 + 2 * H * dk
    bias = torch.randn(2 * H, generator=g)
    st_gpu = torch.full((4, ops.scan_state_floats("matrix_memory", H, dk, dv)), float("nan"), device=DEV)
    state, seen = {}, 0
    for n, (q_lens, slots, fresh, chunks) in enumerate(CALLS):
        T = sum(q_lens)
        seen += max(q_lens)
        proj = (torch.randn(T, width, generator=g) * 0.7).to(dtype)
        gates = torch.randn(T, 2 * H, generator=g) * spread
        want, size = matrix_memory(proj, q_off, k_off, v_off, gates, bias, state, make_batch(q_lens, slots, fresh, "cpu"),
                                   H, dk, dv, 15.0, 1e-6)
        out = torch.full((T, H * dv), float("nan"), device=DEV)
        before = st_gpu.clone()
        ops.matrix_memory_scan(proj.to(DEV), q_off, k_off, v_off, gates.to(DEV), bias.to(DEV), st_gpu,
                               make_batch(q_lens, slots, fresh, DEV), H, dk, dv, 15.0, dk ** -0.5, 1e-6, out, chunks=chunks)
        # a term of the sums is rounded once a key entry, some twenty times in its chunk and twice in every later one, and
        # the gates' exponents (up to 15 and a chain of maxima) move its factor by 40 such roundings
        bound = (dk + 80 + seen / 8) * 2.0 ** -24 * size + 1e-12
        assert ((out.double().cpu() - want).abs() <= bound).all(), n
        untouched = [s for s in range(4) if s not in slots]
        assert torch.equal(torch.nan_to_num(st_gpu[untouched], nan=7.0), torch.nan_to_num(before[untouched], nan=7.0))


@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 40), (4, 1, 20, 12), (2, 2, 136, 8), (1, 1, 16, 70), (6, 3, 64, 50), (2, 1, 256, 33)])
@pytest.mark.parametrize("spread", [2.0, 12.0])
def test_delta_rule_in_chunks(H, G, dk, dv, spread):
    ops, ref = kernels.current(), KernelDouble()
    g = torch.Generator().manual_seed(H * 1000 + dk)
    C = 2 * G * dk + H * dv
    a_log, dt_bias = torch.randn(H, generator=g) * 0.5 - 1.0, torch.randn(H, generator=g) * 0.5
    st_gpu = torch.full((4, ops.scan_state_floats("delta_rule", H, dk, dv)), float("nan"), device=DEV)
    st_ref = torch.full((4, ref.scan_state_floats("delta_rule", H, dk, dv)), float("nan"))
    for n, (q_lens, slots, fresh, chunks) in enumerate(CALLS):
        T = sum(q_lens)
        # keys that resemble one another: the triangle inside a chunk is far from the identity
        qkv = torch.randn(T, C, generator=g)
        qk = qkv[:, :2 * G * dk].view(T, 2 * G, dk) + 0.5
        qkv[:, :2 * G * dk] = (qk / qk.norm(dim=-1, keepdim=True)).view(T, -1)
        ba = torch.randn(T, 2 * H, generator=g) * spread
        out_ref = torch.empty(T, H * dv)
        ref.delta_rule_scan(qkv, ba.clone(), a_log, dt_bias, st_ref, make_batch(q_lens, slots, fresh, "cpu"), H, G, dk, dv, out_ref)
        out = torch.full((T, H * dv), float("nan"), device=DEV)
        before = st_gpu.clone()
        ops.delta_rule_scan(qkv.to(DEV), ba.to(DEV), a_log.to(DEV), dt_bias.to(DEV), st_gpu,
                            make_batch(q_lens, slots, fresh, DEV), H, G, dk, dv, out, chunks=chunks)
        close(out, out_ref, 3e-5, f"call {n}")
        untouched = [s for s in range(4) if s not in slots]
        assert torch.equal(torch.nan_to_num(st_gpu[untouched], nan=7.0), torch.nan_to_num(before[untouched], nan=7.0))


@pytest.mark.parametrize("kind", ["memory", "delta"])
@pytest.mark.parametrize("gate", [0, 1])                 # input and forget gate; beta and decay
@pytest.mark.parametrize("at", [0, 20, 47])
def test_a_gate_that_is_no_number_stays_one(kind, gate, at):
    """From its token on, and in the state it leaves, as in the token-by-token scans; the chunks before it and the other head
    know nothing of it (tokens before it in its own chunk may: they share its products)."""
    ops = kernels.current()
    g = torch.Generator().manual_seed(at)
    H, dk, dv, T = 2, 64, 24, 50
    rows = torch.randn(T, 2 * H * dk + H * dv, generator=g) * 0.5
    gates = torch.randn(T, 2 * H, generator=g)
    gates[at, gate * H] = float("nan")
    found = []
    for chunks in (True, False):
        batch, out = make_batch([T], [0], [1], DEV), torch.zeros(T, H * dv, device=DEV)
        st = torch.zeros(1, ops.scan_state_floats("matrix_memory" if kind == "memory" else "delta_rule", H, dk, dv), device=DEV)
        more = [torch.full((n,), 0.1, device=DEV) for n in (2 * H, H, H)]
        if kind == "memory":
            ops.matrix_memory_scan(rows.to(DEV), 0, H * dk, 2 * H * dk, gates.to(DEV), more[0], st, batch, H, dk, dv, 15.0,
                                   dk ** -0.5, 1e-6, out, chunks=chunks)
        else:
            ops.delta_rule_scan(rows.to(DEV), gates.to(DEV), more[1], more[2], st, batch, H, H, dk, dv, out, chunks=chunks)
        found.append((torch.isnan(out).cpu().view(T, H, dv), torch.isnan(st).cpu()))
    (chunked, chunked_state), (single, single_state) = found
    assert torch.equal(chunked_state, single_state)
    assert single[at:, 0].all() and not single[:at].any() and chunked[at:, 0].all()
    assert not chunked[:at // 16 * 16].any() and not chunked[:, 1].any()


def test_errors_in_chunks_are_those_of_single_tokens():
    """Over gates from mild to vanishing, 400 tokens: the read-outs' errors in units of one rounding of their terms' sizes."""
    ops = kernels.current()
    for H, dk, dv in ((2, 128, 64), (1, 20, 12)):
        for spread, base in ((1.0, 3.0), (3.0, 0.0), (30.0, 0.0)):
            g = torch.Generator().manual_seed(dk)
            T, off = 400, (0, H * dk, 2 * H * dk)
            proj = (torch.randn(T, 2 * H * dk + H * dv, generator=g) * 0.7).to(torch.bfloat16)
            gates, bias = torch.randn(T, 2 * H, generator=g) * spread, torch.cat([torch.zeros(H), torch.full((H,), base)])
            want, size = matrix_memory(proj, *off, gates, bias, {}, make_batch([T], [0], [1], "cpu"), H, dk, dv, 15.0, 1e-6)
            errs = []
            for chunks in (True, False):
                out, st = torch.empty(T, H * dv, device=DEV), torch.zeros(1, ops.scan_state_floats("matrix_memory", H, dk, dv), device=DEV)
                ops.matrix_memory_scan(proj.to(DEV), *off, gates.to(DEV), bias.to(DEV), st, make_batch([T], [0], [1], DEV), H,
                                       dk, dv, 15.0, dk ** -0.5, 1e-6, out, chunks=chunks)
                errs.append(float(((out.double().cpu() - want) / (size * 2.0 ** -24 + 1e-30)).pow(2).mean().sqrt()))
            # both are sums of some thousands of independent roundings: their root mean squares are known to a few percent
            assert errs[0] <= 1.15 * errs[1], (H, dk, spread, errs)
