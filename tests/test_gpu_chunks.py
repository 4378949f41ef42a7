"""Recurrences over matrix states by chunks of 16 tokens (``csrc/delta_chunks.hip``) against the recurrences themselves in
64 bits, and beside the token-by-token kernels: the chunks are as far off as those (0.90 to 1.01 times over the states of 32
heads, single heads more or less by chance), which the bounds hold them to row by row and head by head."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EPS = 1e-5


def _rows(lengths):
    """int32 offsets of rows of these lengths; rows of one token come first, as in a step."""
    lengths = sorted(lengths, key=lambda n: n != 1)
    offsets = torch.zeros(len(lengths) + 1, dtype=torch.int32)
    offsets[1:] = torch.tensor(lengths).cumsum(0)
    return lengths, offsets, sum(n == 1 for n in lengths)


def _walk64(q, k, v, decay, beta, state):
    """``S <- diag(decay) S; u = beta (v - S^T k) (beta None: v); S <- S + k u^T; o = S^T q`` for one sequence; q, k
    [n, H, dk], v [n, H, dv], decay [n, H, dk], state [H, dk, dv], all 64-bit."""
    out = []
    for t in range(q.shape[0]):
        state = decay[t][:, :, None] * state
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - (state * k[t][:, :, None]).sum(1))
        state = state + k[t][:, :, None] * u[:, None, :]
        out.append((state * q[t][:, :, None]).sum(1))
    return torch.stack(out), state


def _over_rms(o):
    return o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS)


def _check(outs, states, want, want_states, offsets, heads, chunked=True):
    """``outs`` = (by chunks, walked): results within the rounding to bfloat16 and 32-bit sums of the 64-bit ones, and every
    row's state of every head as near as the walk's: one and a half times its distance (sums in another order) and two
    roundings.  ``heads``: a state row is [heads, ..]."""
    assert not bool(torch.isnan(outs[0].float()).any())
    for r in range(offsets.numel() - 1):
        at = slice(int(offsets[r]), int(offsets[r + 1]))
        scale = want[at].abs().max()
        assert (outs[0][at].double() - want[at]).abs().max() <= 2.0 ** -8 * scale + 2 * (outs[1][at].double() - want[at]).abs().max()
    truth = want_states.view(want_states.shape[0], heads, -1)
    err = [(s.double().view(truth.shape) - truth).norm(dim=-1) / truth.norm(dim=-1) for s in states]
    assert bool((err[0] <= 1.5 * err[1] + 2.0 ** -23).all()), err
    if chunked:  # (and they did go by chunks: sums in another order)
        assert not torch.equal(states[0], states[1])


LENGTHS = [[1, 1, 16, 1, 17, 33], [15, 1, 130, 31], [250], [2049 + 40]]


@pytest.mark.parametrize("rule", ["head", "channel", "plain"])
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("H,G,dk,dv", [(2, 1, 64, 24), (8, 8, 128, 16), (4, 4, 64, 130), (3, 3, 64, 130)])
def test_delta_rule_and_linear_attention_by_chunks(rule, lengths, H, G, dk, dv):
    """Rows that end inside a chunk, rows of single tokens before them, a row beyond a window of tokens; decays near one,
    decays that forget at once (and to zero exactly) beside them, in one channel or in all; a written key read back late.  Rows
    of an odd number of pairs (the last sizes) are walked."""
    from torchllms_amd.kernels import ops

    if rule == "plain":
        G = H
    lengths, offsets, singles = _rows(lengths)
    n = int(offsets[-1])
    g = torch.Generator().manual_seed(n + dk + dv)
    qkv = torch.randn((n, 2 * G * dk + H * dv), generator=g)
    qkv[n // 3, G * dk : 2 * G * dk] *= 6.0
    qkv[n - 1, : G * dk] = qkv[n // 3, G * dk : 2 * G * dk]
    qkv = qkv.bfloat16()
    a = torch.randn((n, H if rule == "head" else H * dk), generator=g) * 2 - 6.0
    a[n // 2] += 300.0 if rule != "plain" else -300.0  # everything is forgotten at one token
    a[:, ::5] += 9.0 if rule != "plain" else -9.0  # some heads or channels forget within a token or two
    if rule == "plain":
        a[:, 1::5] += 14.0
    b, gate = torch.randn((n, H), generator=g).bfloat16(), torch.randn((n, H * dv), generator=g).bfloat16()
    A_log, bias, norm_w = torch.rand(H, generator=g) * 2, torch.randn(a.shape[1], generator=g) * 0.5, torch.rand(dv, generator=g) + 0.5
    start = torch.randn((len(lengths), H * dv * dk), generator=g)
    slots = torch.randperm(len(lengths), generator=g).int()
    if rule == "head":
        a = a.bfloat16()
    size = (len(lengths), 4 + H * dv * dk)

    outs, states = [], []
    for longest in (max(lengths), 0):
        state = torch.zeros(size, device=DEV)
        state[:, 4:] = start.to(DEV)
        rows = (offsets.to(DEV), slots.to(DEV))
        if rule == "plain":
            out = ops.gated_linear(qkv.to(DEV), a.to(DEV), bias.to(DEV), 0.25, gate.to(DEV), 0, norm_w.to(DEV), EPS, state, 4, *rows, H, dk, dv,
                                   longest=longest, single_rows=singles)
        else:
            proj = torch.cat([b, a if rule == "head" else b], dim=1).to(DEV)
            out = ops.gated_delta(qkv.to(DEV), proj, 0, 0, H, A_log.to(DEV), bias.to(DEV), norm_w.to(DEV), EPS, state, 4, *rows, H, G, dk, dv,
                                  gate=gate.to(DEV), channel_decay=a.to(DEV) if rule == "channel" else None, longest=longest, single_rows=singles)
        outs.append(out.cpu())
        states.append(state[:, 4:].cpu())

    x = qkv.double()
    q, k, v = x[:, : G * dk].view(n, G, dk), x[:, G * dk : 2 * G * dk].view(n, G, dk), x[:, 2 * G * dk :].view(n, H, dv)
    q, k = (u.repeat_interleave(H // G, 1) for u in (q, k))
    pre = a.double() + bias.double()
    if rule == "plain":
        decay, beta = torch.sigmoid(pre).pow(0.25).view(n, H, dk), None
    else:
        q, k = (u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6) for u in (q, k))
        step = torch.nn.functional.softplus(pre, threshold=1e9).view(n, H, -1)
        decay, beta = torch.exp(-torch.exp(A_log.double())[:, None] * step).expand(n, H, dk), torch.sigmoid(b.double())
    q = q * dk ** -0.5
    want, want_states = torch.empty(n, H, dv, dtype=torch.float64), torch.empty(len(lengths), H * dv * dk, dtype=torch.float64)
    for r in range(len(lengths)):
        at = slice(int(offsets[r]), int(offsets[r + 1]))
        s0 = start[slots[r]].double().view(H, dv, dk).transpose(1, 2)
        want[at], last = _walk64(q[at], k[at], v[at], decay[at], None if beta is None else beta[at], s0)
        want_states[slots[r]] = last.transpose(1, 2).reshape(-1)
    want = (_over_rms(want) * norm_w.double()).reshape(n, -1) * torch.nn.functional.silu(gate.double())
    _check(outs, states, want, want_states, offsets, H, chunked=qkv.shape[1] % 4 == 0)


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("H,dk,dv", [(2, 64, 24), (8, 128, 16), (4, 64, 128), (3, 64, 128)])
def test_matrix_memory_by_chunks(lengths, H, dk, dv):
    """Input gates that jump above the running maximum inside a chunk and far below it, forget gates that drop everything,
    gates beyond the cap; the normaliser's column behind a full group of columns and inside one.  Rows of an odd number of
    pairs (the last sizes) are walked."""
    from torchllms_amd.kernels import ops

    lengths, offsets, singles = _rows(lengths)
    n, cap = int(offsets[-1]), 9.0
    g = torch.Generator().manual_seed(n + dk + dv)
    qk, vw = H * dk, H * dv
    proj = torch.randn((n, 2 * qk + 2 * vw + 2 * H), generator=g)
    gi, gf = proj[:, 2 * qk + 2 * vw : 2 * qk + 2 * vw + H], proj[:, 2 * qk + 2 * vw + H :]
    gi.mul_(3.0)
    gf.mul_(2.0).add_(4.0)
    gi[n // 2] = 30.0
    gi[n // 2 + 1 : n // 2 + 20] = -30.0
    gf[n // 4] = -40.0
    proj = proj.bfloat16()
    i_b, f_b, norm_w = torch.randn(H, generator=g), torch.randn(H, generator=g), torch.rand(vw, generator=g) + 0.5
    size = ops.matrix_memory_state_size(H, dk, dv)
    slots = torch.randperm(len(lengths), generator=g).int()
    outs, states = [], []
    for longest in (max(lengths), 0):
        state = torch.zeros((len(lengths), size + 4 - size % 4), device=DEV)
        out = ops.matrix_memory(proj.to(DEV), 0, qk, 2 * qk, 2 * qk + 2 * vw, 2 * qk + 2 * vw + H, 2 * qk + vw, i_b.to(DEV), f_b.to(DEV), cap,
                                norm_w.to(DEV), EPS, state, 0, offsets.to(DEV), slots.to(DEV), H, dk, dv, longest=longest, single_rows=singles)
        outs.append(out.cpu())
        states.append(state.cpu())

    x = proj.double()
    q, k = x[:, :qk].view(n, H, dk) * dk ** -0.5, x[:, qk : 2 * qk].view(n, H, dk)
    v = torch.cat([x[:, 2 * qk : 2 * qk + vw].view(n, H, dv), torch.ones(n, H, 1, dtype=torch.float64)], -1)
    i_g, f_g = (cap * torch.tanh((x[:, at : at + H] + bias.double()) / cap) for at, bias in ((2 * qk + 2 * vw, i_b), (2 * qk + 2 * vw + H, f_b)))
    f_g = torch.nn.functional.logsigmoid(f_g)
    want, matrices = torch.empty(n, H, dv, dtype=torch.float64), torch.empty(len(lengths), H * (dv + 1) * dk, dtype=torch.float64)
    tops = torch.empty(len(lengths), H, dtype=torch.float64)
    for r in range(len(lengths)):
        m, keep, take, ms = torch.zeros(H, dtype=torch.float64), [], [], []
        for t in range(int(offsets[r]), int(offsets[r + 1])):
            new = torch.maximum(f_g[t] + m, i_g[t])
            keep.append(torch.exp(f_g[t] + m - new))
            take.append(torch.exp(i_g[t] - new))
            m = new
            ms.append(new)
        at = slice(int(offsets[r]), int(offsets[r + 1]))
        o, last = _walk64(q[at], k[at] * torch.stack(take)[..., None], v[at], torch.stack(keep)[..., None].expand(-1, H, dk), None,
                          torch.zeros(H, dk, dv + 1, dtype=torch.float64))
        want[at] = o[..., :dv] / (torch.maximum(o[..., dv].abs(), torch.exp(-torch.stack(ms))) + 1e-6)[..., None]
        matrices[slots[r]] = last.transpose(1, 2).reshape(-1)
        tops[slots[r]] = m
    want = _over_rms(want).reshape(n, -1) * norm_w.double() * torch.sigmoid(x[:, 2 * qk + vw : 2 * qk + 2 * vw])
    _check(outs, [s[:, : H * (dv + 1) * dk] for s in states], want, matrices, offsets, H, chunked=proj.shape[1] % 4 == 0)
    for s in states:
        top = s[:, H * (dv + 1) * dk : H * (dv + 1) * (dk + 1)].view(len(lengths), H, dv + 1).double()
        assert bool(((top - tops[..., None]).abs() <= 1e-5 * (1 + tops[..., None].abs())).all())


@pytest.mark.parametrize("what", ["q", "k", "v"])
@pytest.mark.parametrize("rule", ["head", "channel", "plain", "memory"])
def test_a_token_that_is_not_finite_spoils_no_earlier_one(rule, what):
    """An infinity in a query, key or value at the start, in the middle and at the end of a chunk, of one head of one request:
    earlier tokens, the other head and the other requests keep their bits; from it on, and in the states, the same places
    are finite as in the token-by-token walk."""
    from torchllms_amd.kernels import ops

    H, dk, dv, lengths = 2, 64, 24, [1, 40, 50, 17]
    offsets = torch.tensor([0] + lengths).cumsum(0).int()
    n, rows = int(offsets[-1]), len(lengths)
    g = torch.Generator().manual_seed(7)
    qk, vw = H * dk, H * dv
    data = torch.randn((n, 2 * qk + 2 * vw + 2 * H), generator=g).bfloat16()  # queries, keys, values, gate, two gates a head
    a = torch.randn((n, H * dk), generator=g) - 4.0
    A_log, bias, norm_w = torch.rand(H, generator=g), torch.randn(H * dk, generator=g) * 0.5, torch.rand(vw, generator=g) + 0.5
    per = ops.matrix_memory_state_size(H, dk, dv) if rule == "memory" else H * dv * dk
    start = torch.randn((rows, per + -per % 4), generator=g)
    if rule == "memory":
        start.zero_()
    where = (offsets.to(DEV), torch.arange(rows, dtype=torch.int32, device=DEV))

    def run(x, longest):
        state, x = start.to(DEV), x.to(DEV)
        kw = dict(longest=longest, single_rows=1)
        if rule == "memory":
            out = ops.matrix_memory(x, 0, qk, 2 * qk, 2 * qk + 2 * vw, 2 * qk + 2 * vw + H, 2 * qk + vw, bias[:H].to(DEV), bias[H : 2 * H].to(DEV),
                                    9.0, norm_w.to(DEV), EPS, state, 0, *where, H, dk, dv, **kw)
        elif rule == "plain":
            out = ops.gated_linear(x[:, : 2 * qk + vw], a.to(DEV), bias.to(DEV), 0.25, x, 2 * qk + vw, norm_w[:dv].to(DEV), EPS, state, 0, *where, H, dk, dv, **kw)
        else:
            out = ops.gated_delta(x[:, : 2 * qk + vw], x, 2 * qk + vw, 2 * qk + 2 * vw, 2 * qk + 2 * vw + H, A_log.to(DEV),
                                  (bias if rule == "channel" else bias[:H]).to(DEV), norm_w[:dv].to(DEV), EPS, state, 0, *where, H, H, dk, dv,
                                  channel_decay=a.to(DEV) if rule == "channel" else None, **kw)
        return out.cpu().float(), state.cpu()

    clean, clean_state = run(data, max(lengths))
    assert bool(torch.isfinite(clean).all())
    for place in (16, 21, 31, 39):  # of the second row, tokens 1 .. 40
        at = 1 + place
        x = data.clone()
        x[at, {"q": 0, "k": qk, "v": 2 * qk}[what] + 5] = float("inf")  # of head 0
        out, state = run(x, max(lengths))
        walked, walked_state = run(x, 0)
        spoiled = torch.zeros(n, vw, dtype=torch.bool)
        spoiled[at : at + 1 if what == "q" else 41, :dv] = True
        assert torch.equal(out[~spoiled], clean[~spoiled])
        assert torch.equal(torch.isfinite(out), torch.isfinite(walked)) and not bool(torch.isfinite(out[at, :dv]).all())
        assert torch.equal(torch.isfinite(state), torch.isfinite(walked_state))
        assert torch.equal(state[[0, 2, 3]], clean_state[[0, 2, 3]])
