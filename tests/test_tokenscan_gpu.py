"""The exact fp32 token scan (ops.nsgdn_scan: archbench::nsgdn_fwd / nsgdn_bwd, nsgdn.py:80-216) against the
oracle's token recurrence (oracle/nsgdn_oracle.py::recurrent_fwd / recurrent_bwd, fp64 on the CPU): y and every
gradient (dq, dk, du, dv, dla) at fp32 accuracy -- max-abs error <= 1e-4 for y and rel-L2 <= 1e-6 for y and each
gradient, the achieved errors printed -- over K in {64, 128}, V below, at and above one 64-row block (96: a
partial block), T around the 32-token checkpoint interval and the backward's 4-token groups (1, 31, 32, 33, 45, 100)
and over 32 checkpoint chunks (1024), B and H > 1."""

import pytest
import torch
import torch.nn.functional as F

from archbench_amd import ops
from oracle import nsgdn_oracle as NS
from tests.gpu_util import banner, max_abs, rel_l2

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, K, V, seed):
    g = torch.Generator().manual_seed(seed)
    q = F.normalize(torch.randn(B, T, H, K, generator=g), dim=-1) * K ** -0.5
    k = F.normalize(torch.randn(B, T, H, K, generator=g), dim=-1)
    u = k * torch.rand(B, T, H, 1, generator=g) + 0.1 * torch.randn(B, T, H, K, generator=g) / K ** 0.5
    v = torch.randn(B, T, H, V, generator=g)
    la = -F.softplus(torch.randn(B, T, H, generator=g)) * 0.5
    dy = torch.randn(B, T, H, V, generator=g)
    return q, k, u, v, la, dy


CASES = [  # B, T, H, K, V
    (2, 100, 2, 64, 64),
    (1, 33, 3, 128, 128),
    (2, 32, 2, 128, 256),
    (1, 31, 2, 64, 96),
    (3, 1, 2, 128, 64),
    (1, 45, 2, 64, 64),
    (1, 1024, 1, 128, 64),
]


@pytest.mark.parametrize("B,T,H,K,V", CASES)
def test_token_scan_matches_recurrence(B, T, H, K, V):
    banner(f"token scan B={B} T={T} H={H} K={K} V={V}")
    q, k, u, v, la, dy = _inputs(B, T, H, K, V, seed=B * 100 + T + K + V)
    leaves = [t.cuda().requires_grad_() for t in (q, k, u, v, la)]
    y = ops.nsgdn_scan(*leaves)
    y.backward(dy.cuda())
    torch.cuda.synchronize()
    y_ref, _ = NS.recurrent_fwd(q, k, u, v, la)
    grads_ref = NS.recurrent_bwd(q, k, u, v, la, dy)[:5]
    assert y.dtype == torch.float32
    errs = {"y": (max_abs(y, y_ref), rel_l2(y, y_ref))}
    for n, t, gr in zip(("dq", "dk", "du", "dv", "dla"), leaves, grads_ref):
        errs[n] = (max_abs(t.grad, gr), rel_l2(t.grad, gr))
    print("[max-abs, rel-L2] " + ", ".join(f"{n} {a:.1e} {r:.1e}" for n, (a, r) in errs.items()), flush=True)
    assert errs["y"][0] <= 1e-4
    for n, (a, r) in errs.items():
        assert r <= 1e-6, (n, r)


def test_token_scan_edges():
    banner("token scan: empty batch, unsupported K, shape errors")
    q, k, u, v, la, _ = _inputs(1, 8, 2, 64, 64, seed=1)
    d = [t.cuda() for t in (q, k, u, v, la)]
    e = ops.nsgdn_scan(*(t[:0] for t in d))
    assert e.shape == (0, 8, 2, 64)
    with pytest.raises(ValueError, match="K=96"):
        z = torch.zeros(1, 8, 2, 96, device="cuda")
        ops.nsgdn_scan(z, z, z, d[3], d[4])
    with pytest.raises(ValueError, match="la"):
        ops.nsgdn_scan(d[0], d[1], d[2], d[3], d[4][:, :4])


def test_gdn_op_fp32_k128_runs_exact_token_scan(monkeypatch):
    """chunk_gated_delta_rule with fp32 inputs at K = 128 (no fp32 chunk kernels there) runs the token scan with
    u = beta k: o, the final state and every gradient including dh0 (with a final-state gradient) against the gated
    delta rule oracle (fp64), rel-L2 <= 1e-6; T = 0 returns the initial state."""
    from oracle import gdn_oracle as O
    banner("gdn op fp32 K=128 V=256 through the token scan, with h0 / hT")
    monkeypatch.setattr(ops, "_TOKEN_ROUTE_WARNED", [False])
    B, T, H, K, V = 2, 70, 2, 128, 256
    g_ = torch.Generator().manual_seed(12)
    q = F.normalize(torch.randn(B, T, H, K, generator=g_), dim=-1)
    k = F.normalize(torch.randn(B, T, H, K, generator=g_), dim=-1)
    v = torch.randn(B, T, H, V, generator=g_)
    g = F.logsigmoid(torch.randn(B, T, H, generator=g_) + 3)
    beta = torch.rand(B, T, H, generator=g_)
    h0 = torch.randn(B, H, K, V, generator=g_) * 0.1
    do = torch.randn(B, T, H, V, generator=g_)
    dhT = torch.randn(B, H, K, V, generator=g_) * 0.1
    leaves = [t.cuda().requires_grad_() for t in (q, k, v, g, beta, h0)]
    with pytest.warns(UserWarning, match="token scan"):
        o, hT = ops.chunk_gated_delta_rule(*leaves[:5], scale=0.5, initial_state=leaves[5], output_final_state=True)
    torch.autograd.backward((o, hT), (do.cuda(), dhT.cuda()))
    o_ref, hT_ref = O.chunk_fwd(q, k, v, g, beta, 0.5, h0)
    grads_ref = O.chunk_bwd(q, k, v, g, beta, do, 0.5, h0, dhT)
    errs = {"o": rel_l2(o, o_ref), "hT": rel_l2(hT, hT_ref)}
    for n, t, gr in zip(("dq", "dk", "dv", "dg", "dbeta", "dh0"), leaves, grads_ref):
        errs[n] = rel_l2(t.grad, gr)
    print("[rel-L2] " + ", ".join(f"{n} {e:.1e}" for n, e in errs.items()), flush=True)
    for n, e in errs.items():
        assert e <= 1e-6, (n, e)
    o0, hT0 = ops.chunk_gated_delta_rule(*(t[:, :0].detach() for t in leaves[:5]), scale=0.5,
                                         initial_state=leaves[5].detach(), output_final_state=True)
    assert o0.shape == (B, 0, H, V) and torch.equal(hT0, leaves[5].detach())


def test_token_scan_is_deterministic():
    """Row sums are added in a fixed order (no atomics): two runs of the forward and backward on the same inputs agree
    bit for bit, at a shape with several 64-row blocks, checkpoint chunks and a short last group."""
    banner("token scan determinism B=2 T=77 H=3 K=128 V=192")
    q, k, u, v, la, dy = (t.cuda() for t in _inputs(2, 77, 3, 128, 192, seed=5))
    runs = []
    for _ in range(2):
        y, r, st, _ = ops.nsgdn_token_fwd(q, k, u, v, la, None, False)
        grads = ops.nsgdn_token_bwd(q, k, u, la, r, st, dy, None, False)
        runs.append([y, r] + [g for g in grads if g is not None])
    torch.cuda.synchronize()
    for a, b in zip(*runs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,T,H,V,rows", [(1, 3, 1, 1, 16), (2, 70, 3, 17, 16), (1, 36, 2, 49, 16), (64, 9, 2, 56, 32),
                                          (85, 33, 1, 96, 32), (86, 33, 1, 96, 64), (128, 3, 2, 64, 64),
                                          (64, 37, 1, 256, 64), (64, 8, 4, 124, 64)])
@pytest.mark.parametrize("K", [64, 128])
def test_token_scan_row_blocks(B, T, H, V, rows, K):
    """16, 32 and 64 rows per workgroup (by the rounds over 256 CUs): full and partial row blocks, tokens
    that end inside a group, a block and a checkpoint chunk, with initial and final states and their gradients.  The
    bound is test_token_scan_matches_recurrence's, 1e-6: fp32 sums of at most 128 products of operands of order 1 (2^-24
    per step, decayed over the tokens)."""
    banner(f"token scan rows {rows}: B={B} T={T} H={H} K={K} V={V}")
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        nb = ops._token_sizes(ops._lib.load(), B, T, H, K, V)[2]
        assert nb == -(-V // rows), nb
    q, k, u, v, la, dy = _inputs(B, T, H, K, V, seed=B + T + K + V)
    g = torch.Generator().manual_seed(7)
    h0, dhT = (0.1 * torch.randn(B, H, K, V, generator=g) for _ in range(2))
    d = [t.cuda() for t in (q, k, u, v, la, dy, h0, dhT)]
    y, r, st, hT = ops.nsgdn_token_fwd(*d[:5], d[6], True)
    dq, dk, du, dv, dla, dh0 = ops.nsgdn_token_bwd(d[0], d[1], d[2], d[4], r, st, d[5], d[7], True)
    y_ref, hT_ref = NS.recurrent_fwd(q, k, u, v, la, h0=h0)
    ref = NS.recurrent_bwd(q, k, u, v, la, dy, h0=h0, dhT=dhT)
    errs = {n: rel_l2(a, b) for n, a, b in zip(("y", "hT", "dq", "dk", "du", "dv", "dla", "dh0"),
                                               (y, hT, dq, dk, du, dv, dla, dh0), (y_ref, hT_ref) + tuple(ref))}
    print("[rel-L2] " + ", ".join(f"{n} {e:.1e}" for n, e in errs.items()), flush=True)
    for n, e in errs.items():
        assert e <= 1e-6, (n, e)


@pytest.mark.parametrize("B,T,H,V,rows", [(1, 256, 2, 17, 16), (2, 257, 2, 1, 16), (3, 290, 1, 100, 16),
                                          (4, 199, 4, 250, 64), (17, 300, 1, 256, 64)])
@pytest.mark.parametrize("K", [64, 128])
def test_token_scan_split_backward(B, T, H, V, rows, K):
    """The backward with the state gradient's recurrence in its own launch (16 and 32 rows per workgroup) and the chunks
    in parallel (16 and 64 rows, more chunks than workgroups in the larger ones): whole and partial row blocks, last chunks
    of 1 to 32 tokens, with and without states.  The bound is test_token_scan_row_blocks's."""
    banner(f"token scan split backward rows {rows}: B={B} T={T} H={H} K={K} V={V}")
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        st_bytes, sc_bytes, nb = ops._token_sizes(ops._lib.load(), B, T, H, K, V)
        assert nb == -(-V // rows), nb
        wgs = min(B * H * nb * -(-T // 32), 512 if rows == 16 else 256)
        assert sc_bytes == -(-st_bytes // 16) * 16 + wgs * 8 * K * rows * 4
    q, k, u, v, la, dy = _inputs(B, T, H, K, V, seed=B + T + K + V)
    g = torch.Generator().manual_seed(7)
    h0, dhT = (0.1 * torch.randn(B, H, K, V, generator=g) for _ in range(2))
    d = [t.cuda() for t in (q, k, u, v, la, dy, h0, dhT)]
    y, r, st, _ = ops.nsgdn_token_fwd(*d[:5], d[6], True)
    got = ops.nsgdn_token_bwd(d[0], d[1], d[2], d[4], r, st, d[5], d[7], True)
    assert all(torch.equal(a, b) for a, b in
               zip(got, ops.nsgdn_token_bwd(d[0], d[1], d[2], d[4], r, st, d[5], d[7], True)))
    ref = NS.recurrent_bwd(q, k, u, v, la, dy, h0=h0, dhT=dhT)
    _, r0, st0, _ = ops.nsgdn_token_fwd(*d[:5], None, False)
    got0 = ops.nsgdn_token_bwd(d[0], d[1], d[2], d[4], r0, st0, d[5], None, False)[:5]
    ref0 = NS.recurrent_bwd(q, k, u, v, la, dy)[:5]
    names = ("dq", "dk", "du", "dv", "dla", "dh0")
    errs = {n: rel_l2(a, b) for n, a, b in zip(names, got, ref)}
    errs.update({n + " (no states)": rel_l2(a, b) for n, a, b in zip(names, got0, ref0)})
    print("[rel-L2] " + ", ".join(f"{n} {e:.1e}" for n, e in errs.items()), flush=True)
    for n, e in errs.items():
        assert e <= 1e-6, (n, e)


@pytest.mark.parametrize("T", [1, 9, 12, 31])
def test_infinite_state_at_a_ragged_end(T):
    """A state that overflows at the last token is returned as it is, infinite where it overflowed, also where the
    sequence ends inside a block of tokens (whose padding must not turn it into NaN)."""
    B, H, K, V = 1, 2, 64, 40
    banner(f"token scan infinite state T={T}")
    q, k, u = (torch.zeros(B, T, H, K, device="cuda") for _ in range(3))
    v, la = torch.zeros(B, T, H, V, device="cuda"), torch.zeros(B, T, H, device="cuda")
    q[:, -1], u[:, -1, :, 0], v[:, -1] = 1.0, 4.0, 3e38
    y, r, _, hT = ops.nsgdn_token_fwd(q, k, u, v, la, None, True)
    assert torch.isinf(hT[:, :, 0]).all() and not hT[:, :, 1:].any()
    assert torch.isinf(y[:, -1]).all() and (r[:, -1] == v[:, -1]).all()
    if T > 8:  # beside the infinite rows (the first 16 are one workgroup's), ordinary ones keep their values
        q, k, u, v0, la, _ = (t.cuda() for t in _inputs(B, T, H, K, V, seed=T))
        ref = ops.nsgdn_token_fwd(q, k, u, v0, la, None, True)[3]
        v = v0.clone()
        v[:, -1, :, 5] = float("inf")
        hT = ops.nsgdn_token_fwd(q, k, u, v, la, None, True)[3]
        keep = [i for i in range(V) if i != 5]
        assert torch.equal(hT[..., keep], ref[..., keep]) and torch.isinf(hT[..., 5]).all()
