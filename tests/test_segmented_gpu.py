"""Segmented sweeps on the GPU: with few (b, h) and a long sequence the library cuts each sequence into segments
of whole chunks (T = 4096 with one or two heads gives four segments of 1024 tokens), sweeps them in parallel from
a prefix pass (each segment's state from zero and its transition) and a scan across segments, and mirrors this in
the backward with the transposed transitions.  Every path that segments is checked against the fp64 oracle on
the same rounded inputs: the training pair with initial state and final-state gradient (bf16, rel-L2 <= 1e-2),
the recompute backward and the plain forward in fp32 (max-abs <= 1e-4), the separate-write-key variant, and the
segmented forward against the unsegmented allocation-free forward.  The event timer confirms the prefix pass and
the scans ran."""

import ctypes

import pytest
import torch

from archbench_amd import _lib, ops
from oracle import gdn_oracle as O
from oracle import nsgdn_oracle as NSO
from tests.gpu_util import assert_fp32_close, banner, device_inputs, rel_l2

pytestmark = pytest.mark.gpu
NAMES = ["dq", "dk", "dv", "dg", "dbeta", "dh0"]


@pytest.mark.parametrize("K,V", [(128, 128), (64, 256)])
def test_training_pair_segmented(K, V):
    B, T, H = 1, 4096, 2
    banner(f"segmented training pair B={B} T={T} H={H} K={K} V={V} bf16")
    host, dev = device_inputs(B, T, H, K, V, torch.bfloat16, seed=41, h0_std=0.1, with_do=True)
    dhT = torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(42)) * 0.1
    with _lib.StageTimer() as st:
        o, hT, stash = ops.chunk_fwd_stash(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, 0.8)
        got = ops.chunk_bwd_stashed(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, dev.do, dhT.cuda(), stash, 0.8)
    torch.cuda.synchronize()
    assert {"prefix", "seg_scan", "bwd_local"} <= set(st.result), st.result
    assert st.result["seg_scan"][1] == 2  # one scan forward, one backward
    o_r, hT_r = O.chunk_fwd(host.q, host.k, host.v, host.g, host.beta, 0.8, host.h0)
    ref = O.chunk_bwd(host.q, host.k, host.v, host.g, host.beta, host.do, 0.8, host.h0, dhT)
    errs = {"o": rel_l2(o, o_r), "hT": rel_l2(hT, hT_r)}
    errs.update({n: rel_l2(a, b) for n, a, b in zip(NAMES, got, ref)})
    print(f"[segmented K={K} V={V}] rel-L2 " + ", ".join(f"{n} {e:.2e}" for n, e in errs.items()), flush=True)
    assert all(e <= 1e-2 for e in errs.values()), errs


def test_fp32_forward_and_recompute_backward_segmented():
    B, T, H, K, V = 1, 4096, 1, 64, 64
    banner(f"segmented fp32 forward + recompute backward B={B} T={T} H={H} K={K} V={V}")
    host, dev = device_inputs(B, T, H, K, V, torch.float32, seed=43, h0_std=0.1, with_do=True)
    dhT = torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(44)) * 0.1
    with _lib.StageTimer() as st:
        o, hT = ops.chunk_fwd(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, 0.5)
        got = ops.chunk_bwd(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, dev.do, dhT.cuda(), 0.5)
    torch.cuda.synchronize()
    assert st.result["prefix"][1] == 2 and st.result["seg_scan"][1] == 3, st.result
    o_r, hT_r = O.chunk_fwd(host.q, host.k, host.v, host.g, host.beta, 0.5, host.h0)
    ref = O.chunk_bwd(host.q, host.k, host.v, host.g, host.beta, host.do, 0.5, host.h0, dhT)
    assert_fp32_close("segmented fp32", ["o", "hT", *NAMES], [o, hT, *got], [o_r, hT_r, *ref], 1e-4)


def test_segmented_forward_matches_unsegmented():
    """gdn_chunk_fwd segments this shape; the allocation-free forward never does: same result to the bf16 bar."""
    B, T, H, K, V = 2, 4096, 1, 128, 128
    banner(f"segmented vs unsegmented forward B={B} T={T} H={H} K={K} V={V} bf16")
    _, dev = device_inputs(B, T, H, K, V, torch.bfloat16, seed=45, h0_std=0.1)
    o, hT = ops.chunk_fwd(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, 1.0)
    o2, hT2 = torch.empty_like(o), torch.empty_like(hT)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = _lib.load().gdn_chunk_fwd_noalloc(p(dev.q), p(dev.k), p(dev.v), p(dev.g), p(dev.beta), p(dev.h0), p(o2),
                                           p(hT2), B, T, H, K, V, 1.0, _lib.DTYPE_BF16, _lib.stream_ptr(o.device))
    _lib.check(rc, "gdn_chunk_fwd_noalloc")
    torch.cuda.synchronize()
    assert rel_l2(o, o2) <= 1e-2 and rel_l2(hT, hT2) <= 1e-2, (rel_l2(o, o2), rel_l2(hT, hT2))


@pytest.mark.parametrize("with_states", [True, False])
def test_nsgdn_segmented(with_states):
    B, T, H, K, V = 1, 4096, 2, 128, 128
    banner(f"segmented nsgdn B={B} T={T} H={H} K={K} V={V} bf16, S0 and dS given: {with_states}")
    gen = torch.Generator().manual_seed(46)
    r = lambda *s: torch.randn(*s, generator=gen)
    bf = torch.bfloat16
    q = (torch.nn.functional.normalize(r(B, T, H, K), dim=-1) * K ** -0.5).to(bf).float()
    k = torch.nn.functional.normalize(r(B, T, H, K), dim=-1).to(bf).float()
    beta = torch.sigmoid(r(B, T, H))
    u = (beta[..., None] * k + 0.05 * r(B, T, H, K)).to(bf).float()
    v = r(B, T, H, V).to(bf).float()
    la = torch.nn.functional.logsigmoid(r(B, T, H) + 4)
    dy = r(B, T, H, V).to(bf).float()
    S0, dS = 0.1 * r(B, H, K, V), 0.1 * r(B, H, K, V)
    if not with_states:  # without them the prefix starts from zero and the reverse scan from a zero gradient
        S0, dS = None, None
    d = lambda t, dt=bf: None if t is None else t.to("cuda", dt)
    with _lib.StageTimer() as st:
        y, hT, stash = ops.nsgdn_chunk_fwd(d(q), d(k), d(u), d(v), d(la, torch.float32), d(S0, torch.float32), 1.0)
        grads = ops.nsgdn_chunk_bwd(d(q), d(k), d(u), d(v), d(la, torch.float32), d(S0, torch.float32), d(dy),
                                    d(dS, torch.float32), stash, 1.0)
    torch.cuda.synchronize()
    assert "prefix" in st.result and "bwd_local" in st.result, st.result
    y_r, hT_r = NSO.chunk_fwd(q, k, u, v, la, 1.0, S0)
    ref = NSO.recurrent_bwd(q, k, u, v, la, dy, 1.0, S0, dS)
    errs = {"y": rel_l2(y, y_r), "hT": rel_l2(hT, hT_r)}
    errs.update({n: rel_l2(g, rr) for n, g, rr in zip(("dq", "dk", "du", "dv", "dla", "dh0"), grads, ref)
                 if rr is not None})  # (the oracle gives no dh0 without an initial state)
    print("[segmented nsgdn] rel-L2 " + ", ".join(f"{n} {e:.2e}" for n, e in errs.items()), flush=True)
    assert all(e <= 1e-2 for e in errs.values()), errs


@pytest.mark.parametrize("with_h0, with_dhT", [(False, False), (False, True), (True, False)])
def test_segmented_batch_without_states(with_h0, with_dhT):
    """Two sequences of four segments each.  The main sweeps write hT from each sequence's last segment and dh0
    from its first, at the sequence's own index; without h0 the first segment's transition is never built (the
    scan starts from zero), and without dhT the reverse scan does.  Every output against the fp64 oracle."""
    B, T, H, K, V = 2, 4096, 1, 128, 128
    banner(f"segmented training pair B={B} T={T} H={H} K={K} V={V} bf16, h0={with_h0} dhT={with_dhT}")
    host, dev = device_inputs(B, T, H, K, V, torch.bfloat16, seed=47, h0_std=0.1 if with_h0 else None,
                              with_do=True)
    dhT = torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(48)) * 0.1 if with_dhT else None
    with _lib.StageTimer() as st:
        o, hT, stash = ops.chunk_fwd_stash(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, 1.0)
        got = ops.chunk_bwd_stashed(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, dev.do,
                                    None if dhT is None else dhT.cuda(), stash, 1.0)
    torch.cuda.synchronize()
    assert {"prefix", "seg_scan", "bwd_local"} <= set(st.result), st.result
    o_r, hT_r = O.chunk_fwd(host.q, host.k, host.v, host.g, host.beta, 1.0, host.h0)
    ref = O.chunk_bwd(host.q, host.k, host.v, host.g, host.beta, host.do, 1.0, host.h0, dhT)
    errs = {"o": rel_l2(o, o_r), "hT": rel_l2(hT, hT_r)}
    errs.update({n: rel_l2(a, b) for n, a, b in zip(NAMES, got, ref)})
    print("[segmented batch] rel-L2 " + ", ".join(f"{n} {e:.2e}" for n, e in errs.items()), flush=True)
    assert all(e <= 1e-2 for e in errs.values()), errs


@pytest.mark.parametrize("B,T,H,K,V,dtype", [
    (1, 1025, 2, 64, 64, torch.bfloat16),    # the last segment is one chunk of one token
    (1, 1985, 2, 128, 128, torch.bfloat16),  # the last chunk one token; states kept for every second chunk
    (2, 1601, 1, 64, 64, torch.bfloat16),    # a ragged last chunk; a short last segment
    (1, 2111, 3, 128, 256, torch.bfloat16),  # every state stored; heads not a multiple of the XCDs
    (1, 1090, 1, 64, 128, torch.float32),
])
def test_segments_of_any_length(B, T, H, K, V, dtype):
    """A sequence of any length is segmented (the last segment shorter, its last chunk ragged): output, final state
    and every gradient against the fp64 oracle, at the bars of the equal segments above."""
    banner(f"segments of any length B={B} T={T} H={H} K={K} V={V} {dtype}")
    host, dev = device_inputs(B, T, H, K, V, dtype, seed=50, h0_std=0.1, with_do=True)
    dhT = torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(51)) * 0.1
    with _lib.StageTimer() as st:
        o, hT, stash = ops.chunk_fwd_stash(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, 0.7)
        got = ops.chunk_bwd_stashed(dev.q, dev.k, dev.v, dev.g, dev.beta, dev.h0, dev.do, dhT.cuda(), stash, 0.7)
    torch.cuda.synchronize()
    assert {"prefix", "seg_scan", "bwd_local"} <= set(st.result), st.result
    o_r, hT_r = O.chunk_fwd(host.q, host.k, host.v, host.g, host.beta, 0.7, host.h0)
    ref = O.chunk_bwd(host.q, host.k, host.v, host.g, host.beta, host.do, 0.7, host.h0, dhT)
    if dtype == torch.float32:
        assert_fp32_close("segments of any length", ["o", "hT", *NAMES], [o, hT, *got], [o_r, hT_r, *ref], 1e-4)
        return
    errs = {"o": rel_l2(o, o_r), "hT": rel_l2(hT, hT_r)}
    errs.update({n: rel_l2(a, b) for n, a, b in zip(NAMES, got, ref)})
    print("[segments of any length] rel-L2 " + ", ".join(f"{n} {e:.2e}" for n, e in errs.items()), flush=True)
    assert all(e <= 1e-2 for e in errs.values()), errs


def test_fp32_segments_add_no_error():
    """In fp32 the scan across segments sums each product as a tree, so cutting a sequence (here into segments of four
    chunks) puts its results no further from 64 bits than sweeping it whole does, as a batch too large to be cut is
    (sums in two chains put o, dq and dv 0.7% further; the bound is 0.3%)."""
    B, n, T, H, K, V = 65, 8, 2048, 1, 64, 64
    banner(f"segmented fp32 errors B={n} T={T} H={H} K={K} V={V}")
    host, dev = device_inputs(B, T, H, K, V, torch.float32, seed=63, with_do=True)

    def run(m):
        q, k, v, g, beta, do = (t[:m].contiguous() for t in (dev.q, dev.k, dev.v, dev.g, dev.beta, dev.do))
        with _lib.StageTimer() as st:
            o, _, stash = ops.chunk_fwd_stash(q, k, v, g, beta, None, 1.0)
            got = ops.chunk_bwd_stashed(q, k, v, g, beta, None, do, None, stash, 1.0)
        torch.cuda.synchronize()
        return ("seg_scan" in st.result), [t[:n] for t in (o, *got[:3])]

    (cut, seg), (whole_cut, whole) = run(n), run(B)
    assert cut and not whole_cut
    h = [t[:n] for t in (host.q, host.k, host.v, host.g, host.beta)]
    o_r, _ = O.chunk_fwd(*h, 1.0, None)
    ref = [o_r, *O.chunk_bwd(*h, host.do[:n], 1.0, None)[:3]]
    for name, a, b, r in zip(("o", "dq", "dk", "dv"), seg, whole, ref):
        ea, eb = rel_l2(a.double().cpu(), r.double()), rel_l2(b.double().cpu(), r.double())
        print(f"[segmented fp32] {name}: {ea:.4e} cut, {eb:.4e} whole", flush=True)
        assert ea <= 1.003 * eb, name


@pytest.mark.parametrize("K,V,sep", [(64, 64, False), (64, 128, False), (64, 64, True), (64, 256, True),
                                     (128, 128, True), (128, 256, True)])
def test_narrow_sweep_blocks_equal_wide(K, V, sep):
    """fp32 and separate-write-key sweeps in 32-column blocks (a grid that fits the 256 CUs) and in 64-column ones (one
    that does not): a column's arithmetic is the same in both, so a sequence alone equals itself in the batch bit for
    bit.  (Their agreement with the oracle: the tests above and those of each op.)"""
    T, H = 100, 2
    B = 256 * 32 // (V * H) + 1  # one sequence past the narrow grid's limit
    banner(f"narrow and wide sweep blocks B={B} T={T} H={H} K={K} V={V} separate write keys {sep}")
    dt = torch.bfloat16 if sep else torch.float32
    _, d = device_inputs(B, T, H, K, V, dt, seed=61, h0_std=0.1, with_do=True)
    dhT = 0.1 * torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(62)).cuda()
    u = (d.k.float() * d.beta.float()[..., None]).to(dt)

    def run(n):
        q, k, v, g, beta, h0, do, dh, uu = (t[:n].contiguous() for t in (d.q, d.k, d.v, d.g, d.beta, d.h0, d.do, dhT, u))
        if sep:
            o, hT, stash = ops.nsgdn_chunk_fwd(q, k, uu, v, g, h0, 0.5)
            return (o, hT) + tuple(ops.nsgdn_chunk_bwd(q, k, uu, v, g, h0, do, dh, stash, 0.5))
        o, hT = ops.chunk_fwd(q, k, v, g, beta, h0, 0.5)
        _, _, stash = ops.chunk_fwd_stash(q, k, v, g, beta, h0, 0.5)
        return (o, hT) + tuple(ops.chunk_bwd(q, k, v, g, beta, h0, do, dh, 0.5)) + tuple(
            ops.chunk_bwd_stashed(q, k, v, g, beta, h0, do, dh, stash, 0.5))

    wide, narrow = run(B), run(1)
    torch.cuda.synchronize()
    for a, b in zip(wide, narrow):
        assert torch.isfinite(b.float()).all() and torch.equal(a[:1], b)
