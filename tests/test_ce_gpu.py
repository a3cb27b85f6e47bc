"""Cross-entropy kernel and the fused linear + cross-entropy on the GPU against oracle/ce_oracle.py: per-row
loss and logsumexp (fp32 arithmetic: relative error <= 1e-5), the in-place gradient (fp32 max-abs <= 1e-4
relative, bf16 rel-L2 <= 1e-2), ignored rows, invalid targets, vocabularies up to 65536, and the whole op (loss,
dx, dW) over several chunkings."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from archbench_amd import fused_ce, ops
from oracle import ce_oracle as CE
from tests.gpu_util import banner, max_abs, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("N,V", [(1, 8), (33, 1000), (64, 50304), (5, 65536), (17, 8200)])
def test_ce_kernel_matches_oracle(dtype, N, V):
    banner(f"cross entropy N={N} V={V} {dtype}")
    gen = torch.Generator().manual_seed(V + N)
    x = (torch.randn(N, V, generator=gen) * 3).to(dtype)
    t = torch.randint(0, V, (N,), generator=gen)
    if N > 2:
        t[1] = -100
    d = x.cuda()
    dloss = torch.tensor([0.25], device="cuda")
    loss, lse = ops.cross_entropy_fwd_bwd_(d, t.cuda(), dloss, -100)
    torch.cuda.synchronize()
    rows, lse_r, g = CE.ce_rows(x.float(), t, -100, 0.25)
    assert max_abs(loss, rows) <= 1e-5 * max(1.0, rows.abs().max().item())
    assert max_abs(lse, lse_r) <= 1e-5 * max(1.0, lse_r.abs().max().item())
    if dtype == torch.float32:
        assert max_abs(d, g) <= 1e-4 * max(1.0, g.abs().max().item())
    else:
        assert rel_l2(d, g) <= 1e-2
    if N > 2:
        assert not d[1].any() and loss[1] == 0


def test_ce_invalid_target_and_shapes():
    banner("cross entropy invalid target / shapes")
    x = torch.randn(3, 64, device="cuda")
    loss, _ = ops.cross_entropy_fwd_bwd_(x, torch.tensor([0, 64, -1], device="cuda"), None, -100)
    assert torch.isfinite(loss[0]) and torch.isnan(loss[1]) and torch.isnan(loss[2])
    with pytest.raises(ValueError, match="not compiled"):
        ops.cross_entropy_fwd_bwd_(torch.randn(2, 60, device="cuda"), torch.zeros(2, dtype=torch.long,
                                                                                    device="cuda"), None, -100)


@pytest.mark.parametrize("num_chunks,V", [(1, 4096), (3, 4096), (8, 4096), (1, 4000), (3, 4000)])
def test_fused_linear_ce_matches_oracle(num_chunks, V):
    """The whole LCE against the oracle, at a vocabulary of whole 256-wide GEMM tiles and one that is not."""
    banner(f"fused linear CE chunks={num_chunks} V={V}")
    gen = torch.Generator().manual_seed(num_chunks)
    B, T, H = 2, 300, 256
    x = torch.randn(B, T, H, generator=gen).bfloat16()
    w = (torch.randn(V, H, generator=gen) * 0.05).bfloat16()
    t = torch.randint(0, V, (B, T), generator=gen)
    t[0, :7] = -100
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    loss = fused_ce.fused_linear_cross_entropy(xd, t.cuda(), wd, num_chunks=num_chunks)
    loss.backward()
    l_r, dx_r, dw_r = CE.linear_ce(x.float().reshape(-1, H), t.reshape(-1), w.float())
    assert abs(loss.item() - l_r.item()) <= 1e-3 * abs(l_r.item())
    assert rel_l2(xd.grad.reshape(-1, H), dx_r) <= 1e-2
    assert rel_l2(wd.grad, dw_r) <= 1e-2
    assert wd.grad.shape == w.shape and xd.grad.shape == x.shape


@pytest.mark.parametrize("N,H,V,num_chunks", [
    (700, 256, 4096, 8),   # two passes, the second ragged; dx in two parts
    (1100, 128, 8192, 8),  # four passes; dx in eight parts
    (257, 64, 1000, 4),    # a vocabulary that allows no parts
    (90, 512, 16384, 1),   # one pass; dx in sixteen parts
])
def test_fused_linear_ce_passes_and_parts(monkeypatch, N, H, V, num_chunks):
    """The rows per pass, the accumulation of dW across passes and the parts of dx (which calls this small would not
    take by themselves) against the oracle."""
    monkeypatch.setattr(fused_ce, "_outlasts_host", lambda *a: True)
    rows = fused_ce._rows_per_pass(N, num_chunks, H, 2)
    banner(f"fused linear CE N={N} H={H} V={V}: {rows} rows per pass, {fused_ce._dx_split(rows, H, V)} parts")
    gen = torch.Generator().manual_seed(N)
    x = torch.randn(1, N, H, generator=gen).bfloat16()
    w = (torch.randn(V, H, generator=gen) * 0.05).bfloat16()
    t = torch.randint(0, V, (1, N), generator=gen)
    t[0, ::9] = -100
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    loss = fused_ce.fused_linear_cross_entropy(xd, t.cuda(), wd, num_chunks=num_chunks)
    (3.0 * loss).backward()
    l_r, dx_r, dw_r = CE.linear_ce(x.float().reshape(-1, H), t.reshape(-1), w.float())
    assert abs(loss.item() - l_r.item()) <= 1e-3 * abs(l_r.item())
    assert rel_l2(xd.grad.reshape(-1, H), 3.0 * dx_r) <= 1e-2
    assert rel_l2(wd.grad, 3.0 * dw_r) <= 1e-2


@pytest.mark.parametrize("num_chunks", [1, 8])
def test_fused_linear_ce_feature_major_x(monkeypatch, num_chunks):
    """Hidden states laid out feature by feature (a dense transposed x, whose gradient has its strides), at a size whose
    dx may be taken in parts: the same result as for the row-major copy to the rounding of dx."""
    banner(f"fused linear CE feature-major x chunks={num_chunks}")
    monkeypatch.setattr(fused_ce, "_outlasts_host", lambda *a: True)
    N, H, V = 1100, 128, 8192
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(1, H, N, generator=gen).bfloat16().cuda().transpose(1, 2)
    w = (torch.randn(V, H, generator=gen) * 0.05).bfloat16()
    t = torch.randint(0, V, (1, N), generator=gen)
    assert fused_ce._dx_split(fused_ce._rows_per_pass(N, num_chunks, H, 2), H, V) > 1 and not x[0].is_contiguous()
    xd, wd = x.requires_grad_(), w.cuda().requires_grad_()
    loss = fused_ce.fused_linear_cross_entropy(xd, t.cuda(), wd, num_chunks=num_chunks)
    loss.backward()
    l_r, dx_r, dw_r = CE.linear_ce(x.detach().float().cpu().reshape(-1, H), t.reshape(-1), w.float())
    assert abs(loss.item() - l_r.item()) <= 1e-3 * abs(l_r.item())
    assert rel_l2(xd.grad.reshape(-1, H), dx_r) <= 1e-2 and rel_l2(wd.grad, dw_r) <= 1e-2


@pytest.mark.parametrize("N,x_dtype", [(96, torch.bfloat16), (1100, torch.bfloat16), (96, torch.float32)])
def test_fused_linear_ce_fp32_weight_under_autocast(N, x_dtype):
    """bf16 (and, in one pass, fp32) hidden states and an fp32 weight under bf16 autocast: over several chunks the weight's gradient holds fp32
    sums, also where every row fits one pass (a sum rounded to bf16 on the way would be a bf16 number throughout)."""
    H, V, num_chunks = 128, 4096, 8
    rows = fused_ce._rows_per_pass(N, num_chunks, H, 2)
    banner(f"fused linear CE fp32 weight N={N}: {rows} rows per pass")
    gen = torch.Generator().manual_seed(N)
    x = torch.randn(1, N, H, generator=gen).bfloat16()
    w = (torch.randn(V, H, generator=gen) * 0.05).bfloat16().float()
    t = torch.randint(0, V, (1, N), generator=gen)
    xd, wd = x.to("cuda", x_dtype).requires_grad_(), w.cuda().requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss = fused_ce.fused_linear_cross_entropy(xd, t.cuda(), wd, num_chunks=num_chunks)
    loss.backward()
    assert wd.grad.dtype == torch.float32
    assert (wd.grad != wd.grad.bfloat16().float()).float().mean() > 0.9  # 2^-16 of fp32 values are bf16 ones
    assert rel_l2(wd.grad, CE.linear_ce(x.float().reshape(-1, H), t.reshape(-1), w)[2]) <= 1e-2


@pytest.mark.parametrize("num_chunks", [1, 8])
def test_fused_linear_ce_fp16_weight_under_autocast(num_chunks):
    """An fp16 weight under bf16 autocast: its gradient comes back in fp16."""
    banner(f"fused linear CE fp16 weight chunks={num_chunks}")
    N, H, V = 300, 128, 4096
    gen = torch.Generator().manual_seed(5)
    x = torch.randn(1, N, H, generator=gen).bfloat16()
    w = (torch.randn(V, H, generator=gen) * 0.05).bfloat16()
    t = torch.randint(0, V, (1, N), generator=gen)
    xd, wd = x.cuda().requires_grad_(), w.to("cuda", torch.float16).requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss = fused_ce.fused_linear_cross_entropy(xd, t.cuda(), wd, num_chunks=num_chunks)
    (1024.0 * loss).backward()  # a gradient scale that keeps fp16's small values normal
    _, dx_r, dw_r = CE.linear_ce(x.float().reshape(-1, H), t.reshape(-1), w.float())
    assert wd.grad.dtype == torch.float16 and rel_l2(wd.grad, 1024 * dw_r) <= 1e-2
    assert rel_l2(xd.grad.reshape(-1, H), 1024 * dx_r) <= 1e-2


class _Calls(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("N,H,V,parts", [(128, 384, 8192, False), (1024, 1024, 8192, False), (210, 768, 32000, False),
                                         (128, 1024, 50304, True), (1024, 512, 32000, True)])
def test_fused_linear_ce_one_pass_calls(N, H, V, parts):
    """A call that waits for its launches makes the fewest: three products, the loss and torch's scaling of both
    gradients; one whose kernels outlast them takes dx in parts and the HIP scaling of the large gradient."""
    banner(f"fused linear CE one pass N={N} H={H} V={V}")
    gen = torch.Generator("cuda").manual_seed(N)
    x = torch.randn(1, N, H, device="cuda", generator=gen).bfloat16().requires_grad_()
    w = (torch.randn(V, H, device="cuda", generator=gen) * 0.05).bfloat16().requires_grad_()
    t = torch.randint(0, V, (1, N), device="cuda", generator=gen)
    with _Calls() as calls:
        fused_ce.fused_linear_cross_entropy(x, t, w, num_chunks=1).backward()
    n = [sum(k in c for c in calls.names) for k in ("aten.mm", "aten.bmm", "archbench_amd", "aten.copy_", "aten.mul")]
    assert n == ([2, 1, 3, 0, 1] if parts else [3, 0, 1, 0, 2]), calls.names


@pytest.mark.parametrize("hip", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_scaled_gradients(dtype, hip):
    """Both ways of scaling a stored gradient give the fp32 product rounded once, and differentiate under create_graph."""
    banner(f"scaled gradient {dtype} hip={hip}")
    x = torch.randn(4097, 1024, device="cuda", generator=torch.Generator("cuda").manual_seed(7)).to(dtype)
    s = torch.tensor(1 / 3, device="cuda", requires_grad=True)
    with torch.no_grad():
        assert torch.equal(fused_ce._scaled(x, s, hip), (x.float() * s).to(dtype))
    y = fused_ce._scaled(x.requires_grad_(), s, hip)
    assert all(g is not None for g in torch.autograd.grad(y.float().sum(), (x, s)))


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("outlasts", [False, True])
def test_fused_linear_ce_batched_gradients(monkeypatch, outlasts):
    """Several gradients of the loss in one backward (is_grads_batched), however they are scaled."""
    banner(f"fused linear CE batched gradients outlasts={outlasts}")
    monkeypatch.setattr(fused_ce, "_outlasts_host", lambda *a: outlasts)
    gen = torch.Generator("cuda").manual_seed(9)
    x = torch.randn(1, 64, 512, device="cuda", generator=gen).bfloat16().requires_grad_()
    w = (torch.randn(8192, 512, device="cuda", generator=gen) * 0.05).bfloat16().requires_grad_()
    t = torch.randint(0, 8192, (1, 64), device="cuda", generator=gen)
    loss = fused_ce.fused_linear_cross_entropy(x, t, w, num_chunks=1)
    gs = torch.tensor([1.0, 0.5, 1 / 3], device="cuda")
    got = torch.autograd.grad(loss, (x, w), gs, is_grads_batched=True, retain_graph=True)
    for i, g in enumerate(gs):
        for a, b in zip(got, torch.autograd.grad(loss, (x, w), g, retain_graph=True)):
            assert torch.equal(a[i], b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("n,S", [(1, 1), (8, 3), (1001, 2), (4096, 16)])
def test_scale_and_sum_of_parts(dtype, n, S):
    """ops.scaled equals the product in fp32 rounded once, ops.sum_parts_ the ordered 64-bit sum rounded to fp32 and the
    dtype, exactly."""
    banner(f"scaled / sum of parts n={n} S={S} {dtype}")
    gen = torch.Generator("cuda").manual_seed(n)
    x = torch.randn(n, device="cuda", generator=gen).to(dtype)
    s = torch.tensor(0.37, device="cuda")
    assert torch.equal(ops.scaled(x, s), (x.float() * s).to(dtype))
    if n % 8 == 0:
        parts = torch.randn(S, n, device="cuda", generator=gen)
        ref = torch.zeros(n, device="cuda", dtype=torch.float64)
        for p in parts:
            ref += p
        out = torch.empty(n, device="cuda", dtype=dtype)
        ops.sum_parts_(parts, out)
        assert torch.equal(out, ref.float().to(dtype))
