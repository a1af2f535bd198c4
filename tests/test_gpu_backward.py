"""GPU gradients of the lookups against autograd of an independent dense
formulation (fp64, CPU): the latest-k values are a linear gather from the
oracle's source indices, the sums a linear map by per-stream masks."""
import numpy as np
import pytest
import torch

import oracle
from ravel_em import causal_last_k_lookup, causal_sum_lookup

pytestmark = pytest.mark.gpu


def dense_latest_k(payload64: torch.Tensor, src: np.ndarray) -> torch.Tensor:
    B, T, C, D = payload64.shape
    s = torch.from_numpy(src.astype(np.int64)).view(-1)
    rows = payload64.reshape(-1, D).index_select(0, s.clamp_min(0))
    rows = rows * (s >= 0).view(-1, 1).to(rows.dtype)
    return rows.view(B, T, C, src.shape[-1], D)


CASES = [
    # B, T, C, A, masked, separate reads, k
    (2, 50, 3, 7, False, False, 1),
    (2, 50, 3, 7, False, False, 3),
    (2, 50, 3, 7, True, False, 2),
    (2, 50, 3, 7, False, True, 2),
    (1, 5000, 2, 3, False, False, 4),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_latest_k_gradient(device, case, dtype):
    B, T, C, A, masked, sep, k = case
    g = torch.Generator().manual_seed(T + k)
    w = torch.randint(0, A, (B, T, C), generator=g)
    r = torch.randint(0, A, (B, T, C), generator=g) if sep else None
    m = (torch.rand(B, T, generator=g) < 0.6) if masked else None
    p = torch.randn(B, T, C, 4, generator=g).to(dtype)
    gy = torch.randn(B, T, C, k, 4, generator=g).to(dtype)
    pg = p.to(device).requires_grad_(True)
    vals, _ = causal_last_k_lookup(w.to(device), pg, None if r is None else r.to(device), address_space=A, k=k,
                                   write_mask=None if m is None else m.to(device))
    (grad,) = torch.autograd.grad(vals, pg, gy.to(device))
    src = oracle.latest_k_src(w, r, address_space=A, k=k, write_mask=m)
    p64 = p.double().requires_grad_(True)
    (want,) = torch.autograd.grad(dense_latest_k(p64, src), p64, gy.double())
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    torch.testing.assert_close(grad.cpu().double(), want, rtol=tol, atol=tol)


# Separate reads and masked writes take the sorted backward (a stable sort of
# the slots' source ids, then each source's slots summed in slot order): the
# gradient must be bit-identical from run to run, and match fp64 autograd of
# the dense formulation.  Few addresses make long runs of slots per source,
# which cross the summing kernels' parts (walker: 16-byte rows) and chunks
# (other rows).
DET_CASES = [
    # B, T, C, A, kept share of writes (1 = no mask), separate reads, k, D, dtype
    (2, 3000, 3, 4, 1.0, True, 4, 64, torch.bfloat16),
    (1, 5000, 2, 2, 0.7, False, 3, 5, torch.float32),
    (2, 2000, 2, 7, 0.7, True, 8, 16, torch.float16),
    (1, 6000, 1, 1, 1.0, True, 2, 8, torch.float64),
    (2, 500, 4, 300, 0.7, True, 1, 24, torch.bfloat16),
    # one write in 500 kept: ~1500 slots name each source, runs cross parts
    (1, 8000, 2, 1, 0.002, True, 3, 64, torch.bfloat16),
    (1, 8000, 2, 1, 0.002, False, 3, 6, torch.float32),
]


@pytest.mark.parametrize("case", DET_CASES, ids=[str(i) for i in range(len(DET_CASES))])
def test_latest_k_backward_sorted_is_deterministic(device, case):
    B, T, C, A, keep, sep, k, D, dtype = case
    print(f"[sorted backward] {case}", flush=True)
    g = torch.Generator().manual_seed(T + k + D)
    w = torch.randint(0, A, (B, T, C), generator=g)
    r = torch.randint(0, A, (B, T, C), generator=g) if sep else None
    m = (torch.rand(B, T, generator=g) < keep) if keep < 1 else None
    p = torch.randn(B, T, C, D, generator=g).to(dtype)
    gy = torch.randn(B, T, C, k, D, generator=g).to(dtype)
    grads = []
    for _ in range(2):
        pg = p.to(device).requires_grad_(True)
        vals, _ = causal_last_k_lookup(w.to(device), pg, None if r is None else r.to(device),
                                       address_space=A, k=k,
                                       write_mask=None if m is None else m.to(device))
        (grad,) = torch.autograd.grad(vals, pg, gy.to(device))
        grads.append(grad.cpu())
    bits = {2: torch.int16, 4: torch.int32, 8: torch.int64}[grads[0].element_size()]
    assert torch.equal(grads[0].view(bits), grads[1].view(bits)), "two runs differ"
    src = oracle.latest_k_src(w, r, address_space=A, k=k, write_mask=m)
    p64 = p.double().requires_grad_(True)
    (want,) = torch.autograd.grad(dense_latest_k(p64, src), p64, gy.double())
    # a source's slots summed in fp32 (16-bit rows) or fp64, rounded once
    acc_u = 2.0 ** -24 if dtype in (torch.bfloat16, torch.float16) else 2.0 ** -52
    rtol = {torch.bfloat16: 1e-2, torch.float16: 1e-2, torch.float32: 1e-5, torch.float64: 1e-5}[dtype]
    (scale,) = torch.autograd.grad(dense_latest_k(p64, src), p64, gy.double().abs())
    (nterm,) = torch.autograd.grad(dense_latest_k(p64, src), p64, torch.ones_like(gy, dtype=torch.float64))
    err = (grads[0].double() - want).abs()
    bound = rtol * want.abs() + 1.01 * nterm * acc_u * scale + 1e-30
    print(f"[sorted backward] max err/bound {(err / bound).max().item():.3f}, "
          f"longest run {int(nterm.max().item())}", flush=True)
    assert (err <= bound).all()


def dense_sum(payload64, write, read, A, mask):
    """out[r] = sum over earlier same-stream writes, as an explicit masked matmul."""
    B, T, C, D = payload64.shape
    rd = write if read is None else read
    wa = torch.remainder(write, A)
    ra = torch.remainder(rd, A)
    tt = torch.arange(T)
    earlier = tt.view(T, 1) > tt.view(1, T)  # [t_read, t_write]
    outs = []
    for b in range(B):
        heads = []
        for c in range(C):
            same = ra[b, :, c].view(T, 1) == wa[b, :, c].view(1, T)
            M = (same & earlier).double()
            if mask is not None:
                M = M * mask[b].double().view(1, T)
            heads.append(M @ payload64[b, :, c])
        outs.append(torch.stack(heads, dim=1))
    return torch.stack(outs)


@pytest.mark.parametrize("case", CASES[:4], ids=[str(i) for i in range(4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sum_gradient(device, case, dtype):
    B, T, C, A, masked, sep, _ = case
    g = torch.Generator().manual_seed(T + 99)
    w = torch.randint(0, A, (B, T, C), generator=g)
    r = torch.randint(0, A, (B, T, C), generator=g) if sep else None
    m = (torch.rand(B, T, generator=g) < 0.6) if masked else None
    p = torch.randn(B, T, C, 4, generator=g).to(dtype)
    gy = torch.randn(B, T, C, 4, generator=g).to(dtype)
    pg = p.to(device).requires_grad_(True)
    out, _ = causal_sum_lookup(w.to(device), pg, None if r is None else r.to(device), address_space=A,
                               write_mask=None if m is None else m.to(device))
    (grad,) = torch.autograd.grad(out, pg, gy.to(device))
    p64 = p.double().requires_grad_(True)
    (want,) = torch.autograd.grad(dense_sum(p64, w, r, A, m), p64, gy.double())
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    torch.testing.assert_close(grad.cpu().double(), want, rtol=tol, atol=tol)


# The joint backward (both outputs' gradients in one segmented walk) at the edges
# of its dispatch: row units of 16, 8, 4 and 2 bytes and several column blocks,
# every state depth (k = 1, 2, 3..4, 5..8), one item to many parts a segment, runs
# inside a walker, across walkers and across parts, and stretches of reads with no
# write for longer than a part.
JOINT_BWD = [
    # B, T, C, A, kept share of writes (1 = no mask), separate reads, k, D, dtype
    (2, 1, 3, 5, 1.0, False, 1, 8, torch.bfloat16),
    (1, 63, 2, 9, 0.5, True, 2, 24, torch.float16),
    (3, 257, 2, 300, 1.0, False, 8, 32, torch.float32),
    (2, 1000, 3, 40, 0.8, True, 4, 64, torch.bfloat16),
    (1, 1025, 1, 1, 1.0, True, 3, 21, torch.bfloat16),    # one run, 2-byte units
    (1, 2100, 2, 3, 0.6, False, 5, 50, torch.bfloat16),   # 4-byte units
    (1, 4097, 2, 700, 1.0, True, 4, 96, torch.bfloat16),  # global sort of the merged tape
    (1, 4097, 1, 50, 1.0, False, 8, 128, torch.float32),  # several column blocks
    (1, 3000, 2, 2, 0.7, True, 1, 5, torch.float64),
    (1, 9000, 1, 1, 0.002, True, 8, 16, torch.float16),   # rare writes: runs of reads
    (1, 5000, 2, 70000, 1.0, True, 2, 130, torch.float16),  # 32-bit tape
    (1, 1500, 1, 4, 0.9, True, 7, 300, torch.bfloat16),   # five column blocks of 4-byte units
]


def stream_suffix_sums(write, read, A, mask, grad64):
    """Per write: the sum of grad64 over the later reads of its stream (fp64)."""
    B, T, C, D = grad64.shape
    stream = torch.arange(B).view(B, 1, 1) * C + torch.arange(C)
    t = torch.arange(T).view(1, T, 1)
    wk = ((stream * A + write.remainder(A)) * T + t).reshape(-1)
    rk, order = ((stream * A + read.remainder(A)) * T + t).reshape(-1).sort()
    csum = torch.cat([torch.zeros(1, D, dtype=torch.float64), grad64.reshape(-1, D)[order].cumsum(0)])
    lo = torch.searchsorted(rk, wk, right=True)
    hi = torch.searchsorted(rk, (wk // T + 1) * T)
    out = (csum[hi] - csum[lo]).view(B, T, C, D)
    n = (hi - lo).view(B, T, C, 1).double()
    if mask is not None:
        out, n = out * mask.view(B, T, 1, 1), n * mask.view(B, T, 1, 1)
    return out, n


@pytest.mark.parametrize("case", JOINT_BWD, ids=[str(i) for i in range(len(JOINT_BWD))])
def test_joint_gradient(device, case):
    """|err| <= u |x| (one rounding) + n 2^-24 (2^-52 for fp32/fp64 rows) sum|terms|:
    a sum of n terms in any order; the reference's own cumulative sums add
    T 2^-52 of theirs."""
    from ravel_em import causal_last_k_and_sum_lookup

    B, T, C, A, keep, sep, k, D, dtype = case
    print(f"[joint backward] {case}", flush=True)
    g = torch.Generator().manual_seed(T + k + D)
    w = torch.randint(0, A, (B, T, C), generator=g)
    r = torch.randint(0, A, (B, T, C), generator=g) if sep else None
    m = (torch.rand(B, T, generator=g) < keep) if keep < 1 else None
    p = torch.randn(B, T, C, D, generator=g).to(dtype)
    gv = torch.randn(B, T, C, k, D, generator=g).to(dtype)
    gs = torch.randn(B, T, C, D, generator=g).to(dtype)

    def run(*which):
        pg = p.to(device).requires_grad_(True)
        vals, _, summed, _ = causal_last_k_and_sum_lookup(
            w.to(device), pg, None if r is None else r.to(device), address_space=A, k=k,
            write_mask=None if m is None else m.to(device))
        outs = [(vals, gv), (summed, gs)]
        (grad,) = torch.autograd.grad([outs[i][0] for i in which], pg,
                                      [outs[i][1].to(device) for i in which])
        return grad.cpu()

    src = oracle.latest_k_src(w, r, address_space=A, k=k, write_mask=m)
    p64 = p.double().requires_grad_(True)

    def lin(x):
        return torch.autograd.grad(dense_latest_k(p64, src), p64, x)[0]

    rd = w if r is None else r
    v = (lin(gv.double()), lin(gv.double().abs()), lin(torch.ones_like(gv, dtype=torch.float64)))
    s64, n = stream_suffix_sums(w, rd, A, m, gs.double())
    s = (s64, stream_suffix_sums(w, rd, A, m, gs.double().abs())[0], n)
    wide = dtype in (torch.float32, torch.float64)
    acc_u = 2.0 ** -52 if wide else 2.0 ** -24
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24,
         torch.float64: 2.0 ** -52}[dtype]
    for which in ((0, 1), (0,), (1,)):
        got = run(*which)
        want, scale, terms = (sum(x[i] for j, x in enumerate((v, s)) if j in which) for i in range(3))
        err = (got.double() - want).abs()
        bound = u * want.abs() + (1.01 * terms * acc_u + 4 * T * 2.0 ** -52) * scale + \
            T * 2.0 ** -50 * (1 in which) + 2.0 ** -24 * (not wide)
        assert (err <= bound).all(), (which, (err / bound).max().item())
        if which == (0, 1):
            bits = {2: torch.int16, 4: torch.int32, 8: torch.int64}[got.element_size()]
            assert torch.equal(got.view(bits), run(0, 1).view(bits)), "two runs differ"


@pytest.mark.parametrize("sep,masked", [(False, False), (True, False), (False, True)])
def test_eager_functions_equal_the_custom_ops(device, sep, masked):
    """Plain eager training calls take autograd functions: same results and
    gradients as the custom ops bit for bit, saved tensors go through the hooks,
    a missing gradient is none, and a second derivative raises as the ops do."""
    from ravel_em import _ops, causal_last_k_and_sum_lookup

    B, T, C, D, A, k = 2, 300, 3, 16, 11, 3
    g = torch.Generator().manual_seed(5)
    w = torch.randint(0, A, (B, T, C), generator=g, dtype=torch.int32).to(device)
    r = torch.randint(0, A, (B, T, C), generator=g, dtype=torch.int32).to(device) if sep else None
    m = (torch.rand(B, T, generator=g) < 0.6).to(device) if masked else None
    p = torch.randn(B, T, C, D, generator=g).to(device).requires_grad_(True)
    gv = torch.randn(B, T, C, k, D, generator=g).to(device)
    gs = torch.randn(B, T, C, D, generator=g).to(device)
    kw = dict(address_space=A, write_mask=m)
    pairs = [
        (lambda: causal_last_k_lookup(w, p, r, k=k, **kw)[:1],
         lambda: _ops.latest_k(w, p, r, m, A, k, True)[:1] if r is None and m is None
         else _ops.latest_k_taped(w, p, r, m, A, k)[:1], (gv,)),
        (lambda: causal_sum_lookup(w, p, r, **kw)[:1],
         lambda: _ops.seg_sum(w, p, r, m, A)[:1], (gs,)),
        (lambda: causal_last_k_and_sum_lookup(w, p, r, k=k, **kw)[0::2],
         lambda: _ops.latest_k_sum(w, p, r, m, A, k, False)[0::3], (gv, gs)),
    ]
    for fn, op, grads in pairs:
        a, b = fn(), op()
        ga, = torch.autograd.grad(a, p, grads, retain_graph=True)
        gb, = torch.autograd.grad(b, p, grads)
        assert all(torch.equal(x, y) for x, y in zip(a, b)) and torch.equal(ga, gb)
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t), t.clone())[1],
                                                      lambda t: t):
            c = fn()
        gc, = torch.autograd.grad(c, p, grads)
        assert seen and torch.equal(gc, ga)
        lead = [x.clone().requires_grad_(True) for x in grads]
        gg, = torch.autograd.grad(a, p, lead, create_graph=True)
        with pytest.raises(RuntimeError):
            gg.sum().backward()
        assert torch.autograd.grad(a[0], p, grads[0], allow_unused=True)[0] is not None


@pytest.mark.parametrize("sep,masked", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("B,T,C,A", [(2, 5000, 3, 200), (1, 4200, 2, 70000), (1, 4300, 1, 1 << 21),
                                     (2, 2000, 2, 30)])
def test_kept_keys_give_the_gradient_of_the_sorted_addresses(device, sep, masked, B, T, C, A):
    """A training forward that sorts keeps its keys: the backward that walks them
    equals, bit for bit, the one that sorts the addresses again (keys of one to
    three digit passes, 32 and 64 bits, and a tape sorted by one block a segment)."""
    from ravel_em import _ops, causal_last_k_and_sum_lookup

    D, k = 16, 2
    g = torch.Generator().manual_seed(T)
    w = torch.randint(0, A, (B, T, C), generator=g).to(device)
    r = torch.randint(0, A, (B, T, C), generator=g).to(device) if sep else None
    m = (torch.rand(B, T, generator=g) < 0.7).to(device) if masked else None
    p = torch.randn(B, T, C, D, generator=g).to(torch.bfloat16).to(device).requires_grad_(True)
    gv = torch.randn(B, T, C, k, D, generator=g).to(torch.bfloat16).to(device)
    gs = torch.randn(B, T, C, D, generator=g).to(torch.bfloat16).to(device)
    keys = _ops.kept_keys(p, r, m, A, k)
    records = B * T * C * (2 if sep or masked else 1)
    assert keys.numel() in (4 * records, 8 * records)
    summed = causal_sum_lookup(w, p, r, address_space=A, write_mask=m)[0]
    got, = torch.autograd.grad(summed, p, gs)
    assert torch.equal(summed, _ops.seg_sum(w, p, r, m, A)[0])
    assert torch.equal(got, _ops.seg_sum_backward(w, r, m, gs, A))
    vals, _, summed, _ = causal_last_k_and_sum_lookup(w, p, r, address_space=A, k=k, write_mask=m)
    got, = torch.autograd.grad((vals, summed), p, (gv, gs))
    assert torch.equal(got, _ops.latest_k_sum_backward(w, r, m, gv, gs, A, k, False))
