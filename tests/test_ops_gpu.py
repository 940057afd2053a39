"""The sparse round's op ABI (gather of the selected cells, grouped unit MLP, CSR messages, gated
delta update, their backwards) on the GPU against the reference's golden vectors and the CPU
oracle, through the custom ops of ``hsn_amd.kernels.ops``. GPU only.

The vectors' inputs lie on an f16/bf16-exact grid and their outputs come from the reference's
f64 oracle rounded once to f32, so one vector serves every dtype: f32 within 1e-5, f16 and bf16
within 1e-2 (atol = rtol, the reference's tolerances, tests/golden/MANIFEST.json).
"""

from __future__ import annotations

import pytest
import torch

from conftest import load_golden

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.float16: 1e-2, torch.bfloat16: 1e-2}
SIZES = ["tiny", "ref", "odd"]
DTYPES = [torch.float32, torch.float16, torch.bfloat16]


@pytest.fixture(scope="module")
def ops(cuda_device):
    from hsn_amd.kernels import ops

    assert ops.available(), "the HIP library must be built for the GPU tests"
    return ops


def _close(got, want, dtype, what, scaled=False):
    """``scaled``: the absolute tolerance relative to the largest expected value, for sums so
    long that fp32 rounding alone passes the fixed tolerance where they cancel (at d = 1024 a
    dot product rounds to about sqrt(d) 2^-24 of its terms' scale, and grad_a sums d-long
    products of d-long sums)."""
    tol = TOL[dtype]
    got, want = got.float().cpu(), want.float()
    atol = tol * max(1.0, float(want.abs().max())) if scaled else tol
    err = float((got - want).abs().max()) if want.numel() else 0.0
    torch.testing.assert_close(got, want, atol=atol, rtol=tol,
                               msg=f"{what}: max |error| {err:.3g}, max |want| "
                                   f"{float(want.abs().max()) if want.numel() else 0.0:.3g}")


def _put(v, dev, dtype):
    return {k: (t.to(dev, dtype) if t.is_floating_point() else t.to(dev)) for k, t in v.items()}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("size", SIZES)
def test_gated_update_matches_golden(ops, cuda_device, size, dtype):
    v = load_golden(f"{size}_gated_delta_update.safetensors")
    D = _put(v, cuda_device, dtype)
    h, q, age = D["h"].clone(), D["q"].clone(), D["age"].clone()
    old = ops.update_inplace(h, q, age, D["cell_idx"], D["valid"], D["c"], D["b"])
    _close(h, v["h_out"], dtype, "h_out")
    _close(q, v["q_out"], dtype, "q_out")
    assert torch.equal(age.cpu(), v["age_out"])
    _close(old, v["h_old_saved"], dtype, "h_old_saved")
    gh, gq, gc, gb = ops.update_backward(D["cell_idx"], D["valid"], D["c"], D["b"],
                                                     D["h_old_saved"], D["grad_h_out"],
                                                     D["grad_q_out"])
    for name, got in zip(("grad_h", "grad_q", "grad_c", "grad_b"), (gh, gq, gc, gb)):
        _close(got, v[name], dtype, name)


@pytest.mark.parametrize("size", SIZES)
def test_functional_update_autograd_matches_golden(ops, cuda_device, size):
    """The functional op leaves its inputs alone and its autograd gives the golden gradients."""
    v = load_golden(f"{size}_gated_delta_update.safetensors")
    D = _put(v, cuda_device, torch.float32)
    h = D["h"].clone().requires_grad_(True)
    q = D["q"].clone().requires_grad_(True)
    c = D["c"].clone().requires_grad_(True)
    b = D["b"].clone().requires_grad_(True)
    for op in (ops.update_op, ops.state_update_op):
        hn, qn, an, old = op(h, q, D["age"], D["cell_idx"], D["valid"], c, b)
        assert torch.equal(h.detach(), D["h"]) and torch.equal(D["age"].cpu(), v["age"])
        _close(hn.detach(), v["h_out"], torch.float32, "h_out")
        assert torch.equal(an.cpu(), v["age_out"])
        grads = torch.autograd.grad((hn, qn), (h, q, c, b), (D["grad_h_out"], D["grad_q_out"]))
        for name, got in zip(("grad_h", "grad_q", "grad_c", "grad_b"), grads):
            _close(got, v[name], torch.float32, name)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("size", SIZES)
def test_gather_concat_matches_golden(ops, cuda_device, size, dtype):
    v = load_golden(f"{size}_gather_concat.safetensors")
    D = _put(v, cuda_device, dtype)
    out = ops.gather_op(D["u"], D["eps"], D["h"], D["m"], D["cell_idx"])
    _close(out, v["v"], dtype, "v")
    N = v["h"].shape[1]
    gu, ge, gh, gm = ops.gather_backward(D["grad_v"], D["cell_idx"], N)
    for name, got in zip(("grad_u", "grad_eps", "grad_h", "grad_m"), (gu, ge, gh, gm)):
        _close(got, v[name], dtype, name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gather_backward_slot_batches_match_oracle(ops, cuda_device, dtype):
    """K = 19 slots, three of the kernel's batches of 8, with cells repeated inside a batch,
    across batches and three times in a row: grad_h is the scatter-add of the slots' third
    block, in slot order (the float64 oracle adds them in any order)."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(91)
    B, N, K, d = 3, 30, 19, 36
    grad_v = (torch.randn(B, K, 4 * d, generator=g) * 0.5).to(dtype)
    cells = torch.randint(0, N, (B, K), generator=g, dtype=torch.int32)
    cells[0, 5] = cells[0, 2]      # inside the first batch
    cells[1, 17] = cells[1, 3]     # across batches
    cells[2, [4, 9, 18]] = 7       # three batches
    want = O.gather_concat_bwd(grad_v.double(), cells, N)
    dev = cuda_device
    got = ops.gather_backward(grad_v.to(dev), cells.to(dev), N)
    for name, g_, w_ in zip(("grad_u", "grad_eps", "grad_h", "grad_m"), got, want):
        _close(g_, w_, dtype, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gather_backward_rounds_a_repeated_cell_once(ops, cuda_device, dtype):
    """A cell taken by many slots of a row in 16-bit storage: its grad_h is the fp32 sum of the
    slots' third blocks in slot order, rounded once to the storage dtype (the ABI's accumulation),
    not a rounding after every repeat. 40 slots, 30 of them on cell 2 (five of the kernel's
    batches of 8), with small values that a per-repeat rounding would lose."""
    g = torch.Generator().manual_seed(93)
    B, N, K, d = 2, 9, 40, 24
    grad_v = torch.randn(B, K, 4 * d, generator=g)
    grad_v[:, :, 2 * d:3 * d] = 1.0 + torch.rand(B, K, d, generator=g) * 2.0 ** -6
    grad_v = grad_v.to(dtype)
    cells = torch.randint(0, N, (B, K), generator=g, dtype=torch.int32)
    cells[:, torch.randperm(K, generator=g)[:30]] = 2
    # the expectation: slot-order fp32 sums per (row, cell), each rounded once
    want = torch.zeros(B, N, d)
    third = grad_v[:, :, 2 * d:3 * d].float()
    for r in range(B):
        acc = {}
        for k in range(K):
            c = int(cells[r, k])
            acc[c] = acc.get(c, torch.zeros(d)) + third[r, k]
        for c, v in acc.items():
            want[r, c] = v
    want = want.to(dtype)
    got = ops.gather_backward(grad_v.to(cuda_device), cells.to(cuda_device), N)[2].cpu()
    assert torch.equal(got, want)


def test_gather_autograd_matches_golden(ops, cuda_device):
    v = load_golden("odd_gather_concat.safetensors")
    D = _put(v, cuda_device, torch.float32)
    leaves = [D[k].clone().requires_grad_(True) for k in ("u", "eps", "h", "m")]
    out = ops.gather_op(*leaves, D["cell_idx"])
    grads = torch.autograd.grad(out, leaves, D["grad_v"])
    for name, got in zip(("grad_u", "grad_eps", "grad_h", "grad_m"), grads):
        _close(got, v[name], torch.float32, name)


def test_inplace_update_rejects_a_strided_state(ops, cuda_device):
    """The ABI updates h, q, age in place through plain pointers: a strided view is refused
    rather than silently copied."""
    v = load_golden("ref_gated_delta_update.safetensors")
    D = _put(v, cuda_device, torch.float32)
    h = D["h"].transpose(1, 2).contiguous().transpose(1, 2)
    with pytest.raises(ValueError, match="contiguous"):
        ops.update_inplace(h, D["q"].clone(), D["age"].clone(), D["cell_idx"], D["valid"],
                               D["c"], D["b"])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("size", SIZES)
def test_grouped_unit_mlp_matches_golden(ops, cuda_device, size, dtype):
    """Forward and backward against the vectors (the odd one has a unit without pairs: zero
    gradients); in f16 / bf16 the saved z1 is the storage dtype's, as the ABI stores it."""
    v = load_golden(f"{size}_grouped_unit_mlp.safetensors")
    D = _put(v, cuda_device, dtype)
    out, hidden = ops.mlp_op(D["v"], D["unit_idx"], D["W1"], D["b1"], D["W2"], D["b2"])
    _close(hidden, v["hidden_saved"], dtype, "hidden_saved")
    _close(out, v["out"], dtype, "out")
    got = ops.mlp_backward(D["v"], D["unit_idx"], D["W1"], D["W2"],
                                        D["hidden_saved"], D["grad_out"])
    for name, g_ in zip(("grad_v", "grad_W1", "grad_b1", "grad_W2", "grad_b2"), got):
        _close(g_, v[name], dtype, name)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("size", SIZES)
def test_csr_messages_match_golden(ops, cuda_device, size, dtype):
    """Forward and backward against the vectors: repeated slots (tiny: cell 1 twice in row 1) and
    edges of rows no slot selects (their grad_a is exactly zero)."""
    v = load_golden(f"{size}_csr_messages.safetensors")
    D = _put(v, cuda_device, dtype)
    m = ops.messages_op(D["h"], D["indptr"], D["indices"], D["a"], D["V"], D["cell_idx"])
    _close(m, v["m"], dtype, "m")
    gh, ga, gV = ops.messages_backward(D["h"], D["indptr"], D["indices"], D["a"], D["V"],
                                           D["cell_idx"], D["grad_m"])
    for name, g_ in zip(("grad_h", "grad_a", "grad_V"), (gh, ga, gV)):
        _close(g_, v[name], dtype, name)
    assert bool((ga.cpu()[v["grad_a"] == 0] == 0).all())


def test_unit_mlp_and_messages_autograd_match_golden(ops, cuda_device):
    """The custom ops' autograd registrations give the vectors' gradients."""
    v = load_golden("odd_grouped_unit_mlp.safetensors")
    D = _put(v, cuda_device, torch.float32)
    leaves = [D[k].clone().requires_grad_(True) for k in ("v", "W1", "b1", "W2", "b2")]
    out, _ = ops.mlp_op(leaves[0], D["unit_idx"], *leaves[1:])
    grads = torch.autograd.grad(out, leaves, D["grad_out"])
    for name, g_ in zip(("grad_v", "grad_W1", "grad_b1", "grad_W2", "grad_b2"), grads):
        _close(g_, v[name], torch.float32, name)
    v = load_golden("odd_csr_messages.safetensors")
    D = _put(v, cuda_device, torch.float32)
    h, a, V = (D[k].clone().requires_grad_(True) for k in ("h", "a", "V"))
    m = ops.messages_op(h, D["indptr"], D["indices"], a, V, D["cell_idx"])
    for name, g_ in zip(("grad_h", "grad_a", "grad_V"),
                        torch.autograd.grad(m, (h, a, V), D["grad_m"])):
        _close(g_, v[name], torch.float32, name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_unit_mlp_and_messages_match_oracle_on_ragged_shapes(ops, cuda_device, dtype):
    """Shapes the vectors leave open: units with more than 16 pairs (several row chunks), one
    unit without pairs, H and 4d off the 64-column tiles, d past one tile; a CSR with empty rows,
    self loops, repeated slots and d = 100 (two column tiles). Inputs rounded to the storage
    dtype first, the oracle run on them in float64."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(41)
    tol = TOL[dtype]
    P, M, d, H = 70, 5, 24, 200
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.5).to(dtype)  # noqa: E731
    v, W1, b1, W2, b2 = rnd(P, 4 * d), rnd(M, 4 * d, H), rnd(M, H), rnd(M, H, d), rnd(M, d)
    idx = torch.randint(0, M - 1, (P,), generator=g, dtype=torch.int32)  # unit M-1 unused
    dout = rnd(P, d)
    f64 = lambda t: t.double()  # noqa: E731
    want_out, want_h = O.grouped_unit_mlp(f64(v), idx, f64(W1), f64(b1), f64(W2), f64(b2))
    dev = cuda_device
    out, hidden = ops.mlp_op(v.to(dev), idx.to(dev), W1.to(dev), b1.to(dev),
                                       W2.to(dev), b2.to(dev))
    _close(hidden, want_h, dtype, "hidden")
    _close(out, want_out, dtype, "out")
    want = O.grouped_unit_mlp_bwd(f64(v), idx, f64(W1), f64(W2), f64(hidden.cpu()), f64(dout))
    got = ops.mlp_backward(v.to(dev), idx.to(dev), W1.to(dev), W2.to(dev), hidden,
                                        dout.to(dev))
    for name, g_, w_ in zip(("dv", "dW1", "db1", "dW2", "db2"), got, want):
        _close(g_, w_, dtype, name)
    assert bool((got[1][M - 1] == 0).all()) and bool((got[3][M - 1] == 0).all())
    B, N, K, d = 3, 50, 7, 100
    deg = torch.randint(0, 4, (N,), generator=g)
    deg[[3, 17]] = 0  # empty rows
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), deg.cumsum(0)]).to(torch.int32)
    E = int(indptr[-1])
    indices = torch.randint(0, N, (E,), generator=g, dtype=torch.int32)
    indices[0] = 0  # a self loop where row 0 has an edge
    a = torch.rand(E, generator=g).to(dtype)
    h, V = rnd(B, N, d), rnd(d, d)
    cell_idx = torch.randint(0, N, (B, K), generator=g, dtype=torch.int32)
    cell_idx[0, 1] = cell_idx[0, 0]  # a repeated slot
    cell_idx[1, 2] = 3  # an empty row
    gm = rnd(B, K, d)
    want_m = O.csr_messages(f64(h), indptr, indices, f64(a), f64(V), cell_idx)
    m = ops.messages_op(h.to(dev), indptr.to(dev), indices.to(dev), a.to(dev), V.to(dev),
                         cell_idx.to(dev))
    _close(m, want_m, dtype, "m")
    assert bool((m[1, 2] == 0).all())
    want = O.csr_messages_bwd(f64(h), indptr, indices, f64(a), f64(V), cell_idx, f64(gm))
    got = ops.messages_backward(h.to(dev), indptr.to(dev), indices.to(dev), a.to(dev),
                                    V.to(dev), cell_idx.to(dev), gm.to(dev))
    for name, g_, w_ in zip(("dh", "da", "dV"), got, want):
        _close(g_, w_, dtype, name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gated_update_slot_groups_match_oracle_and_slot_order(ops, cuda_device, dtype):
    """K = 19 slots (three groups of the kernel's 8) with padded slots. Rows without repeated
    cells: against the float64 oracle. Rows with a cell repeated inside a group and across
    groups: against 19 single-slot calls in slot order, since the ABI's update is in place and
    each slot reads h after the slots before it."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(77)
    B, N, K, d = 3, 40, 19, 70
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.5).to(dtype)  # noqa: E731
    h, q, c, b = rnd(B, N, d), rnd(B, d), rnd(B, K, d), torch.rand(B, K, d, generator=g).to(dtype)
    age = torch.randint(0, 9, (B, N), generator=g, dtype=torch.int32)
    cells = torch.stack([torch.randperm(N, generator=g)[:K] for _ in range(B)]).to(torch.int32)
    valid = (torch.rand(B, K, generator=g) > 0.2).to(torch.int32)
    dev = cuda_device
    f64 = lambda t: t.double()  # noqa: E731
    want = O.gated_delta_update_abi(f64(h), f64(q), age, cells, valid, f64(c), f64(b))
    got = ops.update_op(h.to(dev), q.to(dev), age.to(dev), cells.to(dev),
                                            valid.to(dev), c.to(dev), b.to(dev))
    for name, g_, w_ in zip(("h", "q", "age", "h_old"), got, want):
        _close(g_, w_, dtype, name)
    G, gq = rnd(B, N, d), rnd(B, d)  # the backward over the same three groups of slots
    old = got[3].cpu()
    want = O.gated_delta_update_bwd(cells, valid, f64(c), f64(b), f64(old), f64(G), f64(gq))
    back = ops.update_backward(cells.to(dev), valid.to(dev), c.to(dev), b.to(dev),
                                           old.to(dev), G.to(dev), gq.to(dev))
    for name, g_, w_ in zip(("grad_h", "grad_q", "grad_c", "grad_b"), back, want):
        _close(g_, w_, dtype, name)
    rep = cells.clone()
    rep[0, 3] = rep[0, 1]     # inside the first group
    rep[1, 12] = rep[1, 2]    # across groups
    rep[2, 18] = rep[2, 9]
    rep[2, 10] = rep[2, 9]
    valid[:, [1, 2, 3, 9, 10, 12, 18]] = 1
    got = ops.update_op(h.to(dev), q.to(dev), age.to(dev), rep.to(dev),
                                            valid.to(dev), c.to(dev), b.to(dev))
    hs, qs, ages = h.to(dev), q.to(dev), age.to(dev)
    olds = []
    for k in range(K):
        one = torch.zeros_like(valid)
        one[:, k] = valid[:, k]
        hs, qs, ages, old = ops.update_op(hs, qs, ages, rep.to(dev),
                                                              one.to(dev), c.to(dev), b.to(dev))
        olds.append(old[:, k])
    _close(got[0], hs.cpu(), dtype, "h")
    _close(got[1], qs.cpu(), dtype, "q")
    assert torch.equal(got[2].cpu(), ages.cpu())
    _close(got[3], torch.stack(olds, 1).cpu(), dtype, "h_old")


@pytest.mark.parametrize("B,N,K,d,deg,dtype", [
    (32, 256, 8, 64, 8, torch.float32),    # the model's round: grad_V over 16 groups of slots
    (32, 256, 8, 64, 8, torch.bfloat16),   # the same in bf16 (half the room for the partials)
    (8, 40, 80, 24, 3, torch.float32),     # K above 64: the per-wavefront grad_h kernel
    (4, 300, 64, 40, 60, torch.float32),   # rows of thousands of edges, 3 cell blocks, d off 16
    (2, 24, 4, 1024, 3, torch.float32),    # d at its limit: the forward's [16][d] rows past 64 KiB
    (3, 17, 5, 900, 2, torch.bfloat16),    # d just past the 64 KiB default, bf16
])
def test_csr_messages_backward_paths_match_oracle(ops, cuda_device, B, N, K, d, deg, dtype):
    """The CSR forward's and backward's kernels at the shapes that pick each path, against the float64
    oracle on inputs rounded to the storage dtype; hubs (cells of in-degree up to 4 deg) make
    the rows' edge lists run past one LDS block."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(B * 1000 + K)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.5).to(dtype)  # noqa: E731
    degs = torch.randint(0, deg + 1, (N,), generator=g)
    degs[: N // 10] *= 4
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), degs.cumsum(0)]).to(torch.int32)
    E = int(indptr[-1])
    indices = torch.randint(0, N, (E,), generator=g, dtype=torch.int32)
    a = torch.rand(E, generator=g).to(dtype)
    h, V, gm = rnd(B, N, d), rnd(d, d), rnd(B, K, d)
    cell_idx = torch.randint(0, N, (B, K), generator=g, dtype=torch.int32)
    cell_idx[:, 0] = 0  # every row selects a hub
    f64 = lambda t: t.double()  # noqa: E731
    dev = cuda_device
    m = ops.messages_op(h.to(dev), indptr.to(dev), indices.to(dev), a.to(dev), V.to(dev),
                         cell_idx.to(dev))  # hubs: slot lists past the forward's LDS list
    wide = d > 256
    _close(m, O.csr_messages(f64(h), indptr, indices, f64(a), f64(V), cell_idx), dtype, "m",
           scaled=wide)
    want = O.csr_messages_bwd(f64(h), indptr, indices, f64(a), f64(V), cell_idx, f64(gm))
    got = ops.messages_backward(h.to(dev), indptr.to(dev), indices.to(dev), a.to(dev),
                                    V.to(dev), cell_idx.to(dev), gm.to(dev))
    for name, g_, w_ in zip(("dh", "da", "dV"), got, want):
        _close(g_, w_, dtype, name, scaled=wide)
    again = ops.messages_backward(h.to(dev), indptr.to(dev), indices.to(dev), a.to(dev),
                                      V.to(dev), cell_idx.to(dev), gm.to(dev))
    assert all(torch.equal(x, y) for x, y in zip(got, again))


def test_unit_mlp_and_messages_are_reproducible(ops, cuda_device):
    """Every sum has a fixed order: two runs agree bit for bit."""
    v = load_golden("ref_grouped_unit_mlp.safetensors")
    D = _put(v, cuda_device, torch.float32)
    args = (D["v"], D["unit_idx"], D["W1"], D["W2"], D["hidden_saved"], D["grad_out"])
    first = ops.mlp_backward(*args)
    second = ops.mlp_backward(*args)
    assert all(torch.equal(x, y) for x, y in zip(first, second))
    v = load_golden("ref_csr_messages.safetensors")
    D = _put(v, cuda_device, torch.float32)
    args = (D["h"], D["indptr"], D["indices"], D["a"], D["V"], D["cell_idx"], D["grad_m"])
    first, second = ops.messages_backward(*args), ops.messages_backward(*args)
    assert all(torch.equal(x, y) for x, y in zip(first, second))


@pytest.mark.parametrize("P,M,d,H", [
    (40, 3, 6, 50),      # d not a multiple of 4: the scanning kernels
    (64, 4, 16, 77),     # H not a multiple of 4: the row tiles' unaligned loads
    (20000, 2, 4, 8),    # many pairs of a narrow bank: in unit order
    (300, 6, 64, 512),   # the reference model's widths: forward by row tiles, backward in unit order
    (2000, 2, 8, 64),    # both in unit order, units of several blocks
])
def test_unit_mlp_forward_paths_match_oracle(ops, cuda_device, P, M, d, H):
    """The kernels that the dispatch takes for these shapes, forward and backward, against the oracle in
    float64 on fp32 inputs (each kind of kernels over all of its shapes:
    ``test_unit_mlp_by_either_kernels_matches_oracle``)."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(P + d)
    rnd = lambda *s, scale=1.0: torch.randn(*s, generator=g) * scale  # noqa: E731
    v, b1, b2 = rnd(P, 4 * d), rnd(M, H, scale=0.1), rnd(M, d, scale=0.1)
    W1, W2 = rnd(M, 4 * d, H, scale=(4 * d) ** -0.5), rnd(M, H, d, scale=H ** -0.5)
    idx = torch.randint(0, M, (P,), generator=g, dtype=torch.int32)
    want_out, want_h = O.grouped_unit_mlp(v.double(), idx, W1.double(), b1.double(), W2.double(),
                                          b2.double())
    dev = cuda_device
    out, hidden = ops.mlp_op(v.to(dev), idx.to(dev), W1.to(dev), b1.to(dev),
                                       W2.to(dev), b2.to(dev))
    dout = rnd(P, d)
    grads = ops.mlp_backward(v.to(dev), idx.to(dev), W1.to(dev), W2.to(dev), hidden,
                                          dout.to(dev))
    want_g = O.grouped_unit_mlp_bwd(v.double(), idx, W1.double(), W2.double(),
                                    hidden.double().cpu(), dout.double())
    pairs = [("hidden", hidden, want_h), ("out", out, want_out)]
    pairs += list(zip(("dv", "dW1", "db1", "dW2", "db2"), grads, want_g))
    for name, got, want in pairs:
        # the weight gradients sum over a unit's pairs in fp32: the bar grows with the square
        # root of their count (the random walk of the roundings; 10000 pairs at P = 20000)
        bar = 1e-5 * (max(1.0, (P / M / 64) ** 0.5) if name[1] in "Wb" else 1.0)
        err = (got.double().cpu() - want).abs() / want.abs().clamp(min=1.0)
        assert float(err.max()) <= bar, f"{name}: worst {float(err.max()):.3e} (bar {bar:.1e})"


@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("counts,d,H", [
    ([1], 4, 4),                   # the smallest: one pair
    ([31, 0, 32, 33], 16, 68),     # around the 32-row tile, a unit without pairs, a hidden tail of 4
    ([5, 700, 64], 36, 100),       # 4d = 144 and d off the 64-column tiles, a unit of two blocks
    ([1500], 64, 128),             # one unit of several blocks
    ([3] * 70, 8, 64),             # more units than a wavefront's lanes
])
def test_unit_mlp_in_unit_order_matches_oracle(ops, cuda_device, counts, d, H, dtype, index):
    """The products over the pairs in unit order at the edges of their tiles, blocks and units,
    with pairs whose unit lies outside the bank: those take part in nothing (their rows of
    ``hidden``, ``out`` and ``grad_v`` are not written). Against the float64 oracle on the same
    rounded inputs; the weight gradients' bar grows with the square root of a unit's pairs."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(len(counts) * 1000 + d)
    M = len(counts)
    idx = torch.repeat_interleave(torch.arange(M), torch.tensor(counts))
    idx = idx[torch.randperm(idx.numel(), generator=g)]
    outside = torch.tensor([-1, M, 2**31 - 1])
    all_idx = torch.cat([idx[:1], outside, idx[1:]]) if idx.numel() > 1 else idx
    kept = (all_idx >= 0) & (all_idx < M)
    P = all_idx.numel()
    rnd = lambda *s, scale=0.5: (torch.randn(*s, generator=g) * scale).to(dtype)  # noqa: E731
    v, W1, b1 = rnd(P, 4 * d), rnd(M, 4 * d, H, scale=(4 * d) ** -0.5), rnd(M, H)
    W2, b2, dout = rnd(M, H, d, scale=H ** -0.5), rnd(M, d), rnd(P, d)
    dev = cuda_device
    D = [t.to(dev) for t in (v, all_idx.to(index), W1, b1, W2, b2)]
    out, hidden = ops.mlp_op(*D)
    got = ops.mlp_backward(D[0], D[1], D[2], D[4], hidden, dout.to(dev))
    f64 = [t.double() for t in (v[kept], W1, b1, W2, b2, dout[kept])]
    want_out, want_h = O.grouped_unit_mlp(f64[0], idx, *f64[1:5])
    _close(hidden.cpu()[kept], want_h, dtype, "hidden")
    _close(out.cpu()[kept], want_out, dtype, "out")
    want = O.grouped_unit_mlp_bwd(f64[0], idx, f64[1], f64[3], hidden.cpu()[kept].double(), f64[5])
    _close(got[0].cpu()[kept], want[0], dtype, "grad_v")
    bar = TOL[dtype] * max(1.0, (max(counts) / 64) ** 0.5)
    for name, g_, w_ in zip(("dW1", "db1", "dW2", "db2"), got[1:], want[1:]):
        err = (g_.double().cpu() - w_).abs() / w_.abs().clamp(min=1.0)
        assert float(err.max()) <= bar, f"{name}: worst {float(err.max()):.3e} (bar {bar:.1e})"
    again = ops.mlp_backward(D[0], D[1], D[2], D[4], hidden, dout.to(dev))
    for a, b in zip(got[1:], again[1:]):
        assert torch.equal(a, b)  # every sum has a fixed order


def test_unit_mlp_takes_operands_off_the_four_element_alignment(ops, cuda_device):
    """A view into a buffer, one element in: the kernels without a workspace take it, with the
    same results up to the order of the fp32 sums."""
    g = torch.Generator().manual_seed(5)
    P, M, d, H = 40, 3, 16, 64
    dev = cuda_device
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.3).to(dev)  # noqa: E731
    v, W1, b1, W2, b2 = rnd(P, 4 * d), rnd(M, 4 * d, H), rnd(M, H), rnd(M, H, d), rnd(M, d)
    idx = torch.randint(0, M, (P,), generator=g).to(dev)
    shifted = torch.empty(v.numel() + 1, device=dev)[1:].view(P, 4 * d).copy_(v)
    for a, b in zip(ops.mlp_op(v, idx, W1, b1, W2, b2), ops.mlp_op(shifted, idx, W1, b1, W2, b2)):
        torch.testing.assert_close(a, b, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,N,K,d", [(1, 1, 1, 4), (3, 130, 19, 36), (2, 64, 8, 6), (2, 65, 9, 300)])
def test_update_into_fresh_tensors_equals_the_update_in_place(ops, cuda_device, B, N, K, d, dtype):
    """The copies and their update in two launches give the copies' in-place update bit for bit: an
    element count off the 16-byte copies, d above the workgroup's threads, padded slots, and cells
    repeated inside a batch of 8 slots and across batches."""
    g = torch.Generator().manual_seed(B * 100 + N)
    dev = cuda_device
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    h, q, c, b = rnd(B, N, d), rnd(B, d), rnd(B, K, d), rnd(B, K, d)
    cells = torch.randint(0, N, (B, K), generator=g)
    if K > 8:
        cells[0, 5], cells[0, K - 1] = cells[0, 2], cells[0, 2]
    valid = torch.rand(B, K, generator=g) > 0.2
    age = torch.randint(0, 9, (B, N), generator=g)
    h2, q2, age2 = h.clone(), q.clone(), age.to(torch.int32).to(dev)
    old = ops.update_inplace(h2, q2, age2, cells.to(torch.int32).to(dev),
                             valid.to(torch.int32).to(dev), c, b)
    for dt in (torch.int32, torch.int64):
        got = ops.update_op(h, q, age.to(dt).to(dev), cells.to(dev), valid.to(dev), c, b)
        assert got[2].dtype == dt
        for name, x, y in zip(("h", "q", "age", "old"), got, (h2, q2, age2.to(dt), old)):
            assert torch.equal(x, y), name


@pytest.mark.parametrize("E_extra", [0, 5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ops_read_either_index_width(ops, cuda_device, dtype, E_extra):
    """int64 indices and bool flags read in place give the int32 arrays' results bit for bit, in
    every op that takes them; the messages on uneven rows, more than one block of cells a
    workgroup, and (``E_extra``) edges past the last row, whose grad_a is zero."""
    from oracle import hsn_oracle as O

    g = torch.Generator().manual_seed(77 + E_extra)
    dev = cuda_device
    B, N, K, d = 300, 270, 5, 20
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.5).to(dtype)  # noqa: E731
    cells = torch.randint(0, N, (B, K), generator=g)
    valid = torch.rand(B, K, generator=g) > 0.2
    deg = torch.randint(0, 6, (N,), generator=g)
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), deg.cumsum(0)])
    E = int(indptr[-1]) + E_extra
    indices = torch.randint(0, N, (E,), generator=g)
    h, V, a, dm = rnd(B, N, d), rnd(d, d), rnd(E), rnd(B, K, d)
    u, eps, q, G, dv = rnd(B, d), rnd(B, d), rnd(B, d), rnd(B, N, d), rnd(B, K, 4 * d)
    D = {k: t.to(dev) for k, t in dict(h=h, V=V, a=a, dm=dm, u=u, eps=eps, q=q, G=G, dv=dv).items()}

    def run(i, f):
        cell, ip, ix, ok = (cells.to(i).to(dev), indptr.to(i).to(dev), indices.to(i).to(dev),
                            valid.to(f).to(dev))
        out = [ops.messages_op(D["h"], ip, ix, D["a"], D["V"], cell),
               *ops.messages_backward(D["h"], ip, ix, D["a"], D["V"], cell, D["dm"]),
               ops.gather_op(D["u"], D["eps"], D["h"], D["dm"], cell),
               *ops.gather_backward(D["dv"], cell, N),
               *ops.update_backward(cell, ok, D["dm"], D["dm"], D["dm"], D["G"], D["q"])]
        return out

    wide, narrow = run(torch.int64, torch.bool), run(torch.int32, torch.int32)
    for i, (x, y) in enumerate(zip(wide, narrow)):
        assert torch.equal(x, y), i
    want = O.csr_messages_bwd(h.double(), indptr, indices[:E - E_extra], a[:E - E_extra].double(),
                              V.double(), cells, dm.double())
    _close(wide[1], want[0], dtype, "grad_h")
    _close(wide[2][:E - E_extra], want[1], dtype, "grad_a", scaled=True)
    assert bool((wide[2][E - E_extra:] == 0).all())
    _close(wide[3], want[2], dtype, "grad_V", scaled=True)
    mixed = ops.messages_op(D["h"], indptr.to(dev), indices.to(torch.int32).to(dev), D["a"], D["V"],
                            cells.to(dev))
    assert torch.equal(mixed, wide[0])


def _through(monkeypatch, ops, path):
    """Sends the unit MLP through one kind of kernels whatever the dispatch would take: ``unit order``
    (a workspace) or ``by rows`` (none)."""
    real = ops._mlp_space

    def space(P, M, d, H, backward, idx, v, *operands):
        if path == "by rows":
            return None
        if backward:
            return real(P, M, d, H, backward, idx, v, *operands)
        nbytes = 4 * P * (H + 3) + 16 * M + 8192  # a forward's rows, pairs and units
        ws = torch.empty(nbytes, dtype=torch.uint8, device=v.device)
        return idx.contiguous(), 64 if idx.dtype == torch.int64 else 32, ws, nbytes

    monkeypatch.setattr(ops, "_mlp_space", space)


def _mlp_problem(P, M, d, H, dtype, seed, dev, index=torch.int32):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s, scale=0.5: (torch.randn(*s, generator=g) * scale).to(dtype).to(dev)  # noqa: E731
    return dict(v=rnd(P, 4 * d), idx=torch.randint(0, M, (P,), generator=g).to(index).to(dev),
                W1=rnd(M, 4 * d, H, scale=(4 * d) ** -0.5), b1=rnd(M, H),
                W2=rnd(M, H, d, scale=H ** -0.5), b2=rnd(M, d), dout=rnd(P, d))


def _mlp_run(ops, x):
    out, hidden = ops.mlp_op(x["v"], x["idx"], x["W1"], x["b1"], x["W2"], x["b2"])
    return out, hidden, ops.mlp_backward(x["v"], x["idx"], x["W1"], x["W2"], hidden, x["dout"])


@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("path", ["unit order", "by rows"])
@pytest.mark.parametrize("P,M,d,H", [
    (130, 3, 16, 68),     # several row tiles a unit, a hidden tail; the forward of few pairs
    (700, 6, 64, 512),    # the model's widths, more pairs than the forward of few takes in fp32
    (17000, 2, 4, 8),     # more pairs than the row tiles' slot table: the scanning kernels
    (2000, 2, 8, 64),     # grad_W2 too small to hold dz1: grad_v in one launch by rows
    (2000, 2, 8, 66),     # the same, W1's rows off the four-element loads (by rows only)
])
def test_unit_mlp_by_either_kernels_matches_oracle(ops, cuda_device, monkeypatch, P, M, d, H, path, dtype,
                                                   index):
    """The kernels over the pairs in unit order and those over rows, each at both sides of the sizes
    at which the dispatch changes from one to the other, forward and backward against the float64
    oracle on the same rounded inputs; the weight gradients' bar grows with the square root of a
    unit's pairs."""
    from oracle import hsn_oracle as O

    if H % 4:
        path = "by rows"
    x = _mlp_problem(P, M, d, H, dtype, P + d, cuda_device, index)
    _through(monkeypatch, ops, path)
    out, hidden, got = _mlp_run(ops, x)
    c = {k: t.cpu().double() if t.is_floating_point() else t.cpu() for k, t in x.items()}
    want_out, want_h = O.grouped_unit_mlp(c["v"], c["idx"], c["W1"], c["b1"], c["W2"], c["b2"])
    _close(hidden, want_h, dtype, "hidden")
    _close(out, want_out, dtype, "out")
    want = O.grouped_unit_mlp_bwd(c["v"], c["idx"], c["W1"], c["W2"], hidden.cpu().double(), c["dout"])
    _close(got[0], want[0], dtype, "grad_v")
    bar = TOL[dtype] * max(1.0, (P / M / 64) ** 0.5)
    for name, g_, w_ in zip(("dW1", "db1", "dW2", "db2"), got[1:], want[1:]):
        err = (g_.double().cpu() - w_).abs() / w_.abs().clamp(min=1.0)
        assert float(err.max()) <= bar, f"{name}: worst {float(err.max()):.3e} (bar {bar:.1e})"


def _four_shares(x, W, b):
    """``x @ W + b`` as four running fp32 sums of a quarter of the reduction each, added in order."""
    K, total = x.shape[1], None
    for s in range(4):
        acc = torch.zeros(x.shape[0], W.shape[1], device=x.device)
        for k in range(s * K // 4, (s + 1) * K // 4):
            acc = (acc.double() + x[:, k:k + 1].double() * W[k].double()).float()
        total = acc if total is None else total + acc
    return total + b


@pytest.mark.parametrize("path", ["unit order", "by rows"])
@pytest.mark.parametrize("d,H", [(4, 64), (16, 64), (16, 512), (32, 64), (64, 64), (64, 512)])
def test_unit_mlp_sums_are_no_further_off_than_four_running_sums(ops, cuda_device, monkeypatch, d, H, path):
    """In fp32 both layers' results are no further from 64 bits than four running sums of a quarter of
    the reduction each leave them on the same inputs. Within 10%: the matrix instruction's order inside
    four products and the activation's erf are not torch's, at most a rounding each of the some fifteen
    and more behind a result; longer sums were 1.2 to 1.7 times as far off."""
    x = _mlp_problem(2000, 1, d, H, torch.float32, d + H, cuda_device)
    _through(monkeypatch, ops, path)
    out, hidden = ops.mlp_op(x["v"], x["idx"], x["W1"], x["b1"], x["W2"], x["b2"])
    gelu = lambda z: 0.5 * z * (1 + torch.erf(z * 0.5 ** 0.5))  # noqa: E731
    c = {k: x[k].double() if x[k].dim() < 3 else x[k][0].double() for k in ("v", "W1", "b1", "W2", "b2")}
    want_z = c["v"] @ c["W1"] + c["b1"]
    want = gelu(want_z) @ c["W2"] + c["b2"]
    z = _four_shares(x["v"], x["W1"][0], x["b1"])
    act = 0.5 * z * (1 + torch.erf(z * 0.5 ** 0.5))  # in fp32, as the kernels take it
    y = _four_shares(act, x["W2"][0], x["b2"])
    off = lambda a, b: float((a.double() - b).norm() / b.norm())  # noqa: E731
    assert off(hidden, want_z) <= 1.1 * off(z, want_z)
    assert off(out, want) <= 1.1 * off(y, want)


def test_unit_mlp_without_memory_for_a_workspace(ops, cuda_device, monkeypatch):
    """Where no workspace can be had the kernels over rows take the call: a bank that fits the memory
    runs, with the same results up to the order of the fp32 sums."""
    x = _mlp_problem(600, 4, 16, 64, torch.float32, 9, cuda_device)
    out, hidden, got = _mlp_run(ops, x)
    real = torch.empty

    def full(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no memory")
        return real(*size, **kw)

    monkeypatch.setattr(ops.torch, "empty", full)
    out2, hidden2, got2 = _mlp_run(ops, x)
    for a, b in zip((out, hidden, *got), (out2, hidden2, *got2)):
        torch.testing.assert_close(a, b, atol=2e-5, rtol=2e-5)
