"""Recurrences with one decay a head in steps of about a token a row: the kernel that takes four columns a lane forms every sum in the order of the one
that walks rows of many tokens (equal bits), at the edges of its channels, columns and alignments, and agrees with 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


@pytest.mark.parametrize("types", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("heads, group, dim, vdim, offset", [(3, 1, 8, 4, 0), (4, 2, 64, 64, 0), (2, 1, 56, 68, 0), (6, 3, 112, 100, 0), (8, 1, 128, 256, 0), (4, 4, 128, 64, 0),
                                                             (2, 1, 72, 32, 0), (2, 1, 128, 66, 0), (2, 1, 64, 64, 1), (1, 1, 256, 64, 0)])
def test_one_token_a_row(ops, types, heads, group, dim, vdim, offset):
    print(f"memory single {types} {heads} {group} {dim} {vdim} {offset}", flush=True)
    torch.manual_seed(dim + vdim)
    T, V = types
    code = lambda dtype: 0 if dtype == torch.float32 else 1
    lengths, before = [1, 0, 1, 2, 0, 1, 1], [0, 0, 5, 3, 9, 1, 7]            # as many tokens as six of the seven rows
    rows, n = len(lengths), sum(lengths)
    keys = heads // group
    q, k = (torch.randn(n * keys * dim + offset, device="cuda").to(T)[offset:].view(n, keys * dim) for _ in range(2))
    v = torch.randn(n, heads * vdim, device="cuda").to(V)
    log_keep, take = -torch.rand(n, heads, device="cuda"), torch.rand(n, heads, device="cuda")
    start_state = torch.randn(rows + 2, heads * dim * vdim, device="cuda")
    slots = torch.randperm(rows + 2)[:rows].int().cuda()
    to = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    first, length, context = to([sum(lengths[:r]) for r in range(rows)]), to(lengths), to([a + b for a, b in zip(lengths, before)])
    lib, p, results = ops._part_library("recurrent"), lambda tensor: tensor.data_ptr(), []
    for tokens in (0, n):                                                         # not known: the walk over many tokens
        state, out = start_state.clone(), torch.full((n, heads * vdim), float("nan"), device="cuda")
        assert lib.lsa_decayed_recurrence(code(T), p(q), q.stride(0), p(k), k.stride(0), code(V), p(v), v.stride(0), p(log_keep), heads, p(take), 0.5, p(state),
                                          state.stride(0), p(slots), p(first), p(length), p(context), p(out), rows, heads, group, dim, vdim, None, None, tokens,
                                          torch.cuda.current_stream().cuda_stream) == 0
        results.append((out, state))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    out, state = results[1]
    want, moved = torch.empty_like(out, dtype=torch.float64), start_state.double()
    for r in range(rows):
        S = moved[slots[r]].view(heads, dim, vdim).clone() * (before[r] > 0)
        for t in range(int(first[r]), int(first[r]) + lengths[r]):
            kk, qq = (x[t].double().view(keys, dim).repeat_interleave(group, 0) for x in (k, q))
            S = S * log_keep[t].double().exp()[:, None, None] + take[t].double()[:, None, None] * kk[:, :, None] * v[t].double().view(heads, 1, vdim)
            want[t] = (S * qq[:, :, None] * 0.5).sum(1).flatten()
        if lengths[r]:
            moved[slots[r]] = S.flatten()
    # chains of 8 or 16 products and 8 sums in float32: a few dozen roundings of numbers of a sum's size
    torch.testing.assert_close(out.double(), want, rtol=1e-5, atol=64 * 2.0 ** -24 * float(want.abs().max()))
    torch.testing.assert_close(state.double(), moved, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, dim, vdim", [(2, 64, 64), (3, 128, 256), (2, 24, 40), (1, 128, 60)])
def test_one_token_a_row_with_a_normaliser(ops, dtype, heads, dim, vdim):
    print(f"memory single normaliser {dtype} {heads} {dim} {vdim}", flush=True)
    torch.manual_seed(dim + vdim)
    rows = n = 5
    q, k, v = (torch.randn(n, heads * size, device="cuda").to(dtype) for size in (dim, dim, vdim))
    gates = torch.randn(n, 2 * heads, device="cuda")
    start_state = torch.randn(rows + 1, heads * dim * vdim + heads * dim + heads + -heads % 4, device="cuda")
    slots = torch.randperm(rows + 1)[:rows].int().cuda()
    first, length = torch.arange(n, device="cuda", dtype=torch.int32), torch.ones(n, device="cuda", dtype=torch.int32)
    context = torch.tensor([1, 2, 9, 1, 4], dtype=torch.int32, device="cuda")
    lib, p, results = ops._part_library("recurrent"), lambda tensor: tensor.data_ptr(), []
    for tokens in (0, n):
        state, out = start_state.clone(), torch.full((n, heads * vdim), float("nan"), device="cuda")
        below, coef = torch.full((n, heads, 2), float("nan"), device="cuda"), torch.empty(n, heads, 2, device="cuda")
        assert lib.lsa_matrix_memory(0 if dtype == torch.float32 else 1, p(q), q.stride(0), p(k), k.stride(0), p(v), v.stride(0), p(gates), 15.0, 0.125, p(state),
                                     state.stride(0), p(slots), p(first), p(length), p(context), p(coef), p(out), p(below), rows, heads, dim, vdim, None, None, tokens,
                                     torch.cuda.current_stream().cuda_stream) == 0
        results.append((out, state, below))
    assert all(torch.equal(a, b) for a, b in zip(*results)) and torch.isfinite(results[1][0]).all() and torch.isfinite(results[1][2]).all()
