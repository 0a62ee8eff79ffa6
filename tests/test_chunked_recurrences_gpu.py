"""The recurrences that run long portions in chunks, against the same recurrence token by token in float64.

What a result may be off by is what the kernel that walks the tokens one by one is off by on the same numbers (2-norm over a step): both
form sums of as many float32 products, the chunks in short partial sums that meet in 64 bits.  A quarter more, and half a unit in the
last place (HALF_UNIT) for results of a few numbers, of which the norm is a chance matter, bound the chunked form's; read-outs of the
kernel of 64 columns, which adds scores' and state's products in one long 32-bit sum, are allowed twice the walk's."""
import pytest
import torch

from test_latent_experts_kernels_gpu import batch

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]
HALF_UNIT = 2.0 ** -25


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


def off(x, exact):
    return float((x.double() - exact).norm() / exact.norm())


def plain_recurrence(q, k, v, decay, bonus, state):
    """One row in float64: q, k, decay [T, heads, dim], v [T, heads, vdim], state [heads, dim, vdim] -> (read-outs, state)."""
    out = []
    for t in range(q.shape[0]):
        kv = k[t][..., None] * v[t][:, None]
        read = state * decay[t][..., None] + kv if bonus is None else state + bonus[..., None] * kv
        out.append((q[t][:, None] @ read)[:, 0])
        state = state * decay[t][..., None] + kv
    return torch.stack(out), state


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,dim,vdim,mode,spread", [(2, 128, 128, "double_exp", 1.0), (3, 24, 40, "sigmoid_root", 2.0), (1, 64, 130, "double_exp", 3.0),
                                                        (2, 65, 256, "sigmoid_root", 1.0), (1, 5, 1, "double_exp", 6.0)])
def test_linear_recurrence_in_chunks(ops, dtype, heads, dim, vdim, mode, spread):
    """Rows that end inside a block of 16, inside and at the end of a chunk of 64, a single token, an empty row; a second step from kept
    states, a used slot that starts again; decays from next to nothing to next to one; scratch memory full of what is no number."""
    print(f"linear_recurrence in chunks {dtype} {heads} {dim} {vdim} {mode}", flush=True)
    generator = torch.Generator("cuda").manual_seed(dim)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    size, offset = heads * dim * vdim, 3
    start = draw(6, offset + size)
    slots = torch.tensor([4, 0, 2, 5, 1], dtype=torch.int32, device="cuda")
    bias = draw(heads * dim)
    bonus = draw(heads, dim) if mode == "double_exp" else None
    states = {"scan": start.clone(), "chunks": start.clone()}
    exact_states = start.double()
    firsts = [0] * 5
    for step, lengths in enumerate(([130, 1, 64, 0, 79], [15, 200, 65, 3, 128])):
        if step == 1:
            firsts[2] = 0
        _, _, row_start, row_len, row_ctx = batch(lengths, firsts, "cuda")
        n = sum(lengths)
        proj = (0.5 * draw(n, 2 * heads * dim + heads * vdim + 3)).to(dtype)
        q, k, v = proj[:, :heads * dim], proj[:, heads * dim:2 * heads * dim], proj[:, 2 * heads * dim:2 * heads * dim + heads * vdim]
        decay = spread * draw(n, heads * dim) - 1.0
        chunks = n // 64 + len(lengths)
        scratch = {"sums": torch.full((chunks, heads, dim, vdim), float("nan"), device="cuda"),
                   "totals": torch.full((chunks, heads, dim), float("nan"), device="cuda"),
                   "queries": torch.full((n, heads, dim), float("nan"), device="cuda")}
        outs = {}
        for form, more in (("scan", {}), ("chunks", scratch)):
            outs[form] = torch.full((n, heads * vdim), float("nan"), device="cuda")
            ops.linear_recurrence(q, k, v, decay, bias, mode, 4.0, bonus, 0.3, states[form], offset, slots, row_start, row_len, row_ctx, outs[form],
                                  heads, dim, vdim, **more)
        z = decay.double() + bias.double()
        factor = torch.exp(-torch.exp(z)) if mode == "double_exp" else torch.exp(torch.nn.functional.logsigmoid(z) / 4.0)
        wide = lambda x, width: x.double().reshape(n, heads, width)
        exact = torch.empty(n, heads, vdim, device="cuda", dtype=torch.float64)
        at = 0
        for row, length in enumerate(lengths):
            slot, piece = int(slots[row]), slice(at, at + length)
            at += length
            if not length:
                continue
            before = exact_states[slot, offset:].view(heads, dim, vdim)
            before = torch.zeros_like(before) if firsts[row] == 0 else before
            exact[piece], after = plain_recurrence(0.3 * wide(q, dim)[piece], wide(k, dim)[piece], wide(v, vdim)[piece], wide(factor, dim)[piece],
                                                   None if bonus is None else bonus.double(), before)
            exact_states[slot, offset:] = after.reshape(-1)
        errors = {form: (off(outs[form], exact.reshape(n, -1)), off(states[form], exact_states)) for form in outs}
        print(errors, flush=True)
        for scan, chunked in zip(errors["scan"], errors["chunks"]):
            assert chunked <= 1.25 * scan + HALF_UNIT
        assert torch.equal(states["chunks"][3], start[3]) and torch.equal(states["chunks"][:, :offset], start[:, :offset])
        firsts = [first + length for first, length in zip(firsts, lengths)]


def test_which_steps_run_their_recurrences_in_chunks(ops):
    def chunks(lengths, heads=16, dim=128, vdim=128):
        return ops.linear_recurrence_chunks(sum(lengths), len(lengths), max(lengths), heads, dim, vdim)
    assert chunks([2048]) == 33 and chunks([512] + [1] * 16) == 25 and chunks([2048] * 4, vdim=256) == 132
    assert not chunks([64]) and not chunks([1] * 32) and not chunks([16] * 32) and not chunks([112] + [1] * 64) and not chunks([2048], dim=129)


def plain_delta(q, k, v, decay, beta, state):
    """One row in float64: q, k, decay [T, heads, dim], v [T, heads, vdim], beta [T, heads], state [heads, dim, vdim] -> (read-outs, state)."""
    out = []
    for t in range(q.shape[0]):
        state = state * decay[t][..., None]
        u = beta[t][:, None] * (v[t] - (k[t][:, None] @ state)[:, 0])
        state = state + k[t][..., None] * u[:, None]
        out.append((q[t][:, None] @ state)[:, 0])
    return torch.stack(out), state


# Value columns that end inside the second 64 of a workgroup's 128, in its first number, and inside a third.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,dim,vdim", [(2, 96, 100), (1, 128, 65), (2, 33, 150)])
def test_linear_recurrence_in_chunks_at_the_edges_of_value_columns(ops, dtype, heads, dim, vdim):
    test_linear_recurrence_in_chunks(ops, dtype, heads, dim, vdim, "double_exp" if vdim == 100 else "sigmoid_root", 1.0)


def in_chunks(ops, q, k, v, decay, heads, dim, vdim):
    """Read-outs of one row from an empty state, without a bonus and with queries as they are."""
    n, ints = q.shape[0], lambda x: torch.tensor([x], dtype=torch.int32, device="cuda")
    out = torch.full((n, heads * vdim), float("nan"), device="cuda")
    state = torch.zeros(1, heads * dim * vdim, device="cuda")
    scratch = {"sums": torch.full((n // 64 + 1, heads, dim, vdim), float("nan"), device="cuda"), "totals": torch.full((n // 64 + 1, heads, dim), float("nan"), device="cuda"),
               "queries": torch.full((n, heads, dim), float("nan"), device="cuda")}
    ops.linear_recurrence(q, k, v, decay, None, "double_exp", 1.0, None, 1.0, state, 0, ints(0), ints(0), ints(n), ints(n), out, heads, dim, vdim, **scratch)
    return out, state


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("spoilt", [slice(64, 128), slice(0, 64), slice(128, 200)])
def test_values_that_are_no_numbers_leave_other_columns_as_they_are(ops, dtype, spoilt):
    """Whether products run on matrix cores or number by number is decided for 64 value columns, not for all that a workgroup has: the other columns' read-outs and states are the
    same bits with and without infinities beside them."""
    generator = torch.Generator("cuda").manual_seed(3)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    n, heads, dim, vdim = 150, 2, 128, 200
    q, k, v = (0.5 * draw(n, heads * width) for width in (dim, dim, vdim))
    q, k, v, decay = q.to(dtype), k.to(dtype), v.to(dtype), draw(n, heads * dim) - 1.0
    print(f"no numbers in columns {spoilt} {dtype}", flush=True)
    whole, state = in_chunks(ops, q, k, v, decay, heads, dim, vdim)
    v.view(n, heads, vdim)[70, 1, spoilt] = float("inf")
    beside, state_beside = in_chunks(ops, q, k, v, decay, heads, dim, vdim)
    kept = torch.ones(heads, vdim, dtype=torch.bool, device="cuda")
    kept[1, spoilt] = False
    assert bool(whole.isfinite().all()) and not bool(beside.view(n, heads, vdim)[70:, 1, spoilt].isfinite().any())
    assert torch.equal(whole.view(n, heads, vdim)[:, kept], beside.view(n, heads, vdim)[:, kept])
    kept = kept[:, None].expand(heads, dim, vdim)
    assert torch.equal(state.view(heads, dim, vdim)[kept], state_beside.view(heads, dim, vdim)[kept])


@pytest.mark.parametrize("token", [0, 8, 15, 40])
def test_scores_meet_in_the_order_of_the_halves_of_the_channels(ops, token):
    """A score inside a block of tokens is the first half's sum, rounded, and the second half's: 2^24 + 1 and 1 are 2^24 then, however many wavefronts share the channels and the tokens
    back.  The token at `token` reads the one at the start of its block, with nothing lost on the way."""
    n, heads, dim, vdim = 64, 1, 128, 64
    q, k, v = (torch.zeros(n, width, device="cuda") for width in (dim, dim, vdim))
    source = token // 16 * 16
    q[token, 0], k[source, 0] = 2.0 ** 12, 2.0 ** 12
    q[token, 1], k[source, 1] = 1.0, 1.0
    q[token, 64], k[source, 64] = 1.0, 1.0
    v[source] = 1.0
    print(f"order of halves, token {token}", flush=True)
    out, _ = in_chunks(ops, q, k, v, torch.full((n, dim), -200.0, device="cuda"), heads, dim, vdim)
    expected = torch.zeros(n, vdim, device="cuda")
    expected[token] = 2.0 ** 24
    assert torch.equal(out, expected)


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,spread", [(2, 2, 128, 128, 1.0), (3, 3, 24, 40, 2.0), (4, 2, 64, 130, 3.0), (2, 1, 65, 256, 0.5),
                                                            (1, 1, 5, 1, 6.0)])
def test_delta_rule_in_chunks(ops, per_channel, heads, kv_heads, dim, vdim, spread):
    """The same rows, slots and scratch memory; keys that repeat those in front of them, which a write has to take back."""
    print(f"delta_rule in chunks {per_channel} {heads} {kv_heads} {dim} {vdim}", flush=True)
    generator = torch.Generator("cuda").manual_seed(dim)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    columns, group = -(-vdim // 16) * 16, heads // kv_heads
    size = heads * dim * columns
    turned = lambda flat: flat[..., :size].view(-1, heads, columns // 16, dim, 16).permute(0, 1, 3, 2, 4).reshape(-1, heads, dim, columns)[..., :vdim]
    start = draw(6, size + 8)
    start[:, :size].view(6, heads, columns // 16, dim, 16)[:, :, -1, :, vdim - columns + 16:] = 0
    slots = torch.tensor([4, 0, 2, 5, 1], dtype=torch.int32, device="cuda")
    states = {"scan": start.clone(), "chunks": start.clone()}
    exact_states = turned(start).double()
    firsts = [0] * 5
    for step, lengths in enumerate(([130, 1, 64, 0, 79], [15, 200, 65, 3, 128])):
        if step == 1:
            firsts[2] = 0
        _, _, row_start, row_len, row_ctx = batch(lengths, firsts, "cuda")
        n = sum(lengths)
        q, k = draw(n, kv_heads, dim), draw(n, kv_heads, dim)
        k[1::3] = k[0::3][:k[1::3].shape[0]] + 0.1 * k[1::3]
        q, k = q / q.norm(dim=-1, keepdim=True) * dim ** -0.5, k / k.norm(dim=-1, keepdim=True)
        v, beta = draw(n, heads, vdim), torch.sigmoid(2 * draw(n, heads))
        decay = torch.exp(-torch.exp(spread * draw(n, heads * dim if per_channel else heads) - 2.0))
        prepared = torch.cat([x.reshape(n, -1) for x in (q, k, v)], dim=1)
        chunks = n // 64 + len(lengths)
        shape = ops.delta_rule_scratch(n, len(lengths), 10 ** 6, heads, dim, vdim)
        assert shape[:2] == (chunks, heads)
        outs = {}
        for form, more in (("scan", {}), ("chunks", {"scratch": torch.full(shape, float("nan"), device="cuda")})):
            outs[form] = torch.full((n, heads * vdim), float("nan"), device="cuda")
            ops.delta_rule(prepared, beta, decay, per_channel, states[form], 0, slots, row_start, row_len, row_ctx, outs[form], heads, kv_heads, dim,
                           vdim, **more)
        wide = lambda x: x.double().repeat_interleave(group, dim=1)
        factor = decay.double().view(n, heads, -1).expand(n, heads, dim)
        exact = torch.empty(n, heads, vdim, device="cuda", dtype=torch.float64)
        at = 0
        for row, length in enumerate(lengths):
            slot, piece = int(slots[row]), slice(at, at + length)
            at += length
            if not length:
                continue
            before = torch.zeros_like(exact_states[slot]) if firsts[row] == 0 else exact_states[slot]
            exact[piece], exact_states[slot] = plain_delta(wide(q)[piece], wide(k)[piece], v.double()[piece], factor[piece], beta.double()[piece], before)
        errors = {form: (off(outs[form], exact.reshape(n, -1)), off(turned(states[form]), exact_states)) for form in outs}
        print(errors, flush=True)
        for scan, chunked in zip(errors["scan"], errors["chunks"]):
            assert chunked <= 1.25 * scan + HALF_UNIT
        assert torch.equal(states["chunks"][3], start[3]) and torch.equal(states["chunks"][:, size:], start[:, size:])
        padding = states["chunks"][:, :size].view(6, heads, columns // 16, dim, 16)[:, :, -1, :, vdim - columns + 16:]
        assert not padding.any()
        firsts = [first + length for first, length in zip(firsts, lengths)]


def test_which_steps_run_their_delta_rules_in_chunks(ops):
    def shape(lengths, heads=16, dim=128, vdim=128):
        return ops.delta_rule_scratch(sum(lengths), len(lengths), max(lengths), heads, dim, vdim)
    assert shape([1900])[:2] == (30, 16) and shape([512] + [1] * 16)[:2] == (25, 16) and shape([2048] * 4)[:2] == (132, 16)
    assert not shape([160]) and not shape([1] * 32) and not shape([64] * 16) and not shape([2048], dim=129)


@pytest.mark.parametrize("spare", [0, 600])
@pytest.mark.parametrize("heads,key_heads,dim,vdim", [(2, 2, 32, 31), (2, 2, 96, 1), (1, 1, 128, 257), (3, 3, 64, 128), (4, 2, 128, 96), (2, 1, 32, 33)])
def test_read_outs_of_16_bit_queries_in_chunks(ops, heads, key_heads, dim, vdim, spare):
    """Heads of whole steps of 32 channels, rows at multiples of 16 bytes: what a chunk's tokens read is made by wavefronts of 32 columns where the
    scratch memory makes for enough workgroups (``spare`` chunks that the rows do not have).  As many
    heads of keys as heads: the memory with its normaliser; fewer: a decay and a strength a head.  The kept numbers are the kernel's own
    (32-bit), so the float64 walk starts from the same ones."""
    print(f"read-outs in chunks {heads} {key_heads} {dim} {vdim}", flush=True)
    generator = torch.Generator("cuda").manual_seed(vdim)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    lengths, firsts, memory = [130, 1, 64, 79, 15], [0, 7, 3, 0, 2], heads == key_heads
    n, size = sum(lengths), heads * dim * vdim
    _, _, row_start, row_len, row_ctx = batch(lengths, firsts, "cuda")
    slots = torch.tensor([4, 0, 2, 3, 1], dtype=torch.int32, device="cuda")
    width = (2 * key_heads * dim + heads * vdim + 7) // 8 * 8
    proj = (0.5 * draw(n, width)).to(torch.bfloat16)
    q, k, v = (proj[:, at:at + size] for at, size in ((0, key_heads * dim), (key_heads * dim, key_heads * dim), (2 * key_heads * dim, heads * vdim)))
    assert q.stride(0) % 8 == 0 and (q.data_ptr() | k.data_ptr()) % 16 == 0
    start = draw(5, size + heads * dim + heads)
    start[:, -heads:] = 0.5
    chunks, ones = n // 64 + len(lengths) + spare, 1 if memory else 0
    sums = torch.full((chunks, heads, dim, vdim + ones), float("nan"), device="cuda")
    gates = 3 * draw(n, 2 * heads) + 2.0
    log_keep, take = -torch.nn.functional.softplus(2 * draw(n, heads) - 2.0), torch.sigmoid(draw(n, heads))
    results = {}
    for form in ("scan", "chunks"):
        state, out = start.clone(), torch.full((n, heads * vdim), float("nan"), device="cuda")
        below, coefficients = torch.zeros(n, heads, 2, device="cuda"), torch.zeros(n, heads, 2, device="cuda")
        places = (state, slots, row_start, row_len, row_ctx, out)
        if memory:
            more = {} if form == "scan" else {"run": torch.full((n, heads), float("nan"), device="cuda", dtype=torch.float64), "sums": sums}
            ops.matrix_memory(q, k, v, gates, 15.0, 0.25, *places, below, coefficients, heads, dim, vdim, **more)
        else:
            more = {} if form == "scan" else {"sums": sums, "totals": torch.full((chunks, heads), float("nan"), device="cuda")}
            ops.decayed_recurrence(q, k, v, log_keep, take, 0.25, *places, heads, key_heads, dim, vdim, **more)
        results[form] = (out, below[..., 0].clone(), coefficients)
    keep, strength = (results["scan"][2].double().unbind(-1)) if memory else (torch.exp(log_keep.double()), take.double())
    wide = lambda x: 1.0 * x.double().reshape(n, key_heads, dim).repeat_interleave(heads // key_heads, dim=1)
    values = torch.cat([v.double().reshape(n, heads, vdim), torch.ones(n, heads, 1, device="cuda", dtype=torch.float64)], dim=2)
    exact = torch.empty(n, heads, vdim + 1, device="cuda", dtype=torch.float64)
    at = 0
    for row, length in enumerate(lengths):
        kept = start[int(slots[row])].double()
        before = torch.cat([kept[:size].view(heads, dim, vdim), kept[size:size + heads * dim].view(heads, dim, 1)], dim=2)
        piece = slice(at, at + length)
        exact[piece], _ = plain_recurrence(0.25 * wide(q)[piece], wide(k)[piece] * strength[piece][..., None], values[piece],
                                           keep[piece][..., None].expand(-1, -1, dim), None, before if firsts[row] else torch.zeros_like(before))
        at += length
    errors = {form: (off(out, exact[..., :vdim].reshape(n, -1)),) + ((off(below, exact[..., vdim]),) if memory else ())
              for form, (out, below, _) in results.items()}
    print(errors, flush=True)
    for scan, chunked in zip(errors["scan"], errors["chunks"]):
        assert chunked <= (1.25 if spare else 2.0) * scan + HALF_UNIT


NO_NUMBERS = [float("inf"), float("-inf"), float("nan")]


@pytest.mark.parametrize("place", [70, 79, 100, 140])
@pytest.mark.parametrize("what", ["v", "k", "q", "decay"])
@pytest.mark.parametrize("bonus", [False, True])
def test_what_is_no_number_reaches_no_earlier_token_of_a_linear_recurrence(ops, place, what, bonus):
    """A token at the start, at the end and inside a block of 16, of the first chunk of its row and of the next (rows of 20, 130 and 10
    tokens: the second row's chunks begin at 20 and 84): the chunks leave the same numbers numbers as the walk, and those agree."""
    heads, dim, vdim, lengths = 2, 64, 80, [20, 130, 10]
    generator = torch.Generator("cuda").manual_seed(place)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    n = sum(lengths)
    q, k, v, decay = 0.5 * draw(n, heads * dim), 0.5 * draw(n, heads * dim), draw(n, heads * vdim), draw(n, heads * dim) - 1.0
    no_number = NO_NUMBERS[place % 3] if what != "decay" else float("nan")
    {"q": q, "k": k, "v": v, "decay": decay}[what][place, 5] = no_number
    _, _, row_start, row_len, row_ctx = batch(lengths, [3, 0, 0], "cuda")
    slots = torch.tensor([1, 2, 0], dtype=torch.int32, device="cuda")
    start = draw(3, heads * dim * vdim)
    chunks = n // 64 + len(lengths)
    scratch = {"sums": torch.empty(chunks, heads, dim, vdim, device="cuda"), "totals": torch.empty(chunks, heads, dim, device="cuda"),
               "queries": torch.empty(n, heads, dim, device="cuda")}
    results = []
    for more in ({}, scratch):
        state, out = start.clone(), torch.empty(n, heads * vdim, device="cuda")
        ops.linear_recurrence(q, k, v, decay, None, "double_exp", 1.0, draw(heads, dim) * 0 + 0.3 if bonus else None, 0.3, state, 0, slots, row_start,
                              row_len, row_ctx, out, heads, dim, vdim, **more)
        results.append((out, state))
    for walk, chunked in zip(*results):
        assert torch.equal(torch.isfinite(walk), torch.isfinite(chunked))
        keep = torch.isfinite(walk)
        assert float((walk - chunked)[keep].norm()) <= 1e-5 * float(walk[keep].norm())
    assert torch.isfinite(results[0][0][:place]).all() and not torch.isfinite(results[0][0][place:]).all()


@pytest.mark.parametrize("place", [70, 79, 100, 140])
@pytest.mark.parametrize("what", ["v", "k", "q", "decay", "strength"])
@pytest.mark.parametrize("first", [0, 2])
def test_what_is_no_number_reaches_no_earlier_token_of_a_delta_rule(ops, place, what, first):
    heads, dim, vdim, lengths = 2, 72, 48, [20, 130, 10]
    generator = torch.Generator("cuda").manual_seed(place)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    n, size = sum(lengths), heads * dim * vdim
    q, k = draw(n, heads, dim), draw(n, heads, dim)
    q, k = q / q.norm(dim=-1, keepdim=True), k / k.norm(dim=-1, keepdim=True)
    v, strength, decay = draw(n, heads * vdim), torch.sigmoid(draw(n, heads)), torch.exp(-0.2 * torch.rand(n, heads * dim, device="cuda", generator=generator))
    no_number = NO_NUMBERS[place % 3] if what not in ("decay", "strength") else float("nan")
    {"q": q.view(n, -1), "k": k.view(n, -1), "v": v, "decay": decay, "strength": strength}[what][place, 1 if what == "strength" else 5] = no_number
    prepared = torch.cat([q.reshape(n, -1), k.reshape(n, -1), v], dim=1)
    _, _, row_start, row_len, row_ctx = batch(lengths, [3, first, 0], "cuda")
    slots = torch.tensor([1, 2, 0], dtype=torch.int32, device="cuda")
    start = draw(3, size)
    scratch = torch.empty(ops.delta_rule_scratch(n, len(lengths), 10 ** 6, heads, dim, vdim), device="cuda")
    results = []
    for more in ({}, {"scratch": scratch}):
        state, out = start.clone(), torch.empty(n, heads * vdim, device="cuda")
        ops.delta_rule(prepared, strength, decay, True, state, 0, slots, row_start, row_len, row_ctx, out, heads, heads, dim, vdim, **more)
        results.append((out, state))
    for walk, chunked in zip(*results):
        assert torch.equal(torch.isfinite(walk), torch.isfinite(chunked))
        keep = torch.isfinite(walk)
        assert float((walk - chunked)[keep].norm()) <= 1e-5 * float(walk[keep].norm())
    assert torch.isfinite(results[0][0][:place]).all() and not torch.isfinite(results[0][0][place:]).all()


LONG = 2000


@pytest.mark.parametrize("kept", [0.9995, 0.99, 0.6])
@pytest.mark.parametrize("dtype", DTYPES)
def test_a_long_row_of_a_linear_recurrence(ops, dtype, kept):
    """32 chunks of one row from a kept state, decays around ``kept`` a token: the walk over the chunks rounds no more than the walk over the tokens."""
    heads, dim, vdim = 2, 128, 128
    generator = torch.Generator("cuda").manual_seed(int(1e4 * kept))
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    proj = (0.5 * draw(LONG, 2 * heads * dim + heads * vdim)).to(dtype)
    q, k, v = proj[:, :heads * dim], proj[:, heads * dim:2 * heads * dim], proj[:, 2 * heads * dim:]
    z = torch.log(-torch.log(torch.tensor(kept))).item() + 0.5 * draw(LONG, heads * dim)
    _, _, row_start, row_len, row_ctx = batch([LONG], [50], "cuda")
    slots, start = torch.zeros(1, dtype=torch.int32, device="cuda"), draw(1, heads * dim * vdim)
    chunks = ops.linear_recurrence_chunks(LONG, 1, LONG, 16, dim, vdim)
    scratch = {"sums": torch.empty(chunks, heads, dim, vdim, device="cuda"), "totals": torch.empty(chunks, heads, dim, device="cuda"),
               "queries": torch.empty(LONG, heads, dim, device="cuda")}
    wide = lambda x: x.double().reshape(LONG, heads, -1)
    exact, after = plain_recurrence(0.3 * wide(q), wide(k), wide(v), torch.exp(-torch.exp(wide(z))), None, start.view(heads, dim, vdim).double())
    errors = []
    for more in ({}, scratch):
        state, out = start.clone(), torch.empty(LONG, heads * vdim, device="cuda")
        ops.linear_recurrence(q, k, v, z, None, "double_exp", 1.0, None, 0.3, state, 0, slots, row_start, row_len, row_ctx, out, heads, dim, vdim, **more)
        errors.append((off(out, exact.reshape(LONG, -1)), off(state, after.reshape(1, -1))))
    print("long linear", dtype, kept, errors, flush=True)
    for walk, chunked in zip(*errors):
        assert chunked <= 1.1 * walk


@pytest.mark.parametrize("kept", [0.9995, 0.99, 0.6])
@pytest.mark.parametrize("per_channel", [False, True])
def test_a_long_row_of_a_delta_rule(ops, per_channel, kept):
    """The same with keys of which every second repeats one of eight directions, so that writes keep taking back what stands there."""
    heads, dim, vdim = 2, 128, 128
    generator = torch.Generator("cuda").manual_seed(int(1e4 * kept) + per_channel)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    q, k, v = draw(LONG, heads, dim), draw(LONG, heads, dim), draw(LONG, heads, vdim)
    k[::2] = draw(8, heads, dim).repeat(LONG // 16, 1, 1) + 0.05 * k[::2]
    q, k = q / q.norm(dim=-1, keepdim=True) * dim ** -0.5, k / k.norm(dim=-1, keepdim=True)
    strength = torch.sigmoid(2 * draw(LONG, heads))
    decay = torch.exp(torch.log(torch.tensor(kept)).item() * torch.exp(0.5 * draw(LONG, heads * dim if per_channel else heads)))
    prepared = torch.cat([x.reshape(LONG, -1) for x in (q, k, v)], dim=1)
    _, _, row_start, row_len, row_ctx = batch([LONG], [50], "cuda")
    slots, start = torch.zeros(1, dtype=torch.int32, device="cuda"), draw(1, heads * dim * vdim)
    turned = lambda flat: flat.view(heads, vdim // 16, dim, 16).permute(0, 2, 1, 3).reshape(heads, dim, vdim)
    scratch = torch.empty(LONG // 64 + 1, heads, ops._part_library("delta").lsa_delta_chunk_floats(dim, vdim), device="cuda")
    exact, after = plain_delta(q.double(), k.double(), v.double(), decay.double().view(LONG, heads, -1).expand(LONG, heads, dim), strength.double(),
                               turned(start).double())
    errors = []
    for more in ({}, {"scratch": scratch}):
        state, out = start.clone(), torch.empty(LONG, heads * vdim, device="cuda")
        ops.delta_rule(prepared, strength, decay, per_channel, state, 0, slots, row_start, row_len, row_ctx, out, heads, heads, dim, vdim, **more)
        errors.append((off(out, exact.reshape(LONG, -1)), off(turned(state), after)))
    print("long delta", per_channel, kept, errors, flush=True)
    for walk, chunked in zip(*errors):
        assert chunked <= 1.1 * walk


@pytest.mark.parametrize("rule", ["linear", "delta"])
def test_chunks_recorded_in_a_graph_for_rows_of_other_lengths(ops, rule):
    """256 tokens in three rows, recorded once and replayed with the rows cut elsewhere, one of them empty or new: the numbers of an eager call."""
    heads, dim, vdim, n = 2, 64, 48, 256
    generator = torch.Generator("cuda").manual_seed(9)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    slots, start = torch.tensor([2, 0, 1], dtype=torch.int32, device="cuda"), draw(3, heads * dim * vdim)
    out, state, items = torch.empty(n, heads * vdim, device="cuda"), start.clone(), n // 64 + 3
    rows = [torch.zeros(3, dtype=torch.int32, device="cuda") for _ in range(3)]

    def cut(lengths, firsts):
        for kept, value in zip(rows, batch(lengths, firsts, "cuda")[2:]):
            kept.copy_(value)
    if rule == "linear":
        q, k, v, decay = (0.5 * draw(n, heads * width) for width in (dim, dim, vdim, dim))
        scratch = {"sums": torch.empty(items, heads, dim, vdim, device="cuda"), "totals": torch.empty(items, heads, dim, device="cuda"),
                   "queries": torch.empty(n, heads, dim, device="cuda")}
        run = lambda: ops.linear_recurrence(q, k, v, decay, None, "double_exp", 1.0, None, 0.3, state, 0, slots, *rows, out, heads, dim, vdim, **scratch)
    else:
        q, k = (torch.nn.functional.normalize(draw(n, heads, dim), dim=-1).reshape(n, -1) for _ in range(2))
        prepared, strength = torch.cat([q, k, draw(n, heads * vdim)], dim=1), torch.sigmoid(draw(n, heads))
        decay = torch.exp(-0.1 * torch.rand(n, heads, device="cuda", generator=generator))
        scratch = torch.empty(items, heads, ops._part_library("delta").lsa_delta_chunk_floats(dim, vdim), device="cuda")
        run = lambda: ops.delta_rule(prepared, strength, decay, False, state, 0, slots, *rows, out, heads, heads, dim, vdim, scratch=scratch)
    cut([200, 55, 1], [4, 0, 9])
    run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for lengths, firsts in (([200, 55, 1], [4, 0, 9]), ([1, 1, 254], [7, 0, 0]), ([0, 128, 128], [3, 5, 0]), ([85, 85, 86], [0, 64, 2]), ([200, 55, 1], [4, 0, 9])):
        cut(lengths, firsts)
        results = []
        for call in (run, graph.replay):
            state.copy_(start)
            out.fill_(float("nan"))
            call()
            torch.cuda.synchronize()
            results.append((out.clone(), state.clone()))
        assert torch.isfinite(results[0][0]).all()
        for eager, replayed in zip(*results):
            assert torch.equal(eager, replayed)


@pytest.mark.parametrize("design,case", [("barotar", "BD"), ("gogalix", "GC")])
def test_captured_steps_with_portions_in_chunks_and_walked(design, case):
    """256 tokens of three requests in turns, one long portion beside two short ones (in chunks) and three alike (walked): a graph each, and every
    replay's logits are those of the same step run eagerly."""
    import importlib
    from helpers import random_tokens
    from llmserver_amd.engine import StepEntry
    from llmserver_amd.engine.replay import make_runner
    tiny = importlib.import_module(f"tiny_{design}")
    vocab, page = tiny.CASES[case][0]["vocab"], tiny.CASES[case][2]
    print(f"captured portions in chunks {design} {case}", flush=True)
    runners = [make_runner(tiny.model_folder(case), "float32", 4096, page, max_live=4) for _ in range(2)]
    runners[1].use_graphs = False
    forms, worst = {}, 0.0
    for turn in range(10):
        lengths = [250, 3, 3] if turn % 2 else [85, 85, 86]
        logits = []
        for runner in runners:
            entries = [StepEntry(f"{turn} {row}", random_tokens(vocab, length, 10 * turn + row), [length - 1]) for row, length in enumerate(lengths)]
            for entry in entries:
                runner.cache.open(entry.request_id)
            logits.append(runner.step(entries).clone())
            follow = [StepEntry(entry.request_id, [turn], [0]) for entry in entries]              # (the state behind them)
            logits.append(runner.step(follow).clone())
            if runner.use_graphs:
                key = runner._portion_key(entries)
                if key is not None:
                    forms.setdefault(turn % 2, set()).add(key)
            for entry in entries:
                runner.cache.close(entry.request_id)
        torch.cuda.synchronize()
        for replayed, eager in zip(logits[:2], logits[2:]):
            worst = max(worst, float((replayed - eager).norm() / eager.norm()))
    print("worst", worst, "replays", runners[0].graph_replays, flush=True)
    assert len(forms[0]) == len(forms[1]) == 1 and forms[0] != forms[1]
    assert any(next(iter(forms[1]))[5][1:]) and runners[0].graph_replays >= 6
    assert worst < 1e-5
