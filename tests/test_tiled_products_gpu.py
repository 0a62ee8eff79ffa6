"""Products of many rows on this package's own tiles (``csrc/product.hip``) at the edges of the tiles, against 64 bits, and who gets them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
FORMS = ("plain", "gated", "activated", "sums")


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


def drawn(rows, columns, inner, seed):
    generator = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn(rows, inner, device="cuda", generator=generator).to(torch.bfloat16)
    return x, (torch.randn(columns, inner, device="cuda", generator=generator) * inner ** -0.5).to(torch.bfloat16)


def silu(z):
    return z * torch.sigmoid(z)


def gelu(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


# Rows and columns around the edges of tiles of 64, 128 and 256, from one slab of the inner dimension to more than there are buffers for.
@pytest.mark.parametrize("rows,columns,inner", [(1, 8, 64), (63, 72, 128), (64, 64, 192), (65, 136, 256), (127, 128, 320), (129, 264, 384), (191, 40, 448), (255, 256, 512),
                                                (257, 520, 576), (300, 200, 1024)])
@pytest.mark.parametrize("tile", [1, 2, 3, 4])
@pytest.mark.parametrize("form", FORMS)
def test_every_tile_at_its_edges(ops, form, tile, rows, columns, inner):
    """A sum in 32 bits is off by at most (inner + 1) 2^-24 of the sum of its products' sizes, the activations' slopes are below 1.13 (the square's: twice the sum),
    and the one rounding (bfloat16 has eight bits) takes up to 2^-8 of the result."""
    if tile == 4 and form != "gated":
        pytest.skip("tiles of 256 have the gated form only")
    print(f"tiled product {form} {tile} {rows} {columns} {inner}", flush=True)
    x, weight = drawn(rows, 2 * columns if form == "gated" else columns, inner, rows + inner)
    exact, sizes = x.double() @ weight.double().T, x.double().abs() @ weight.double().abs().T
    off = (inner + 1) * 2.0 ** -24 * sizes
    lib = ops._product
    for activation in range({"gated": 2, "activated": 3}.get(form, 1)):
        for parts in (1, 2, 4, 8) if form == "sums" else (1,):
            if parts > inner // 64:
                continue
            margin = 256 * columns                                               # a tile's rows on both sides, in one tensor with the result: nothing writes there
            whole = torch.full((2 * margin + parts * rows * columns,), 7.0, device="cuda", dtype=torch.float32 if form == "sums" else torch.bfloat16)
            out = whole[margin:-margin].view(parts, rows, columns).fill_(float("nan"))
            assert lib.lsa_product(16 * parts + tile, FORMS.index(form), activation, x.data_ptr(), weight.data_ptr(), out.data_ptr(), rows, columns, inner,
                                   torch.cuda.current_stream().cuda_stream) == 0
            got = out.double().sum(0)
            act = (silu, gelu, lambda z: z.clamp(min=0) ** 2)[activation]
            if form == "gated":
                gate, up = exact.split(columns, 1)
                want = act(gate) * up
                bound = 1.13 * off[:, :columns] * up.abs() + act(gate).abs() * off[:, columns:] + 2.0 ** -8 * want.abs() * (1 + 2.0 ** -8)
            elif form == "activated":
                want = act(exact)
                bound = off * (1.13 if activation < 2 else 2 * exact.abs() + off) + 2.0 ** -8 * want.abs()
            else:
                want, bound = exact, off + (2.0 ** -8 * exact.abs() if form == "plain" else 0.0)
            bound = bound * 1.01 + 2.0 ** -18 * want.abs().max()                 # (expf and tanhf: a few parts in 2^23)
            assert torch.isfinite(got).all() and bool(((got - want).abs() <= bound).all()), float(((got - want).abs() - bound).max())
            assert bool((whole[:margin] == 7.0).all()) and bool((whole[-margin:] == 7.0).all())


# On both sides of the line between tiles of 64 x 32 (up to 256 of them, parts of the sums included: 4,096 columns of gated products, 8,192 of the others for one block of rows) and of 64 x 64, from
# one slab to more than either has buffers for.
@pytest.mark.parametrize("rows,columns,inner", [(1, 8200, 64), (33, 4096, 640), (33, 4104, 704), (64, 8192, 704), (64, 8200, 576), (65, 2056, 768), (127, 4160, 384), (250, 1032, 832), (250, 2112, 320)])
@pytest.mark.parametrize("form", FORMS)
def test_small_tiles_on_both_sides_of_their_line(ops, form, rows, columns, inner):
    test_every_tile_at_its_edges(ops, form, 1, rows, columns, inner)


@pytest.mark.parametrize("form,columns", [("plain", 8192), ("gated", 4096), ("activated", 8192), ("sums", 4096)])
def test_both_small_tiles_give_the_same_bits(ops, form, columns):
    """Sixty-four rows, the most columns that tiles of 64 x 32 take (sums: in two parts) and eight more, which tiles of 64 x 64 take: the columns of both are the same numbers."""
    rows, inner, parts = 64, 704, 2 if form == "sums" else 1
    x, weight = drawn(rows, (columns + 8) * (2 if form == "gated" else 1), inner, 11)
    fewer = torch.cat([weight[:columns], weight[columns + 8:2 * columns + 8]]) if form == "gated" else weight[:columns].contiguous()
    results = []
    for count, w in ((columns + 8, weight), (columns, fewer)):
        print(f"small tiles {form} {count}", flush=True)
        out = torch.full((parts, rows, count), float("nan"), device="cuda", dtype=torch.float32 if form == "sums" else torch.bfloat16)
        assert ops._product.lsa_product(16 * parts + 1, FORMS.index(form), 0, x.data_ptr(), w.data_ptr(), out.data_ptr(), rows, count, inner, torch.cuda.current_stream().cuda_stream) == 0
        results.append(out[:, :, :columns])
    assert not bool(results[0].isnan().any()) and torch.equal(*results)


def test_what_does_not_fit_is_refused(ops):
    x, weight = drawn(64, 64, 128, 1)
    out = torch.empty(64, 64, device="cuda", dtype=torch.bfloat16)
    call = lambda plan, form, activation, xp, rows, columns, inner: ops._product.lsa_product(plan, form, activation, xp, weight.data_ptr(), out.data_ptr(), rows, columns, inner,
                                                                                            torch.cuda.current_stream().cuda_stream)
    for plan, form, activation, shift, rows, columns, inner in ((16, 0, 0, 0, 64, 64, 128), (21, 0, 0, 0, 64, 64, 128), (20, 0, 0, 0, 64, 64, 128), (33, 0, 0, 0, 64, 64, 128), (17, 4, 0, 0, 64, 64, 128),
                                                                (17, 0, 3, 0, 64, 64, 128), (17, 1, 2, 0, 64, 32, 128), (17, 0, 0, 2, 63, 64, 128), (17, 0, 0, 0, 64, 60, 128),
                                                                (17, 0, 0, 0, 64, 64, 96), (16 * 9 + 1, 3, 0, 0, 64, 64, 128), (16 * 4 + 1, 3, 0, 0, 64, 64, 128)):
        assert call(plan, form, activation, x.data_ptr() + shift, rows, columns, inner) == -1, (plan, form, activation, shift, rows, columns, inner)
    assert call(17, 0, 0, x.data_ptr(), 0, 64, 128) == 0


@pytest.mark.parametrize("rows", [130, 190, 333])
def test_products_of_a_portion_go_to_the_tiles(ops, rows, monkeypatch):
    """A layer's products at a few hundred rows, through the entry points that the parts call, against 64 bits; and what an entry point gives does not depend on
    where the tensors lie, for other orders and places are the library's."""
    taken = []
    real = ops._tiled_product
    monkeypatch.setattr(ops, "_tiled_product", lambda *a, **k: (lambda done: (taken.append(done is not None), done)[1])(real(*a, **k)))
    x, weight = drawn(rows, 4096, 2048, rows)
    want = x.double() @ weight.double().T

    def tiled():
        got = any(taken)
        taken.clear()
        return got

    def close(got):
        return float((got.double() - want).norm() / want.norm()) < 2.0 ** -8

    assert close(ops.linear(x, weight)) and tiled()
    out = torch.empty(rows, 4096, device="cuda", dtype=torch.bfloat16)
    assert ops.linear(x, weight, out=out) is out and close(out) and tiled()
    exact32 = ops.linear(x, weight, out_float32=True)
    assert exact32.dtype == torch.float32 and float((exact32.double() - want).norm() / want.norm()) < 2.0 ** -18 and tiled()
    moved = torch.empty(rows * 2048 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(rows, 2048).copy_(x)          # (at an odd place)
    wider = torch.zeros(rows, 2056, device="cuda", dtype=torch.bfloat16)
    wider[:, :2048] = x
    for other in (moved, wider[:, :2048], x.t().contiguous().t()):
        assert close(ops.linear(other, weight)) and not tiled()
    column_out = torch.empty(4096, rows, device="cuda", dtype=torch.bfloat16).t()
    assert close(ops.linear(x, weight, out=column_out)) and not tiled()
    followed = x.clone().requires_grad_()
    with torch.enable_grad():
        y = ops.linear(followed, weight)
    assert y.requires_grad and close(y.detach()) and not tiled()
    hidden = ops.linear_gated(x, weight)
    assert hidden is not None and tiled()
    gate, up = want.split(2048, 1)
    assert float((hidden.double() - silu(gate) * up).norm() / (silu(gate) * up).norm()) < 2.0 ** -8


def test_partial_sums_join_the_stream_as_the_product_would(ops):
    """The sums of the parts are rounded to the stream's type as the whole product would be, then added: within one rounding of that."""
    x, weight = drawn(190, 2048, 6144, 5)
    sums = ops.linear_partial_sums(x, weight)
    assert sums is not None and sums.dim() == 3 and sums.shape[0] > 1
    want = x.double() @ weight.double().T
    assert float((sums.double().sum(0) - want).norm() / want.norm()) < 2.0 ** -18
    stream, normed, ones = torch.zeros(190, 2048, device="cuda", dtype=torch.bfloat16), torch.empty(190, 2048, device="cuda", dtype=torch.bfloat16), torch.ones(2048, device="cuda")
    ops.add_rmsnorm(stream, sums, ones, 1e-6, normed)
    assert float((stream.double() - want).norm() / want.norm()) < 2.0 ** -8


@pytest.mark.parametrize("rows", [29, 33, 64, 65, 100, 128])
def test_parts_that_another_launch_adds_up(ops, rows):
    """Plain and gated products of up to 128 rows: the parts' sums are of 32 bits, so that the one rounding is the result's."""
    x, weight = drawn(rows, 4096, 4096, rows)
    plain, gated = (ops._product.lsa_product_plan(form, rows, columns, 4096) for form, columns in ((0, 4096), (1, 2048)))
    print(f"parts added {rows}: plans {plain:#x} {gated:#x}", flush=True)
    assert gated & ops.PRODUCT_ADDED and (plain & ops.PRODUCT_ADDED or rows > 64)
    exact, sizes = x.double() @ weight.double().T, x.double().abs() @ weight.double().abs().T
    off = 4100 * 2.0 ** -24 * sizes
    assert bool(((ops.linear(x, weight).double() - exact).abs() <= (off + 2.0 ** -8 * exact.abs()) * 1.01).all())
    for activation, act in (("silu", silu), ("gelu_tanh", gelu)):
        got = ops.linear_gated(x, weight, activation=activation).double()
        gate, up = exact.split(2048, 1)
        want = act(gate) * up
        bound = 1.13 * off[:, :2048] * up.abs() + act(gate).abs() * off[:, 2048:] + 2.0 ** -8 * want.abs()
        assert bool(((got - want).abs() <= bound * 1.01 + 2.0 ** -18 * want.abs().max()).all())
    sums = ops.linear_partial_sums(x, weight)
    assert sums is not None and bool(((sums.double().sum(0) - exact).abs() <= off * 1.01).all())


def test_a_captured_step_replays_the_tiles(ops):
    x, weight = drawn(190, 4096, 2048, 9)
    ops.linear(x, weight), ops.linear_gated(x, weight)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y, hidden = ops.linear(x, weight), ops.linear_gated(x, weight)
    for seed in (10, 11, 12):
        x.copy_(drawn(190, 8, 2048, seed)[0])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ops.linear(x, weight)) and torch.equal(hidden, ops.linear_gated(x, weight))


@pytest.mark.parametrize("rows", [17, 28, 29])
@pytest.mark.parametrize("columns", [2112, 8448])
def test_activated_products_of_few_rows_are_asked_for_by_the_weights_size(ops, rows, columns, monkeypatch):
    """Up to 28 rows a weight that partial sums take goes there; one that they refuse goes to the tiles, where the activation is formed on the 32-bit sums and the result rounded
    once.  Of a product that stays the library's the plan is asked once."""
    print(f"activated products of few rows {rows} {columns}", flush=True)
    asked = []
    real = ops._tiled_product
    monkeypatch.setattr(ops, "_tiled_product", lambda *a, **k: (lambda done: (asked.append((a[0], done is not None)), done)[1])(real(*a, **k)))
    x, weight = drawn(rows, columns, 2048, rows)
    got = ops.linear_activated(x, weight, "relu2").double()
    assert (("activated", True) in asked) == (rows > 28 or columns == 8448)
    exact, off = x.double() @ weight.double().T, 2049 * 2.0 ** -24 * (x.double().abs() @ weight.double().abs().T)
    want = exact.clamp(min=0) ** 2
    roundings = 1 if rows > 28 or columns == 8448 else 3         # (of the result; behind a rounded product twice that rounding more, for the square)
    assert bool(((got - want).abs() <= off * (2 * exact.abs() + off) + roundings * 2.0 ** -8 * want * 1.01).all())
    asked.clear()
    x, weight = drawn(333, 12288, 2048, rows)
    assert ops.linear_gated(x, weight) is None and asked == [("gated", False)]


@pytest.mark.parametrize("rows", [40, 190])
def test_the_table_of_choices_goes_before_the_plan(ops, rows, monkeypatch):
    """A size that the table gives to the library goes there whatever the plan says of it, an unknown one as the plan says; and what is timed when somebody measures is the way that runs."""
    from llmserver_amd.kernels.choices import ChoiceTable, choice_key
    print(f"table before plan {rows}", flush=True)
    bucket = -(-rows // 8) * 8
    gated, wide = drawn(rows, 12288, 2048, rows)
    down_x, down = drawn(rows, 2048, 6144, rows)
    stream = ops._tiled_product("sums", down_x, down)
    assert ops._tiled_product("gated", gated, wide) is not None and stream is not None
    gated_key, partial_key = choice_key("gated", bucket, 12288, 2048, False, False), choice_key("partial", bucket, 2048, 6144, False, False)
    monkeypatch.setattr(ops, "choices", ChoiceTable(ops.choices.device_name))
    monkeypatch.setattr(ops, "consult_choices", True)
    for library in (False, None, True):
        ops.choices.entries.update({gated_key: library, partial_key: library}) if library is not None else ops.choices.entries.clear()
        for activation in ops.ACTIVATIONS:
            assert (ops.linear_gated(gated, wide, activation=activation) is None) == bool(library)
        sums = ops.linear_partial_sums(down_x, down)
        assert sums is None if library else torch.equal(sums, stream)
    if rows > ops.SPLIT_ROWS:                                     # ... and in ranges there, if the table says so
        ops.choices.entries.update({choice_key(f"parts{parts}", ops._parts_bucket(rows), 2048, 6144, False, False): parts == 4 for parts in (2, 4)})
        assert ops.linear_partial_sums(down_x, down).shape[0] == 4
    ops.choices.entries.clear()
    taken, real = [], ops._tiled_product
    monkeypatch.setattr(ops, "_tiled_product", lambda *a, **k: (lambda done: (taken.append(a[0]) if done is not None else None, done)[1])(real(*a, **k)))
    timed = []
    monkeypatch.setattr(ops, "_second_is_faster", lambda first, second: (taken.clear(), first(), timed.append(list(taken)), second(), True)[-1])
    with ops.measuring():
        assert ops.linear_gated(gated, wide) is None and ops.linear_partial_sums(down_x, down) is None or rows > ops.SPLIT_ROWS
    assert timed == [["gated"], ["sums"]] and ops.choices.entries[gated_key] and ops.choices.entries[partial_key]
