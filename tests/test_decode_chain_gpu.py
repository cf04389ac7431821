"""All layers of a decode step of one or two rows in one launch (csrc/decode_chain.hip): alone against the
same layers in float64, and through an engine against the plain implementation and each layer's own launches."""

import ctypes
import os

import pytest
import torch

import helpers
import plain_gpt2 as plain

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
_i, _vp = ctypes.c_int, ctypes.c_void_p


class Dims(ctypes.Structure):
    _fields_ = [(n, _i) for n in ("n_layers", "width", "inner", "n_heads", "n_kv_heads", "page_size")] + [
        ("page_stride", ctypes.c_size_t), ("eps1", ctypes.c_float), ("eps2", ctypes.c_float), ("scale", ctypes.c_float)]


class Layer(ctypes.Structure):
    _fields_ = [("W", _vp * 4), ("bias", _vp * 4), ("gamma", _vp * 2), ("beta", _vp * 2), ("k", _vp), ("v", _vp)]


def _lib():
    from mlx_lm_amd.ops import build

    lib = build.load("decode_chain")
    lib.decode_chain_bytes.restype = ctypes.c_size_t
    lib.mlxlm_last_error.restype = ctypes.c_char_p
    return lib


def _packed(w):
    """[N, K] in tiles of 16 features x 64 k, in the order the lanes read them; features beyond N are zeros."""
    n, k = w.shape
    t = torch.zeros((n + 15) // 16 * 16, k, dtype=w.dtype, device=w.device)
    t[:n] = w
    return t.view(-1, 16, k // 64, 4, 2, 8).permute(0, 2, 4, 3, 1, 5).contiguous()


# (layers, width, inner, heads, key heads, page size, keys before the step, blocks, patience):
# one k-block, an odd number of them, the widest and longest that a wave holds; no key yet, a tile of keys less one, whole and
# begun, the most keys; features a unit that do not divide the product's; query heads that share a key head; two rows
# of very different lengths; and few blocks of little patience, which do each other's units (below four, nobody's own are
# attention's)
CASES = [
    (2, 64, 64, 1, 1, 16, (0,), 0, 0),
    (3, 64, 192, 2, 1, 8, (7, 8), 0, 0),
    (2, 128, 256, 2, 2, 16, (9, 1024), 0, 0),
    (2, 832, 3328, 13, 13, 16, (300,), 0, 0),
    (2, 1600, 6400, 25, 25, 16, (700, 1001), 0, 0),
    (2, 1600, 6400, 25, 25, 32, (1023,), 0, 0),
    (1, 2048, 7168, 32, 8, 16, (64,), 0, 0),
    (2, 768, 3072, 12, 12, 16, (93,), 3, 100),
    (2, 192, 448, 3, 3, 16, (40, 3), 1, 10),
    (2, 1280, 5120, 20, 20, 16, (100, 500), 100, 100),
]
# ... and units dealt anew among the blocks that run, from the first wait on: all of them (there are more than a product's units,
# or fewer), and five, of which one began as attention's
CASES += [
    (3, 64, 192, 2, 1, 8, (7, 8), 0, 1),
    (2, 832, 3328, 13, 13, 16, (300,), 0, 1),
    (3, 1600, 6400, 25, 25, 16, (700, 1001), 0, 1),
    (1, 2048, 7168, 32, 8, 16, (64,), 0, 1),
    (3, 768, 3072, 12, 12, 16, (93, 20), 5, 1),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[1]}x{c[2]}-{'+'.join(map(str, c[6]))}{f'-{c[7]}blocks' if c[7] else ''}{'-anew' if c[8] == 1 else ''}")
def test_layers_of_a_decode_step_in_one_launch(case):
    n_layers, D, I, H, HK, page, keys, blocks, patience = case
    lib, R, Q, KV = _lib(), len(case[6]), case[3] * 64, case[4] * 64
    g = torch.Generator().manual_seed(D + I + R)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).cuda()

    width = max(keys) // page + 1
    pages = torch.randperm(R * width, generator=g).to(torch.int32).view(R, width).cuda()
    layers, held, table = [], [], (Layer * n_layers)()
    for t in table:
        shapes = ((Q + 2 * KV, D), (D, Q), (I, D), (D, I))
        W, b = [rand(*s, std=s[1] ** -0.5).to(BF) for s in shapes], [rand(s[0], std=0.1) for s in shapes]
        norms = [1 + rand(D, std=0.1), rand(D, std=0.1), 1 + rand(D, std=0.1), rand(D, std=0.1)]
        kv = [rand(R * width, HK, page, 64).to(BF) for _ in range(2)]
        packs = [_packed(w) for w in W]
        held.append((packs, b, norms, kv))
        layers.append((W, b, norms, [x.clone() for x in kv]))
        t.W[:], t.bias[:] = [p.data_ptr() for p in packs], [x.data_ptr() for x in b]
        t.gamma[:], t.beta[:] = [norms[0].data_ptr(), norms[2].data_ptr()], [norms[1].data_ptr(), norms[3].data_ptr()]
        t.k, t.v = kv[0].data_ptr(), kv[1].data_ptr()
    on_gpu = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8).cuda()
    d = Dims(n_layers, D, I, H, HK, page, HK * page * 64, 1e-5, 1e-5, 0.125)
    assert lib.decode_chain_takes(ctypes.byref(d), R) == 1
    memory = torch.zeros(lib.decode_chain_bytes(ctypes.byref(d), R), dtype=torch.uint8, device="cuda")
    req = torch.arange(R, dtype=torch.int32, device="cuda")
    pos = torch.tensor(keys, dtype=torch.int32, device="cuda")

    def launch(h):
        out = torch.full_like(h, float("nan"))
        stream = _vp(torch.cuda.current_stream().cuda_stream)
        p = [_vp(x.data_ptr()) for x in (on_gpu, memory, h, out, pages, req, pos)]
        rc = lib.decode_chain(ctypes.byref(d), R, p[0], p[1], p[2], p[3], D, p[4], width, p[5], p[6], blocks, ctypes.c_uint(patience), stream)
        assert rc == 0, lib.mlxlm_last_error().decode()
        return out

    def plain(h):
        """The layers in 64 bits, and each layer's new keys and values."""
        h, new = h.double(), []
        for W, b, (g1, b1, g2, b2), (k_pages, v_pages) in layers:
            def product(x, i):
                return x @ W[i].double().T + b[i].double()

            x = product(torch.nn.functional.layer_norm(h, (D,), g1.double(), b1.double(), 1e-5), 0)
            o = []
            for m, n in enumerate(keys):
                k, v = ([p[pages[m].long()].permute(1, 0, 2, 3).reshape(HK, -1, 64)[:, :n].double() for p in (k_pages, v_pages)])
                k = torch.cat([k, x[m, Q : Q + KV].view(HK, 1, 64)], 1).repeat_interleave(H // HK, 0)
                v = torch.cat([v, x[m, Q + KV :].view(HK, 1, 64)], 1).repeat_interleave(H // HK, 0)
                p = torch.softmax((k * x[m, :Q].view(H, 1, 64)).sum(-1) / 8, -1)
                o.append((p.unsqueeze(-1) * v).sum(1).reshape(-1))
            new.append(x[:, Q:])
            h = h + product(torch.stack(o), 1)
            h = h + product(torch.nn.functional.gelu(product(torch.nn.functional.layer_norm(h, (D,), g2.double(), b2.double(), 1e-5), 2), approximate="tanh"), 3)
        return h, new

    # Roundings to bfloat16 (2^-9 of a value) between a layer's products: the two norms' rows, q/k/v, the attention's rows,
    # the activations.  Five a layer, each of what is then added to the stream, doubled for the step from each to the
    # next through products whose rows are of one length: 5 x 2^-8 for all layers here, whose shares of the stream differ.
    tol = 5 * 2.0**-8
    runs = []
    for turn in range(3):  # again on the same memory, with other rows, and the first rows once more
        h = rand(R, D, std=2.0) if turn < 2 else first
        first = h if turn == 0 else first
        out = launch(h)
        torch.cuda.synchronize()
        want, new = plain(h)
        assert ((out.double() - want).norm(dim=1) / want.norm(dim=1)).max().item() < tol, turn
        for (_, _, _, kv), want_kv in zip(held, new):
            for m, n in enumerate(keys):
                at = pages[m, n // page].item()
                got = torch.cat([kv[0][at, :, n % page].reshape(-1), kv[1][at, :, n % page].reshape(-1)]).double()
                assert ((got - want_kv[m]).norm() / want_kv[m].norm()).item() < tol, (turn, m)
        runs.append(out)
    assert torch.equal(runs[0], runs[2])
    # no other key or value was touched
    for (_, _, _, kv), (_, _, _, before) in zip(held, layers):
        for a, b in zip(kv, before):
            for m, n in enumerate(keys):
                a[pages[m, n // page].item(), :, n % page] = b[pages[m, n // page].item(), :, n % page]
            assert torch.equal(a, b)


@pytest.mark.parametrize("change", [dict(width=96), dict(width=2112), dict(inner=7232), dict(n_kv_heads=3), dict(n_layers=0), dict(rows=3),
                                    dict(width=1664, inner=6656, n_heads=26, n_kv_heads=26, rows=2)],
                         ids=lambda c: next(iter(c)) + str(next(iter(c.values()))))
def test_sizes_the_one_launch_does_not_take(change):
    sizes = dict(n_layers=2, width=128, inner=256, n_heads=2, n_kv_heads=2, page_size=16, rows=1)
    sizes.update(change)
    rows = sizes.pop("rows")
    d = Dims(*sizes.values(), 2048, 1e-5, 1e-5, 0.125)
    assert _lib().decode_chain_takes(ctypes.byref(d), rows) == 0


def _one_layer(rows=1):
    """(dims, the layers' table on the device and all it points to, launch) of one layer of width 128 without keys in the cache."""
    lib, D, I, Q = _lib(), 128, 256, 128
    g = torch.Generator().manual_seed(rows)
    W = [_packed((torch.randn(*s, generator=g) * s[1] ** -0.5).to(BF).cuda()) for s in ((3 * Q, D), (D, Q), (I, D), (D, I))]
    ones, zeros = torch.ones(D, device="cuda"), torch.zeros(D, device="cuda")
    kv = [torch.zeros(rows, 2, 16, 64, dtype=BF, device="cuda") for _ in range(2)]
    table = (Layer * 1)()
    table[0].W[:], table[0].gamma[:], table[0].beta[:] = [w.data_ptr() for w in W], [ones.data_ptr()] * 2, [zeros.data_ptr()] * 2
    table[0].k, table[0].v = kv[0].data_ptr(), kv[1].data_ptr()
    on_gpu = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8).cuda()
    d = Dims(1, D, I, 2, 2, 16, 2 * 16 * 64, 1e-5, 1e-5, 0.125)
    memory = torch.zeros(lib.decode_chain_bytes(ctypes.byref(d), rows) // 8, dtype=torch.int64, device="cuda")
    index = torch.arange(rows, dtype=torch.int32, device="cuda")
    pos = torch.zeros(rows, dtype=torch.int32, device="cuda")
    h = torch.randn(rows, D, generator=g).cuda()
    held = (W, ones, zeros, kv, on_gpu, index, pos, h)

    def launch():
        out = torch.full_like(h, float("nan"))
        p = [_vp(x.data_ptr()) for x in (on_gpu, memory, h, out, index, index, pos)]
        rc = lib.decode_chain(ctypes.byref(d), rows, p[0], p[1], p[2], p[3], D, p[4], 1, p[5], p[6], 0, ctypes.c_uint(0),
                              _vp(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.mlxlm_last_error().decode()
        torch.cuda.synchronize()
        return out

    return memory, launch, held


def _places(rows, N, Q, D, I):
    """(first word, words) of q/k/v, attention's rows, the stream after attention, the activations, the stream."""
    at, out = 32, []
    for n in (N // 2, Q // 2, D, I // 2, D):
        out.append(slice(at, at + n * rows))
        at += (n * rows + 31) // 32 * 32
    return out


@pytest.mark.parametrize("rows", [1, 2])
def test_late_words_leave_a_later_product_s_alone(rows):
    """Where the places of a product hold words of a later one, as they do for a block that fell behind the others after it
    had read its rows, they stay: an older word put back would be waited past by nobody and waited for without end."""
    memory, launch, _held = _one_layer(rows)
    launch()
    qkv, att, h1, act, h2 = _places(rows, 3 * 128, 128, 128, 256)
    base = memory[0].item() & 0xFFFFFFFF
    assert base == 6 and (memory[h1] >> 32 == base + 2).all() and (memory[act] >> 32 == base + 3).all()
    later = (base + 1000 << 32) + 12345  # (its readers see that their unit is long done: the launch ends)
    memory[h1], memory[act] = later, later
    out = launch()
    assert (memory[qkv] >> 32 == base + 6).all() and (memory[att] >> 32 == base + 7).all()  # computed, and stored over older ones
    assert (memory[h1] == later).all() and (memory[act] == later).all() and out.isnan().all()


def test_tags_where_their_bits_end():
    """The counter of tags goes past its last step: the words start from zeros again and every step's output is the same."""
    memory, launch, _held = _one_layer()
    want = launch()
    memory[0] = 0xFFFFFFFF - 2 * 0x10000 - 13
    bases = []
    for _ in range(6):
        assert torch.equal(launch(), want)
        bases.append(memory[0].item() & 0xFFFFFFFF)
    turn = next(i for i, b in enumerate(bases) if b == 6)
    assert bases == [0xFFFFFFFF - 2 * 0x10000 - 13 + 6 * (i + 1) for i in range(turn)] + [6 * (i + 1) for i in range(6 - turn)] and 0 < turn < 5


@pytest.mark.parametrize("width,rows", [(1664, 1), (2048, 1), (1600, 2), (64, 2)])
def test_widest_sizes_the_one_launch_takes(width, rows):
    """Two rows only where every block has one unit of a product: two units a block are slower than each layer's launches."""
    d = Dims(2, width, min(4 * width, 6656), width // 64, width // 64, 16, width * 16, 1e-5, 1e-5, 0.125)
    assert _lib().decode_chain_takes(ctypes.byref(d), rows) == 1


# keys before the step and key heads: every tile of 8 keys, a wave's tiles and rows of other lengths beside them
@pytest.mark.parametrize("H,HK,page,keys", [(1, 1, 16, (1, 7)), (2, 2, 8, (8, 9)), (4, 2, 16, (95, 96)), (4, 4, 16, (97, 513)), (8, 8, 32, (1023, 40)),
                                            (6, 3, 16, (1024, 1000)), (8, 8, 16, (777,))])
def test_every_key_of_a_row_counts(H, HK, page, keys):
    """One layer whose stream is attention's output alone, over scores so even that every key has its share: what the
    launch gives is nearer to the layer in float64 than any one key left out of it, the step's own among them, would be."""
    lib, R, D, I, Q, KV = _lib(), len(keys), 64 * H, 64, 64 * H, 64 * HK
    g = torch.Generator().manual_seed(sum(keys) + H)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).cuda()

    W = [rand(Q + 2 * KV, D, std=D**-0.5), rand(D, Q, std=Q**-0.5), rand(I, D, std=D**-0.5), torch.zeros(D, I, device="cuda")]
    W[0][:Q] *= 0.25  # (scores of a spread of 0.25)
    W = [w.to(BF) for w in W]
    ones, zeros = torch.ones(D, device="cuda"), torch.zeros(D, device="cuda")
    width = max(keys) // page + 1
    pages = torch.randperm(R * width, generator=g).to(torch.int32).view(R, width).cuda()
    kv = [rand(R * width, HK, page, 64).to(BF) for _ in range(2)]
    packs = [_packed(w) for w in W]
    table = (Layer * 1)()
    table[0].W[:], table[0].gamma[:], table[0].beta[:] = [p.data_ptr() for p in packs], [ones.data_ptr()] * 2, [zeros.data_ptr()] * 2
    table[0].k, table[0].v = kv[0].data_ptr(), kv[1].data_ptr()
    on_gpu = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8).cuda()
    d = Dims(1, D, I, H, HK, page, HK * page * 64, 1e-5, 1e-5, 0.125)
    memory = torch.zeros(lib.decode_chain_bytes(ctypes.byref(d), R), dtype=torch.uint8, device="cuda")
    req, pos = torch.arange(R, dtype=torch.int32, device="cuda"), torch.tensor(keys, dtype=torch.int32, device="cuda")
    h = rand(R, D, std=1e-3)
    h = h / h.std(1, keepdim=True) * 1e-2  # (small beside attention's output; its norm is not)
    x = torch.nn.functional.layer_norm(h.double(), (D,), eps=1e-5) @ W[0].double().T
    # before the launch adds its own: each row's keys and values in 64 bits, the step's own last
    held = [[p[pages[m].long()].permute(1, 0, 2, 3).reshape(HK, -1, 64)[:, :n].double() for p in kv] for m, n in enumerate(keys)]
    out = torch.empty_like(h)
    p = [_vp(t.data_ptr()) for t in (on_gpu, memory, h, out, pages, req, pos)]
    rc = lib.decode_chain(ctypes.byref(d), R, p[0], p[1], p[2], p[3], D, p[4], width, p[5], p[6], 0, ctypes.c_uint(0),
                          _vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.mlxlm_last_error().decode()
    torch.cuda.synchronize()
    # Roundings to bfloat16 on the way: the normed row's, q/k/v's, attention's row's, 2^-9 of a value at most each.
    tol = 3 * 2.0**-9
    for m in range(R):
        k, v = (torch.cat([old, x[m, at : at + KV].view(HK, 1, 64)], 1).repeat_interleave(H // HK, 0) for old, at in zip(held[m], (Q, Q + KV)))
        w = torch.softmax((k * x[m, :Q].view(H, 1, 64)).sum(-1) / 8, -1)
        o = (w.unsqueeze(-1) * v).sum(1)  # [heads, 64]
        without = (o.unsqueeze(1) - w.unsqueeze(-1) * v) / (1 - w).clamp(min=1e-9).unsqueeze(-1)  # [heads, the key left out, 64]
        a = o.reshape(-1) @ W[1].double().T
        off = (without - o.unsqueeze(1)).permute(1, 0, 2).reshape(len(k[0]), -1) @ W[1].double().T
        assert (off.norm(dim=1).min() / a.norm()).item() > 2 * tol  # (the mistake that would be hardest to see)
        assert ((out[m].double() - h[m].double() - a).norm() / a.norm()).item() < tol, m


@pytest.fixture(scope="module")
def gpt2_of_heads_of_64(tmp_path_factory):
    """(folder, config, weights) of a model whose decode steps one launch takes, with more positions than it takes keys."""
    from safetensors.torch import load_file, save_file

    from mlx_lm_amd.weights import write_model_folder

    config = dict(model_type="gpt2", n_layer=3, n_embd=128, n_head=2, n_inner=448, vocab_size=320, n_positions=1100, n_ctx=1100,
                  layer_norm_epsilon=1e-5, activation_function="gelu_new")
    folder = str(tmp_path_factory.mktemp("heads64"))
    write_model_folder(folder, dict(config), 21, "b", dtype="float32")
    f = os.path.join(folder, "model.safetensors")
    tensors = helpers.sharpen({k: v.clone() for k, v in load_file(f).items()}, config, 3.0)
    save_file(tensors, f)
    return folder, config, plain.from_checkpoint_layout({k: v.float() for k, v in tensors.items()}, config["n_layer"])


def _engine_of(folder, use_graphs, chained=True, model=None):
    from mlx_lm_amd.engine import Engine
    from mlx_lm_amd.utils import load_model

    eng = Engine(model or load_model(folder, dtype="bfloat16")[0], dtype="bfloat16", page_size=16, n_pages=160, max_requests=4, use_graphs=use_graphs)
    if not chained:
        eng._chain = False
    return eng


def _decode(eng, tokens, prompts, turns):
    """Requests read up to ``prompts`` tokens each, then turns of one token for each of the first ``n`` requests; logits of every turn's
    rows, and whether its layers were one launch (a replay: as when it was recorded)."""
    from mlx_lm_amd.engine import StepEntry

    at = dict(prompts)
    for r, n in prompts.items():
        eng.add_request(r)
        eng.step([StepEntry(r, tokens[r][:n])])
    got, chained, by_graph = {r: [] for r in prompts}, [], {}
    for n in turns:
        live = list(prompts)[:n]
        before, known = eng.stats.chained, set(eng._graphs)
        key = (n, eng._length_class(max(at[r] for r in live) + 1)[0]) if eng.use_graphs else None
        logits = eng.step([StepEntry(r, [tokens[r][at[r]]], [0]) for r in live])
        if key is not None and key in known:
            assert eng.stats.chained == before  # (a replay walks no parts)
            chained.append(by_graph[key])
        else:
            chained.append(eng.stats.chained > before)
            by_graph[key] = chained[-1]
        for i, r in enumerate(live):
            got[r].append(logits[i : i + 1].clone())
            at[r] += 1
    return {r: torch.cat(x) if x else None for r, x in got.items()}, chained, at


@pytest.mark.parametrize("use_graphs", [False, True])
def test_engine_steps_of_one_two_and_three_rows(gpt2_of_heads_of_64, use_graphs):
    """One and two rows by the one launch, three by each layer's, by turns and with growing contexts, replayed many times over: logits of
    the plain implementation, and of the same steps by each layer's launches."""
    folder, config, weights = gpt2_of_heads_of_64
    tokens = {r: helpers.random_tokens(n + 60, config["vocab_size"], seed=n) for r, n in (("a", 203), ("b", 30), ("c", 90))}
    prompts = {"a": 203, "b": 30, "c": 90}
    turns = [1, 2, 3, 2, 1, 1, 2, 2, 3, 1] * 4
    got, chained, at = _decode(_engine_of(folder, use_graphs), tokens, prompts, turns)
    assert chained == [n < 3 for n in turns]
    own, none, _ = _decode(_engine_of(folder, use_graphs, chained=False), tokens, prompts, turns)
    assert not any(none)
    w = helpers.round_matrices_to_bf16(weights)
    for r in prompts:
        want = plain.forward(w, config, tokens[r][: at[r]])[prompts[r] :]
        for x in (got[r], own[r]):  # (of the largest logit, as in test_engine_gpu.py; each has its own roundings)
            assert (x.double().cpu() - want).abs().max() <= 2.5e-2 * want.abs().max(), r
    if use_graphs:  # a replay has no rounding of its own
        eager, _, _ = _decode(_engine_of(folder, False), tokens, prompts, turns)
        for r in prompts:
            assert torch.equal(eager[r], got[r]), r


@pytest.mark.parametrize("use_graphs", [False, True])
@pytest.mark.parametrize("rows", [1, 2])
def test_engine_steps_across_the_most_keys(gpt2_of_heads_of_64, rows, use_graphs):
    """A row that grows past the keys that the one launch takes: the step that would need one more goes by each layer's launches (a recorded
    one with its class of length), and the logits do not notice."""
    folder, config, weights = gpt2_of_heads_of_64
    tokens = {"long": helpers.random_tokens(1050, config["vocab_size"], seed=5), "short": helpers.random_tokens(80, config["vocab_size"], seed=6)}
    prompts = dict(list({"long": 1010, "short": 40}.items())[:rows])
    eng = _engine_of(folder, use_graphs)
    got, chained, at = _decode(eng, tokens, prompts, [rows] * 40)
    # 1,010 keys before the first step; 1,024 before the last that is chained, or where a recorded step's class of length ends ahead of that
    assert True in chained and False in chained
    assert chained == [(eng._length_class(1011 + i)[1] if use_graphs else 1011 + i) - 1 <= 1024 for i in range(40)]
    w = helpers.round_matrices_to_bf16(weights)
    for r in prompts:
        want = plain.forward(w, config, tokens[r][: at[r]])[prompts[r] :]
        assert (got[r].double().cpu() - want).abs().max() <= 2.5e-2 * want.abs().max(), r


@pytest.mark.parametrize("use_graphs", [False, True])
def test_two_engines_of_one_model_on_two_streams(gpt2_of_heads_of_64, use_graphs):
    """Each engine has its own words and tags: steps of both side by side give what each gives alone."""
    from mlx_lm_amd.engine import StepEntry
    from mlx_lm_amd.utils import load_model

    folder, config, _ = gpt2_of_heads_of_64
    tokens = {"a": helpers.random_tokens(120, config["vocab_size"], seed=1), "b": helpers.random_tokens(120, config["vocab_size"], seed=2)}
    alone = {r: _decode(_engine_of(folder, use_graphs), tokens, {r: 60}, [1] * 50)[0][r] for r in tokens}
    model, _ = load_model(folder, dtype="bfloat16")
    engines = {r: _engine_of(folder, use_graphs, model=model) for r in tokens}
    streams = {r: torch.cuda.Stream() for r in tokens}
    rows = {r: [] for r in tokens}
    for r, eng in engines.items():
        with torch.cuda.stream(streams[r]):
            eng.add_request(r)
            eng.step([StepEntry(r, tokens[r][:60])])
    for i in range(60, 110):
        for r, eng in engines.items():
            with torch.cuda.stream(streams[r]):
                rows[r].append(eng.step([StepEntry(r, [tokens[r][i]], [0])]).clone())
    torch.cuda.synchronize()
    for r in tokens:
        assert torch.equal(torch.cat(rows[r]), alone[r]) and engines[r].stats.chained > 0
