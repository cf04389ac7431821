"""All layers of a decode step of one or two rows in one launch (csrc/decode_chain.hip) against the
same layers in float64."""

import ctypes

import pytest
import torch

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
        assert ((out.double() - want).norm() / want.norm()).item() < tol, turn
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
