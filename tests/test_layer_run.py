"""Runs of whole layers of decode steps in one kernel (`ops.layer_run`): against the same layers in 64 bits, and against the engine's own
kernels for the same step; which steps take it."""
import math

import pytest
import torch

from inferrs_amd import ops

HD, PAGE = 128, 16


def test_rule_of_the_sizes():
    """Rows that fit, and where the rule between the two ways lies (the measured points on both sides of it)."""
    assert ops.layer_run_fits(8, 1024, 3072, 16, 8, 16) and ops.layer_run_fits(1, 5120, 25600, 64, 8, 16)
    assert not ops.layer_run_fits(9, 1024, 3072, 16, 8, 16) and not ops.layer_run_fits(1, 1024, 3072, 16, 8, 32)
    assert not ops.layer_run_fits(1, 1088, 3072, 16, 8, 16) and not ops.layer_run_fits(1, 1024, 3000, 16, 8, 16)
    assert not ops.layer_run_fits(1, 1024, 3072, 18, 2, 16) and not ops.layer_run_fits(1, 1024, 3072, 16, 1, 16)
    assert not ops.layer_run_fits(4, 5120, 25600, 64, 8, 16)                 # (four rows of 25,600 are more than a compute unit's shared memory)
    small, mid, large = (1024, 3072, 16, 8), (4096, 12288, 32, 8), (5120, 25600, 64, 8)
    assert ops.layer_run_pays(8, *small, 4096) and not ops.layer_run_pays(8, *small, 8192) and ops.layer_run_pays(1, *small, 40960)
    # (four rows of the second shape were measured at 0.97 to 0.99 of the speed of five kernels a layer in runs of 10 to 16 layers, three at 1.06 to 1.16)
    assert ops.layer_run_pays(3, *mid, 4096) and not any(ops.layer_run_pays(4, *mid, keys) for keys in (1024, 4096, 8192)) and not ops.layer_run_pays(6, *mid, 1024)
    assert ops.layer_run_pays(2, *large, 8192) and not ops.layer_run_pays(3, *large, 1024)
    # weights of up to 256 MiB: by the key heads, the layers of the run, and what a wave takes of the width
    heads32, width3072, width2560 = (2048, 8192, 32, 32), (3072, 8192, 24, 8), (2560, 9728, 32, 8)
    assert ops.layer_run_pays(5, *heads32, 2048) and not ops.layer_run_pays(6, *heads32, 1024)
    assert ops.layer_run_pays(3, *width3072, 4096) and not ops.layer_run_pays(4, *width3072, 1024)
    assert ops.layer_run_pays(8, *width2560, 4096) and not ops.layer_run_pays(8, *width2560, 1024, 4) and ops.layer_run_pays(6, *width2560, 1024, 4)
    assert ops.layer_run_pays(4, *width2560, 1024, 1) and not ops.layer_run_pays(6, *width2560, 1024, 1)
    # the bytes of the keys
    assert ops.layer_run_pays(1, *heads32, 45056) and ops.layer_run_pays(2, *heads32, 8192) and not ops.layer_run_pays(2, *heads32, 11264)
    heads16 = (1024, 3072, 16, 16)
    assert ops.layer_run_pays(4, *heads16, 8192) and not ops.layer_run_pays(5, *heads16, 8192) and not ops.layer_run_pays(2, *heads16, 16384)
    for keys in (1, 511, 512, 513, 16384, 16385, 40960, 131072):
        splits, chunk = ops.run_shares(keys)
        assert chunk % 32 == 0 and splits * chunk >= keys and splits <= 32 and (splits - 1) * chunk < keys


def _run_status(**change):
    """`ia_layer_run` over addresses that nobody reads unless the checks on the host let them through: (status, message)."""
    import ctypes
    lib = ops.library()
    at, by = change.pop("off", (0, 0))
    a = dict(dict(rows=1, width=512, ff=512, nq=4, nkv=4, page_size=16, max_pages=40, max_kv_len=600, splits=2, chunk=512), **change)
    of = (ctypes.c_void_p * 10)(*[4096 + (by if i == at else 0) for i in range(10)])
    words = lib.ia_layer_run_words(a["rows"], a["width"], a["ff"], a["nq"], a["nkv"], a["splits"])
    status = lib.ia_layer_run(4096, ctypes.addressof(of), 1, 4096, words, 4096, 1, *[4096] * 5, *a.values(), 1e-6, 1e-6, 1e-6, 0, 0, 0, 0.1, None)
    return status, lib.ia_last_error().decode()


@pytest.mark.parametrize("change", [dict(splits=1), dict(chunk=256), dict(max_kv_len=1025), dict(max_kv_len=0), dict(max_pages=37)])
def test_bounds_that_do_not_hold_a_row_are_refused(change):
    """Shares that do not hold the longest row, or pages that do not: such a row would wait for words that no block writes."""
    status, message = _run_status(**change)
    assert status == 1 and message.startswith("layer_run: ") and "keys" in message, message


@pytest.mark.gpu
def test_positions_beyond_the_bound_count_as_the_last_inside():
    """A row longer than the launch is laid out for, and a negative position, read nothing outside their tables and wait for nothing."""
    gen = torch.Generator(device="cuda").manual_seed(0)
    layers = _layers(gen, 2, 512, 512, 4, 2, 40)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    x = torch.empty((2, 512), dtype=torch.bfloat16, device="cuda").normal_(0.0, 1.0, generator=gen)
    table, cos, sin = torch.arange(80, dtype=torch.int32, device="cuda").view(2, 40) % 40, torch.ones((2, 64), device="cuda"), torch.zeros((2, 64), device="cuda")
    kw = dict(nq=4, nkv=2, ff=512, max_kv_len=600, eps=(1e-6,) * 3, add_one=(False,) * 3, scale=HD ** -0.5)
    kept = [(of[8].clone(), of[9].clone()) for of in layers]
    outs = []
    for positions in (i32(5000, -7), i32(599, 0)):
        for of, (k, v) in zip(layers, kept):
            of[8].copy_(k)
            of[9].copy_(v)
        outs.append(ops.layer_run(x.clone(), layers, ops.RunWords(), positions, i32(599, 627), table, cos, sin, **kw))
    assert torch.equal(*outs) and torch.isfinite(outs[0].float()).all()


def _cpu_run(layers=3, **kw):
    """A run of layers over tensors on the host, and what `takes` is asked with, for the choices that read no values."""
    from types import SimpleNamespace as NS
    from inferrs_amd.cache.storage import LayerCache
    from inferrs_amd.parts.assemble import generated_tensors
    from inferrs_amd.parts.base import block_class
    from inferrs_amd.parts.layer_run import LayerRun
    spec = _config(num_hidden_layers=layers, **kw).to_spec()
    tensors = {name: torch.zeros(tuple(t.shape), dtype=torch.bfloat16) for name, t in generated_tensors(spec).items()}
    blocks = [block_class(layer)(layer, {k: v for k, v in tensors.items() if k in block_class(layer).tensors(layer)}, torch.bfloat16, "cpu") for layer in spec.layers]
    run = LayerRun.of_model(spec, blocks)
    nkv = spec.layers[0].mixer.n_kv_heads
    cache = {i: LayerCache(i, 0, torch.zeros((2, nkv, PAGE, HD), dtype=torch.bfloat16), torch.zeros((2, nkv, HD, PAGE), dtype=torch.bfloat16)) for i in range(layers)}
    ctx = NS(max_q_len=1, max_kv_len=32, run_words=ops.RunWords(), groups=[NS(page_size=PAGE)])
    return run, ctx, torch.zeros((1, spec.layers[0].mixer.hidden), dtype=torch.bfloat16), NS(layers=cache)


def test_arrays_off_their_alignment_go_through_the_blocks():
    """A weight or a cache that is a view at an odd offset, which the kernels of the blocks check for, is none of the run's."""
    run, *step = _cpu_run()
    m, c = run.blocks[-1], step[2].layers[2]
    for holder, name in ((m.mixer.qkv, "weight"), (m.mixer.o, "weight"), (m.ffn.gate_up, "weight"), (m.ffn.down, "weight"), (m.norm_mixer, "weight"),
                         (m.norm_ffn, "weight"), (m.mixer, "q_norm_w"), (m.mixer, "k_norm_w"), (c, "k"), (c, "v")):
        assert run.takes(*step)
        t = getattr(holder, name)
        setattr(holder, name, torch.zeros(t.numel() + 1, dtype=t.dtype)[1:].view(t.shape))      # (two bytes past an aligned address, or four)
        assert not run.takes(*step), name
        setattr(holder, name, t)


def test_switches_of_the_products_reach_steps_that_the_run_would_take(monkeypatch):
    """Rows whose products a switch keeps from gemm_mid.hip, or hands to it, go through the blocks, which follow the switch."""
    run, ctx, x, storage = _cpu_run(hidden_size=2560)
    step = lambda rows: run.takes(ctx, x[:1].expand(rows, -1), storage)
    assert step(4) and step(5)
    monkeypatch.setattr(ops, "MID_PRODUCTS", "library")
    assert step(4) and not step(5)                   # (`mid_from_rows` of a width that is no power of two)
    monkeypatch.setattr(ops, "MID_PRODUCTS", "own")
    monkeypatch.setattr(ops, "MID_FROM_ROWS", 2)
    assert step(1) and not step(2)


@pytest.mark.parametrize("at,by", [(0, 2), (3, 8), (4, 4), (7, 4), (8, 2), (9, 8)])
def test_arrays_off_their_alignment_are_refused(at, by):
    status, message = _run_status(off=(at, by))
    assert status == 1 and "aligned" in message, message


def _layers(gen, n, width, ff, nq, nkv, pages):
    def draw(*shape, std=0.02, mean=0.0, dtype=torch.bfloat16):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=gen)
    out = []
    for _ in range(n):
        out.append((draw((nq + 2 * nkv) * HD, width), draw(width, nq * HD), draw(2 * ff, width), draw(width, ff),
                    draw(width, std=0.1, mean=1.0, dtype=torch.float32), draw(width, std=0.1, mean=1.0, dtype=torch.float32),
                    draw(HD, std=0.1, mean=1.0, dtype=torch.float32), draw(HD, std=0.1, mean=1.0, dtype=torch.float32),
                    draw(pages, nkv, PAGE, HD, std=1.0), draw(pages, nkv, HD, PAGE, std=1.0)))
    return out


def _exact(x, layers, lengths, tables, cos, sin, nq, nkv, eps, one):
    """The stream, and the new keys and values a layer, in 64 bits."""
    x = x.double()
    cos, sin = cos.double(), sin.double()
    rms = lambda t, w, e, o: t / torch.sqrt((t * t).mean(-1, keepdim=True) + e) * (w.double() + (1.0 if o else 0.0))
    news = []
    for wqkv, wo, wgu, wd, n1, n2, qn, kn, kc, vc in layers:
        n = x.shape[0]
        qkv = (rms(x, n1, eps[0], one[0]) @ wqkv.double().T).view(n, nq + 2 * nkv, HD)
        q, k, v = rms(qkv[:, :nq], qn, eps[2], one[2]), rms(qkv[:, nq:nq + nkv], kn, eps[2], one[2]), qkv[:, nq + nkv:]
        turn = lambda t: torch.cat([t[..., :64] * cos[:, None] - t[..., 64:] * sin[:, None], t[..., 64:] * cos[:, None] + t[..., :64] * sin[:, None]], -1)
        q, k = turn(q), turn(k)
        a = torch.empty((n, nq, HD), dtype=torch.float64, device="cuda")
        for r, length in enumerate(lengths):
            pages = tables[r][: -(-length // PAGE)] if length else tables[r][:0]
            keys = torch.cat([kc[pages].permute(0, 2, 1, 3).flatten(0, 1)[:length].double(), k[r][None]])
            values = torch.cat([vc[pages].permute(0, 3, 1, 2).flatten(0, 1)[:length].double(), v[r][None]])
            g = nq // nkv
            s = torch.einsum("hgd,khd->hgk", q[r].view(nkv, g, HD), keys) * HD ** -0.5
            a[r] = torch.einsum("hgk,khd->hgd", torch.softmax(s, -1), values).reshape(nq, HD)
        x = x + a.view(n, -1) @ wo.double().T
        h = rms(x, n2, eps[1], one[1]) @ wgu.double().T
        ff = h.shape[1] // 2
        x = x + (torch.nn.functional.silu(h[:, :ff]) * h[:, ff:]) @ wd.double().T
        news.append((k, v))
    return x, news


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm())


# (layers, width, feed-forward, query heads, key heads, cached keys of every row): one step of the inner features and odd counts of them,
# one to eight query heads a key head, rows without a cached key, the edges of pages, of a wave's step and of a block's share, shares that
# the output projection merges and that a phase of its own does, more layers than a launch takes, both forms of the products
CASES = [(1, 512, 512, 4, 4, [0]), (2, 512, 1536, 4, 1, [1, 15]), (2, 1024, 3072, 16, 8, [16, 17, 31]), (33, 512, 512, 4, 2, [32, 33]),
         (2, 1024, 3072, 16, 8, [511]), (2, 1024, 3072, 16, 8, [512, 513, 0, 1023]), (2, 1536, 2560, 8, 1, [1024, 5, 700, 47, 2100]),
         (2, 2048, 6144, 16, 8, [3000]), (1, 2560, 9728, 32, 8, [700, 64]), (1, 2560, 9728, 32, 8, [700, 64, 1]), (2, 1024, 3072, 16, 8, [9000, 40, 511, 512, 513, 3, 0]),
         (2, 1024, 3072, 16, 8, [100, 200, 300, 400, 500, 600, 700, 800]), (1, 5120, 25600, 64, 8, [300, 20]), (1, 6144, 512, 8, 8, [17, 18, 19, 20, 21, 22])]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v).replace(" ", "") for v in c))
@pytest.mark.parametrize("one", [(False, False, False), (True, True, True)])
def test_layer_run_against_64_bits(case, one):
    n, width, ff, nq, nkv, lengths = case
    if any(one) and n > 2:
        pytest.skip("the norms' form once is enough")
    rows, eps = len(lengths), (1e-6, 1e-5, 1e-4)
    gen = torch.Generator(device="cuda").manual_seed(rows * 1000 + width + ff)
    counts = [length // PAGE + 1 for length in lengths]
    pages = sum(counts) + 3
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(5)).tolist()
    widest = max(counts) + 2
    table = torch.zeros((rows, widest), dtype=torch.int32)
    at = 0
    for r, c in enumerate(counts):
        table[r, :c] = torch.tensor(order[at:at + c], dtype=torch.int32)
        at += c
    table = table.cuda()
    positions = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    slots = torch.tensor([int(table[r, length // PAGE]) * PAGE + length % PAGE for r, length in enumerate(lengths)], dtype=torch.int32, device="cuda")
    angle = positions[:, None].double() * 10000.0 ** (-torch.arange(64, device="cuda", dtype=torch.float64) / 64)
    cos, sin = angle.cos().float(), angle.sin().float()
    layers = _layers(gen, n, width, ff, nq, nkv, pages)
    if any(one):
        layers = [tuple(t - 1.0 if 4 <= i < 8 else t for i, t in enumerate(of)) for of in layers]
    x0 = torch.empty((rows, width), dtype=torch.bfloat16, device="cuda").normal_(0.0, 1.0, generator=gen)
    tables = [table[r, :c].long() for r, c in enumerate(counts)]
    want, news = _exact(x0, layers, lengths, tables, cos, sin, nq, nkv, eps, one)
    kept = [(of[8].clone(), of[9].clone()) for of in layers]
    words = ops.RunWords()
    kw = dict(nq=nq, nkv=nkv, ff=ff, max_kv_len=widest * PAGE, eps=eps, add_one=one, scale=HD ** -0.5)

    def run():
        for of, (k, v) in zip(layers, kept):
            of[8].copy_(k)
            of[9].copy_(v)
        return ops.layer_run(x0.clone(), layers, words, positions, slots, table, cos, sin, **kw)

    got = run()
    # Every layer rounds to bfloat16 eight times on the way to the stream (two norms' rows, heads, probabilities, joined heads, activations, two
    # sums), each a relative error of at most 2^-9, 2^-9 / sqrt(3) in the mean; 33 layers walk at random.
    bound = 2.0 ** -9 * math.sqrt(8 * n)
    assert _rel(got, want) < bound, (_rel(got, want), bound)
    for i, (of, (k_old, v_old), (k, v)) in enumerate(zip(layers, kept, news)):
        page, slot = (slots // PAGE).long(), (slots % PAGE).long()
        assert _rel(of[8][page, :, slot], k) < bound and _rel(of[9][page, :, :, slot], v) < bound
        k_old[page, :, slot] = of[8][page, :, slot]                # nothing else in the cache changed
        v_old[page, :, :, slot] = of[9][page, :, :, slot]
        assert torch.equal(of[8], k_old) and torch.equal(of[9], v_old)
    # the words are left ready for the next launch: the same bits again, also behind a launch of another size, and from a graph
    ops.layer_run(x0[:1].clone(), layers[:1], words, positions[:1], slots[:1], table[:1], cos[:1], sin[:1], **kw)
    assert torch.equal(run(), got)
    y = x0.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.layer_run(y, layers, words, positions, slots, table, cos, sin, **kw)
    for _ in range(3):
        y.copy_(x0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, got)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(512, 1024, 8, 2), (2560, 9728, 32, 8)], ids=["products on the matrix cores", "products by dot products"])
def test_what_is_no_number_stays_in_its_row(shape):
    """Infinities and NaN in a row of the stream and in a row's cached keys and values leave the other rows' bits alone; NaN and infinities in slots
    behind a row's length, and in pages that are nobody's, leave all rows' bits alone."""
    width, ff, nq, nkv = shape
    gen = torch.Generator(device="cuda").manual_seed(1)
    lengths, pages = [70, 33, 517], 48
    layers = _layers(gen, 2, width, ff, nq, nkv, pages)
    counts = [length // PAGE + 1 for length in lengths]
    table = torch.zeros((3, 40), dtype=torch.int32)
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(2)).to(torch.int32)
    for r, c in enumerate(counts):
        table[r, :c] = order[sum(counts[:r]):sum(counts[:r]) + c]
    x = torch.empty((3, width), dtype=torch.bfloat16, device="cuda").normal_(0.0, 1.0, generator=gen)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    slots = i32([int(table[r, length // PAGE]) * PAGE + length % PAGE for r, length in enumerate(lengths)])
    cached = torch.zeros((pages, PAGE), dtype=torch.bool)                   # the slots that some row reads, and those of row 1
    of_row_1 = torch.zeros_like(cached)
    for r, length in enumerate(lengths):
        at = torch.arange(length)
        cached[table[r, at // PAGE].long(), at % PAGE] = True
        if r == 1:
            of_row_1[table[r, at // PAGE].long(), at % PAGE] = True
    kept = [(of[8].clone(), of[9].clone()) for of in layers]
    kw = dict(nq=nq, nkv=nkv, ff=ff, max_kv_len=640, eps=(1e-6,) * 3, add_one=(False,) * 3, scale=HD ** -0.5)

    def run(x, where=None, what=0.0):
        for of, (k, v) in zip(layers, kept):
            of[8].copy_(k)
            of[9].copy_(v)
            if where is not None:
                of[8].masked_fill_(where.cuda()[:, None, :, None], what)
                of[9].masked_fill_(where.cuda()[:, None, None, :], what)
        out = ops.layer_run(x.clone(), layers, ops.RunWords(), i32(lengths), slots, table.cuda(), torch.ones((3, 64), device="cuda"), torch.zeros((3, 64), device="cuda"), **kw)
        at = (slots // PAGE).long(), (slots % PAGE).long()
        return [out] + [t for of in layers for t in (of[8][at[0], :, at[1]], of[9][at[0], :, :, at[1]])]

    want = run(x)
    assert all(torch.isfinite(t.float()).all() for t in want)
    for what in (float("nan"), float("inf"), float("-inf")):
        assert all(torch.equal(a, b) for a, b in zip(run(x, ~cached, what), want)), what
        odd = x.clone()
        odd[1, 5] = what
        for got in (run(odd), run(x, of_row_1, what)):
            assert all(torch.equal(a[[0, 2]], b[[0, 2]]) for a, b in zip(got, want)), what
            assert not torch.isfinite(got[0][1].float()).any(), what


@pytest.mark.gpu
def test_words_are_not_made_under_capture():
    x = torch.zeros((1, 512), dtype=torch.bfloat16, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(0)
    layers = _layers(gen, 1, 512, 512, 4, 4, 2)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    args = (i32(0), i32(0), i32(0, 1).view(1, 2), torch.ones((1, 64), device="cuda"), torch.zeros((1, 64), device="cuda"))
    kw = dict(nq=4, nkv=4, ff=512, max_kv_len=32, eps=(1e-6,) * 3, add_one=(False,) * 3, scale=HD ** -0.5)
    torch.cuda.synchronize()
    with pytest.raises(ops.KernelError, match="capture"):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            ops.layer_run(x, layers, ops.RunWords(), *args, **kw)


@pytest.mark.gpu
def test_operands_that_do_not_fit_are_refused():
    x = torch.zeros((1, 512), dtype=torch.bfloat16, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(0)
    (layer,) = _layers(gen, 1, 512, 512, 4, 4, 2)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    good = dict(positions=i32(0), slots=i32(0), block_table=i32(0, 1).view(1, 2), cos=torch.ones((1, 64), device="cuda"), sin=torch.zeros((1, 64), device="cuda"),
                nq=4, nkv=4, ff=512, max_kv_len=32, eps=(1e-6,) * 3, add_one=(False,) * 3, scale=HD ** -0.5)
    words = ops.RunWords()
    for change in (dict(max_kv_len=33), dict(ff=1024), dict(nq=8), dict(positions=i32(0, 1)), dict(cos=torch.ones((1, 32), device="cuda"))):
        with pytest.raises(ops.KernelError):
            ops.layer_run(x, [layer], words, **dict(good, **change))
    with pytest.raises(ops.KernelError):
        ops.layer_run(x.float(), [layer], words, **good)
    with pytest.raises(ops.KernelError):
        ops.layer_run(x, [layer[:3] + (layer[3][:, :256].contiguous(),) + layer[4:]], words, **good)


def test_questions_to_the_host_are_no_kernel_calls():
    """The tables of a step's kernels list what launches something: not the run's words and layers, which are asked for at every call."""
    lib = ops.library()
    with ops.KernelTimer() as timer:
        timed = ops.library()
        for name in ("ia_layer_run_words", "ia_layer_run_layers", "ia_gemm_wide_rows_fits", "ia_attention_mfma_has_fused", "ia_last_error"):
            if hasattr(lib, name):
                assert getattr(timed, name) is getattr(lib, name), name
        assert timed.ia_layer_run is not lib.ia_layer_run and timed.ia_rmsnorm is not lib.ia_rmsnorm
    assert not timer.records


def test_a_wait_given_up_is_an_error_once():
    words = ops.RunWords()
    words.check()
    words.given_up.fill_(1)
    with pytest.raises(ops.KernelError, match="waited in vain"):
        words.check()
    words.check()


@pytest.mark.gpu
def test_a_wait_given_up_ends_the_launch_and_tells_the_host():
    """Waits that end after one read: every block ends, the rows are no numbers, the host's word says so, and the next launch is sound."""
    gen = torch.Generator(device="cuda").manual_seed(0)
    layers = _layers(gen, 3, 512, 512, 4, 4, 4)
    x = torch.empty((2, 512), dtype=torch.bfloat16, device="cuda").normal_(0.0, 1.0, generator=gen)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    args = (i32(5, 20), i32(5, 52), i32(0, 1, 2, 3).view(2, 2), torch.ones((2, 64), device="cuda"), torch.zeros((2, 64), device="cuda"))
    kw = dict(nq=4, nkv=4, ff=512, max_kv_len=32, eps=(1e-6,) * 3, add_one=(False,) * 3, scale=HD ** -0.5)
    kept = [(of[8].clone(), of[9].clone()) for of in layers]

    def run(words, polls):
        for of, (k, v) in zip(layers, kept):
            of[8].copy_(k)
            of[9].copy_(v)
        words.polls = polls
        out = ops.layer_run(x.clone(), layers, words, *args, **kw)
        torch.cuda.synchronize()
        return out

    want, words = run(ops.RunWords(), ops.RunWords.POLLS), ops.RunWords()
    assert torch.isfinite(want.float()).all()
    assert torch.isnan(run(words, 1).float()).any()
    with pytest.raises(ops.KernelError, match="waited in vain"):
        words.check()
    for _ in range(2):
        assert torch.equal(run(words, ops.RunWords.POLLS), want)
        words.check()


@pytest.mark.gpu
def test_an_engine_raises_where_a_wait_was_given_up():
    """The step behind the one whose wait was given up raises, and so does the serving loop before it takes a token; both go on from there."""
    from inferrs_amd.engine import Engine, Entry, GenerationLoop
    from inferrs_amd.sampling import SamplingParams
    engines = [Engine.from_random(_config(), seed=3, page_size=16, num_pages=40, max_seqs=2) for _ in range(2)]
    words = engines[0].builder.run_words
    prompt = list(range(20))
    for e in engines:
        e.step([Entry("a", prompt, [])])
    words.polls = 1
    engines[0].step([Entry("a", [7], [0])], commit=False)
    torch.cuda.synchronize()
    words.polls = ops.RunWords.POLLS
    with pytest.raises(ops.KernelError, match="waited in vain"):
        engines[0].step([Entry("a", [7], [0])], commit=False)
    got, want = (e.step([Entry("a", [7], [0])]).clone() for e in engines)
    assert torch.equal(got, want)
    outputs = []
    for e, disturbed in zip(engines, (True, False)):
        e.end_request("a")
        loop = GenerationLoop(e, max_batch_size=2, decode_run=1)
        r = loop.add(prompt, SamplingParams.greedy(max_tokens=5, bypass_stop_tokens=True))
        loop.step()
        if disturbed:
            before, sample = list(r.output), loop.sampler.sample_with_logprobs

            def sample_behind_such_a_step(*a):
                words.given_up.fill_(1)
                return sample(*a)

            loop.sampler.sample_with_logprobs = sample_behind_such_a_step
            with pytest.raises(ops.KernelError, match="waited in vain"):
                loop.step()
            loop.sampler.sample_with_logprobs = sample
            assert r.output == before
        loop.run()
        outputs.append(list(r.output))
    assert outputs[0] == outputs[1] and len(outputs[0]) == 5


def _config(**kw):
    from inferrs_amd.config import Qwen3Config
    return Qwen3Config.from_dict(dict(dict(
        architectures=["Qwen3ForCausalLM"], model_type="qwen3", vocab_size=1024, hidden_size=512, intermediate_size=1024, num_hidden_layers=5,
        num_attention_heads=8, num_key_value_heads=4, head_dim=128, rope_theta=1000000.0, rms_norm_eps=1e-6, tie_word_embeddings=True,
        max_position_embeddings=4096), **kw))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 3, 8])
def test_engine_steps_with_and_without(rows, monkeypatch):
    """Decode steps behind prompts of several lengths, eager and from graphs, against the same engine without the run of layers: no further
    apart than a few roundings of the last layer's rows."""
    from inferrs_amd.engine import Engine, Entry
    engines = [Engine.from_random(_config(), seed=3, page_size=16, num_pages=400, max_seqs=8) for _ in range(2)]
    assert engines[0].model.layer_run is not None and engines[0].model.layer_run.length == 5
    engines[1].model.layer_run = None
    calls = []
    real = ops.layer_run
    monkeypatch.setattr(ops, "layer_run", lambda x, *a, **k: (calls.append(x.shape[0]), real(x, *a, **k))[1])
    gen = torch.Generator().manual_seed(rows)
    lengths = [5, 600, 33, 511, 512, 1, 64, 15][:rows]
    prompts = [torch.randint(0, 1024, (n,), generator=gen).tolist() for n in lengths]
    for e in engines:
        e.step([Entry(i, p, []) for i, p in enumerate(prompts)])
    assert not calls                                  # (portions of prompts are no steps of the run's)
    for step in range(6):
        tokens = torch.randint(0, 1024, (rows,), generator=gen).tolist()
        got, want = (e.step([Entry(i, [t], [0]) for i, t in enumerate(tokens)]).clone() for e in engines)
        assert _rel(got, want.double()) < 2.0 ** -9 * math.sqrt(8 * 5)
    assert engines[0].graph_replays > 0
    assert set(calls) == {rows} and engines[0].builder.run_words and not engines[1].builder.run_words


@pytest.mark.gpu
def test_steps_past_the_rule_go_through_the_blocks(monkeypatch):
    """Nine rows, a portion beside a single token, and contexts beyond the rule's keys take no run; eight rows of the same engine do."""
    from inferrs_amd.engine import Engine, Entry
    e = Engine.from_random(_config(max_position_embeddings=16384), seed=3, page_size=16, num_pages=3200, max_seqs=9, use_graphs=False)
    calls = []
    real = ops.layer_run
    monkeypatch.setattr(ops, "layer_run", lambda x, *a, **k: (calls.append(x.shape[0]), real(x, *a, **k))[1])
    for i in range(9):
        e.step([Entry(i, [1, 2, 3], [])])
    e.step([Entry(i, [4], [0]) for i in range(9)])
    e.step([Entry(0, [4, 5], [1]), Entry(1, [4], [0])])
    assert not calls
    e.step([Entry(i, [4], [0]) for i in range(8)])
    assert calls == [8]
    for i in range(4):                                # (3 x 12,000 keys are within the rule's 45,056, 4 x 12,000 are not)
        more = 11999 - e.cached_length(i)
        assert e.cache.reserve(i, more)
        e.cache.commit(i, more)
    e.step([Entry(i, [4], [0]) for i in range(4)])
    assert calls == [8]
    e.step([Entry(i, [4], [0]) for i in range(3)])
    assert calls == [8, 3]


@pytest.mark.gpu
def test_two_engines_on_two_streams():
    """Each engine's words are its own: steps that overlap on two streams give what they give one after the other."""
    from inferrs_amd.engine import Engine, Entry
    engines = [Engine.from_random(_config(num_hidden_layers=8), seed=s, page_size=16, num_pages=64, max_seqs=2) for s in (1, 2)]
    streams = [torch.cuda.Stream() for _ in engines]
    tokens = torch.randint(0, 1024, (20,), generator=torch.Generator().manual_seed(0)).tolist()

    def steps(together):
        out = [[], []]
        for i, e in enumerate(engines):
            e.step([Entry("a", tokens[:7], [])])
        for t in tokens:
            for i, (e, s) in enumerate(zip(engines, streams)):
                with torch.cuda.stream(s):
                    out[i].append(e.step([Entry("a", [t], [0])]).clone())
                if not together:
                    torch.cuda.synchronize()
        torch.cuda.synchronize()
        for e in engines:
            e.end_request("a")
        return out

    torch.cuda.synchronize()
    want = steps(False)
    words = [list(e.builder.run_words.values()) for e in engines]
    assert all(len(w) == 1 for w in words) and words[0][0].data_ptr() != words[1][0].data_ptr()
    got = steps(True)
    for a, b in zip(want, got):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_which_layers_form_a_run():
    """Layers that differ end a run, which one layer makes; layers of another kind are none."""
    from inferrs_amd.parts.assemble import generated_tensors
    from inferrs_amd.parts.layer_run import LayerRun
    from inferrs_amd.parts.base import block_class
    import dataclasses

    def run_of(cfg, change=None):
        spec = cfg.to_spec()
        if change:
            spec = change(spec)
        tensors = {name: torch.zeros(tuple(t.shape), dtype=torch.bfloat16) for name, t in generated_tensors(spec).items()}
        blocks = [block_class(layer)(layer, {k: v for k, v in tensors.items() if k in block_class(layer).tensors(layer)}, torch.bfloat16, "cpu") for layer in spec.layers]
        return LayerRun.of_model(spec, blocks)

    run = run_of(_config())
    assert run.length == 5 and run.stops == [0, 1, 2, 3, 4]

    def window(at):
        def change(spec):
            layers = list(spec.layers)
            layers[at] = dataclasses.replace(layers[at], mixer=dataclasses.replace(layers[at].mixer, window=64))
            return dataclasses.replace(spec, layers=type(spec.layers)(layers))
        return change

    # (runs of one and two layers were none, though measured faster: `LayerRun`)
    assert [run_of(_config(), window(n)).length for n in (1, 2, 3, 4)] == [1, 2, 3, 4] and run_of(_config(), window(0)) is None
    assert run_of(_config(num_hidden_layers=1)).length == 1
    assert run_of(_config(head_dim=64)) is None
