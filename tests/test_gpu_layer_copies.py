"""kf_layer_copies: one launch's bf16 copies are kf_dequant's, bit for bit, in every layout (rows back to back, gate | up interleaved in blocks of 16), and the routes that find them give what the
same products give on bf16 weights; what is not served is left to the routes as they were."""
import ctypes as C

import pytest
import torch

from koifish_amd import lib as L
from koifish_amd import runtime as R

pytestmark = pytest.mark.gpu


def _layer(ctx, dim, q, kv, ffn, types=(L.Q4,) * 7):
    g = torch.Generator(device=ctx.device)
    g.manual_seed(dim + ffn)
    shapes = [(q, dim), (kv, dim), (kv, dim), (dim, q), (ffn, dim), (ffn, dim), (dim, ffn)]
    ws = [ctx.quantize((torch.randn(*s, device=ctx.device, generator=g) * 0.05).bfloat16(), t) for s, t in zip(shapes, types)]
    return ws, [w.desc() for w in ws]


def _copies(ctx, descs, n):
    need = ctx.hip.kf_layer_copies_bytes(*[C.byref(d) for d in descs], n)
    if not need:
        return 0, None
    scratch = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device=ctx.device)
    assert ctx.hip.kf_set_scratch(ctx.h, C.c_void_p(scratch.data_ptr()), C.c_size_t(need)) == 0
    assert ctx.hip.kf_layer_copies(ctx.h, *[C.byref(d) for d in descs], n) == 0
    ctx.sync()
    assert bool((scratch[need:] == 0x5A).all())   # nothing past the workspace
    return need, scratch


@pytest.mark.parametrize("dim,q,kv,ffn,n", [(1024, 2048, 1024, 3072, 320), (256, 512, 256, 512, 2047), (2560, 4096, 1024, 9728, 321)])
def test_copies_and_routes(ctx, dim, q, kv, ffn, n):
    ws, descs = _layer(ctx, dim, q, kv, ffn)
    try:
        need, scratch = _copies(ctx, descs, n)
        assert need
        bf = [ctx.dequant(w) for w in ws]
        out, off = scratch.view(torch.bfloat16), 0
        for i in (0, 1, 2, 3):
            assert torch.equal(out[off:off + bf[i].numel()].view_as(bf[i]), bf[i])
            off += bf[i].numel()
        both = torch.stack([bf[4].view(ffn // 16, 16, dim), bf[5].view(ffn // 16, 16, dim)], 1).reshape(2 * ffn, dim)
        assert torch.equal(out[off:off + both.numel()].view_as(both), both)
        off += both.numel()
        assert torch.equal(out[off:off + bf[6].numel()].view_as(bf[6]), bf[6])
        # o and down through kf_linear: the product on the copy, against fp32 on the dequantised values (sums of K bf16 products in fp32, one bf16 rounding: 2^-8 of a value, 2^-8 of the sum's scale)
        for i in (3, 6):
            x = torch.randn(n, ws[i].ne1, device=ctx.device).bfloat16()
            y = torch.zeros(n, ws[i].ne0, device=ctx.device, dtype=torch.bfloat16)
            assert ctx.hip.kf_linear(ctx.h, C.byref(descs[i]), x.data_ptr(), y.data_ptr(), None, n, 1.0, 0.0, 0, None) == 0
            ref = x.float() @ bf[i].float().t()
            assert float((y.float() - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max())
            assert torch.equal(out[:bf[0].numel()].view_as(bf[0]), bf[0])   # the split-K slots do not touch the copies
        x = torch.randn(n, dim, device=ctx.device).bfloat16()
        act, up = (torch.zeros(n, ffn, device=ctx.device, dtype=torch.bfloat16) for _ in range(2))
        assert ctx.hip.kf_gateup_swiglu_batch(ctx.h, C.byref(descs[4]), C.byref(descs[5]), x.data_ptr(), act.data_ptr(), up.data_ptr(), n) == 0
        g, u = x.float() @ bf[4].float().t(), x.float() @ bf[5].float().t()
        ref = torch.nn.functional.silu(g) * u
        assert float((act.float() - ref).abs().max()) <= 2.0 ** -6 * float(ref.abs().max())
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
    finally:
        ctx.sync()
        ctx.hip.kf_set_scratch(ctx.h, None, 0)


def _routes(ctx, ws, descs, dim, q, kv, ffn, n):
    """(first and last matrix of the set, call that returns the outputs, their values from the seven matrices) of every route that looks for copies"""
    x, xo, xd = (torch.randn(n, k, device=ctx.device).bfloat16() for k in (dim, q, ffn))
    res = torch.randn(n, dim, device=ctx.device).bfloat16()
    out = lambda *cols: [torch.zeros(n, c, device=ctx.device, dtype=torch.bfloat16) for c in cols]
    h, p = ctx.hip, [C.byref(d) for d in descs]

    def single(i, xi, residual):
        y, = out(dim)
        assert h.kf_linear(ctx.h, p[i], xi.data_ptr(), y.data_ptr(), None, n, 1.0, 0.0, int(residual), res.data_ptr() if residual else None) == 0
        return [y]

    def stacked(rope):
        y = out(q, kv, kv)
        if rope:   # neither norms nor a table: the products themselves, by the launch that would norm and rotate them
            assert h.kf_qkv_rope_batch(ctx.h, p[0], p[1], p[2], x.data_ptr(), *[t.data_ptr() for t in y], n, None, None, None, 0, q // 128, kv // 128, 128, 1e-6) == 0
        else:
            assert h.kf_linear_multi(ctx.h, 3, (C.POINTER(L.Weight) * 3)(*[C.pointer(d) for d in descs[:3]]), x.data_ptr(), (C.c_void_p * 3)(*[t.data_ptr() for t in y]), n) == 0
        return y

    def gated():
        act, up = out(ffn, ffn)
        assert h.kf_gateup_swiglu_batch(ctx.h, p[4], p[5], x.data_ptr(), act.data_ptr(), up.data_ptr(), n) == 0
        return [act]
    mm = lambda a, w: a.float() @ w.float().t()
    silu = torch.nn.functional.silu
    return [(0, 2, lambda: stacked(True), lambda w: [mm(x, w[i]) for i in range(3)]), (0, 2, lambda: stacked(False), lambda w: [mm(x, w[i]) for i in range(3)]),
            (3, 3, lambda: single(3, xo, False), lambda w: [mm(xo, w[3])]), (3, 3, lambda: single(3, xo, True), lambda w: [mm(xo, w[3]) + res.float()]),
            (4, 5, gated, lambda w: [silu(mm(x, w[4])) * mm(x, w[5])]), (6, 6, lambda: single(6, xd, True), lambda w: [mm(xd, w[6]) + res.float()])]


@pytest.mark.parametrize("dim,q,kv,ffn,n", [(1024, 2048, 1024, 3072, 320), (1024, 2048, 1024, 3072, 2047), (256, 512, 256, 512, 2047), (2560, 4096, 1024, 9728, 321),
                                             (256, 512, 256, 2560, 2047),      # gate | up on 192 x 256 tiles, 5120 rows: no multiple of 192
                                             (512, 4096, 1024, 9728, 2047)])   # q | k | v and gate | up on 256 x 256 tiles
def test_every_route_multiplies_the_copies_until_the_end(ctx, dim, q, kv, ffn, n):
    """with a set's copies halved its products are those of halved matrices, with the copies ended those of the matrices; what another matrix is dequantised to meanwhile lies behind the copies.  2^-6 of
    the result's scale covers every route's roundings (gate and up: each rounded to 2^-9, then their product; behind a residual two roundings); a half would be off by 2^-1"""
    ws, descs = _layer(ctx, dim, q, kv, ffn)
    real = [ctx.dequant(w) for w in ws]
    off = [0]
    for w in real:
        off.append(off[-1] + w.numel())
    near = lambda got, want, tol: all(float((a.float() - b).abs().max()) <= tol * float(b.abs().max()) for a, b in zip(got, want))
    try:
        need, scratch = _copies(ctx, descs, n)
        copies = scratch.view(torch.bfloat16)[:off[-1]]
        before = copies.clone()
        routes = _routes(ctx, ws, descs, dim, q, kv, ffn, n)
        for first, last, call, ref in routes:
            halved = [w * 0.5 if first <= i <= last else w for i, w in enumerate(real)]
            assert near(call(), ref(real), 2.0 ** -6)
            copies[off[first]:off[last + 1]] *= 0.5   # exact
            assert near(call(), ref(halved), 2.0 ** -6)
            copies[off[first]:off[last + 1]] *= 2.0
        other = ctx.quantize_nf4((torch.randn(1024, 1024, device=ctx.device) * 0.05).bfloat16(), 3)   # a row form: dequantised into the scratch
        xs, ys, do = torch.randn(8, 1024, device=ctx.device).bfloat16(), torch.zeros(8, 1024, device=ctx.device, dtype=torch.bfloat16), other.desc()
        assert ctx.hip.kf_linear(ctx.h, C.byref(do), xs.data_ptr(), ys.data_ptr(), None, 8, 1.0, 0.0, 0, None) == 0, ctx.hip.kf_last_error()
        assert near([ys], [xs.float() @ ctx.dequant(other).float().t()], 2.0 ** -7) and torch.equal(copies, before)
        copies *= 0.5
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
        assert all(near(call(), ref(real), 2.0 ** -6) for _, _, call, ref in routes)
    finally:
        ctx.sync()
        ctx.hip.kf_layer_copies_end(ctx.h)
        ctx.hip.kf_set_scratch(ctx.h, None, 0)


def test_not_served_is_left_alone(ctx):
    _, descs = _layer(ctx, 256, 512, 256, 512)
    p = [C.byref(d) for d in descs]
    assert ctx.hip.kf_layer_copies_bytes(*p, 319) == 0 and ctx.hip.kf_layer_copies(ctx.h, *p, 2047) == 1   # too few rows; no workspace
    mixed = [C.byref(d) for d in _layer(ctx, 256, 512, 256, 512, (L.Q4,) * 6 + (L.F8E5M2,))[1]]
    assert ctx.hip.kf_layer_copies_bytes(*mixed, 2047) == 0
    odd = [C.byref(d) for d in _layer(ctx, 256, 384, 128, 512)[1]]   # rows no multiple of 256: the stacked route does not take them
    assert ctx.hip.kf_layer_copies_bytes(*odd, 2047) == 0



def test_a_set_with_a_matrix_of_fewer_rows_is_another_set(ctx):
    """the first 256 rows of q have q's pointer: stacked with k and v they are not the set that resident copies hold"""
    n, dim = 2047, 256
    ws = [ctx.quantize((torch.randn(m, dim, device=ctx.device) * 0.05).bfloat16(), L.F8E5M2) for m in (2048, 1024, 1024)]
    x = torch.randn(n, dim, device=ctx.device).bfloat16()
    arena = torch.zeros((4096 + 2304) * dim * 2 + 4096, dtype=torch.uint8, device=ctx.device)
    try:
        assert ctx.hip.kf_set_dequant_arena(ctx.h, C.c_void_p(arena.data_ptr()), C.c_size_t(arena.numel())) == 0
        for rows in (2048, 256):
            descs = [w.desc() for w in ws]
            descs[0].ne0 = rows
            y = [torch.zeros(n, m, device=ctx.device, dtype=torch.bfloat16) for m in (rows, 1024, 1024)]
            w3, y3 = (C.POINTER(L.Weight) * 3)(*[C.pointer(d) for d in descs]), (C.c_void_p * 3)(*[t.data_ptr() for t in y])
            assert ctx.hip.kf_linear_multi(ctx.h, 3, w3, x.data_ptr(), y3, n) == 0, ctx.hip.kf_last_error()
            for out, w in zip(y, ws):
                want = x.float() @ ctx.dequant(w).float()[: out.shape[1]].t()
                assert float((out.float() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max())   # fp32 sums, one bf16 rounding
    finally:
        ctx.sync()
        ctx.hip.kf_set_dequant_arena(ctx.h, None, 0)


def test_captured_launches_do_without_the_copies(ctx):
    """a product captured between kf_layer_copies and _end is replayed when the copies are gone and their place holds something else"""
    n = 320
    ws, descs = _layer(ctx, 1024, 2048, 1024, 3072)
    x = torch.randn(n, 2048, device=ctx.device).bfloat16()
    y, g = torch.zeros(n, 1024, device=ctx.device, dtype=torch.bfloat16), C.c_void_p()
    want = x.float() @ ctx.dequant(ws[3]).float().t()
    try:
        _, scratch = _copies(ctx, descs, n)
        assert ctx.hip.kf_graph_begin(ctx.h) == 0
        rc = ctx.hip.kf_linear(ctx.h, C.byref(descs[3]), x.data_ptr(), y.data_ptr(), None, n, 1.0, 0.0, 0, None)
        assert ctx.hip.kf_graph_end(ctx.h, C.byref(g)) == 0 and rc == 0
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
        ctx.sync()
        for fill in (0, 0x3C):
            scratch.fill_(fill)
            y.zero_()
            assert ctx.hip.kf_graph_launch(ctx.h, g) == 0
            ctx.sync()
            assert float((y.float() - want).abs().max()) <= 2.0 ** -7 * float(want.abs().max())   # the in-register product: 2^-7 as in the tests of that kernel
    finally:
        ctx.sync()
        if g:
            ctx.hip.kf_graph_destroy(g)
        ctx.hip.kf_set_scratch(ctx.h, None, 0)


def test_flags_written_over_behind_the_copies_are_cleared(ctx):
    """copies that end just below the split-K slots leave too little to lend them; a matrix dequantised there meanwhile lies on their flags, and the next product in k-pieces clears them first"""
    M, K, n, words = 1024, 3072, 384, 2048   # the flags: the last 8 KiB of the slots
    w = ctx.quantize((torch.randn(M, K, device=ctx.device) * 0.05).bfloat16(), L.Q4)
    x, y, d = torch.randn(n, K, device=ctx.device).bfloat16(), torch.zeros(n, M, device=ctx.device, dtype=torch.bfloat16), w.desc()
    want = x.float() @ ctx.dequant(w).float().t()
    _, descs = _layer(ctx, 256, 512, 256, 512)
    slots, need = ctx.hip.kf_resident_scratch_bytes() - 512, ctx.hip.kf_layer_copies_bytes(*[C.byref(e) for e in descs], 2047)
    copies = need - slots - 512
    rows = (slots + 128) // 4096   # of 2048 values: as much as lies behind the copies
    other = ctx.quantize_nf4((torch.randn(rows, 2048, device=ctx.device) * 0.05).bfloat16(), 3)
    xo, yo, do = torch.randn(8, 2048, device=ctx.device).bfloat16(), torch.zeros(8, rows, device=ctx.device, dtype=torch.bfloat16), other.desc()
    arena = torch.zeros(M * K * 2 + 4096, dtype=torch.uint8, device=ctx.device)
    scratch = torch.zeros(copies + slots + 128, dtype=torch.uint8, device=ctx.device)
    assert scratch.data_ptr() % 256 == 0 and copies % 256 == 0 and slots % 256 == 0 and rows * 4096 > slots - 4 * words

    def product():
        assert ctx.hip.kf_set_dequant_arena(ctx.h, C.c_void_p(arena.data_ptr()), C.c_size_t(arena.numel())) == 0
        y.zero_()
        assert ctx.hip.kf_linear(ctx.h, C.byref(d), x.data_ptr(), y.data_ptr(), None, n, 1.0, 0.0, 0, None) == 0
        assert float((y.float() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max())
        assert ctx.hip.kf_set_dequant_arena(ctx.h, None, 0) == 0
    try:
        assert ctx.hip.kf_set_scratch(ctx.h, C.c_void_p(scratch.data_ptr()), C.c_size_t(scratch.numel())) == 0
        product()
        flags = scratch[copies + slots - 4 * words:copies + slots].view(torch.int32)
        assert len(flags.unique()) == 2   # raised ones and zeros
        assert ctx.hip.kf_layer_copies(ctx.h, *[C.byref(e) for e in descs], 2047) == 0
        assert ctx.hip.kf_linear(ctx.h, C.byref(do), xo.data_ptr(), yo.data_ptr(), None, 8, 1.0, 0.0, 0, None) == 0, ctx.hip.kf_last_error()
        assert len(flags.unique()) > 2
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
        product()
        assert len(flags.unique()) == 2
    finally:
        ctx.sync()
        ctx.hip.kf_set_dequant_arena(ctx.h, None, 0)
        ctx.hip.kf_set_scratch(ctx.h, None, 0)


# pieces that a tile's workgroup adds up itself, of 64 x 64 and of 128 x 128 tiles, and pieces of other workgroups; numbers of k-steps that the pieces do not divide
@pytest.mark.parametrize("M,K,n,pieces", [(1024, 3072, 515, 6), (1024, 3072, 2047, 3), (1008, 3200, 700, 6), (656, 9856, 330, 19), (1024, 3072, 2300, 2), (2048, 6144, 1030, 2), (1040, 3200, 2201, 2),
                                          (2048, 6144, 515, 4), (2064, 6272, 515, 4)])
def test_down_is_cut_into_the_same_pieces(ctx, M, K, n, pieces):
    """The cuts of k are part of a product's result, so they are told apart here: two large terms that cancel take with them whatever stands in the same piece as they do and nothing else.  Every term is a small whole
    number or 15 * 2^40 of either sign, the sums of the other pieces are whole numbers below 512: the result is exact but for its rounding."""
    steps = K // 64
    cut = torch.tensor([steps * p // pieces * 64 for p in range(pieces + 1)], device=ctx.device)
    w = torch.randint(0, 16, (M, K), device=ctx.device).float()
    w[:, 64::128], w[:, 65::128] = 0.0, 15.0                     # a group's range is 0 .. 15: its 4-bit storage holds the numbers as they are
    lo, hi = cut[:-1], cut[1:]
    first, last, mid = lo + 32, hi - 32, lo + 200
    w[:, first], w[:, last] = 15.0, 15.0
    ws, _ = _layer(ctx, 1024, 2048, 1024, 3072)
    ws[6] = ctx.quantize(w.bfloat16(), L.Q4)                     # (the last matrix: widths are not compared)
    assert torch.equal(ctx.dequant(ws[6]).float().view_as(w), w)
    descs = [e.desc() for e in ws]
    x, at = torch.zeros(n, K, device=ctx.device), torch.arange(n, device=ctx.device) % pieces
    x[:, mid] = 1.0
    x[torch.arange(n), first[at]], x[torch.arange(n), last[at]] = 2.0 ** 40, -2.0 ** 40
    small = w[:, mid].t()                                        # [pieces, M]
    want = (small.sum(0) - small[at]).bfloat16()
    x, y = x.bfloat16(), torch.zeros(n, M, device=ctx.device, dtype=torch.bfloat16)
    try:
        need, scratch = _copies(ctx, descs, n)
        assert need and ctx.hip.kf_linear(ctx.h, C.byref(descs[6]), x.data_ptr(), y.data_ptr(), None, n, 1.0, 0.0, 0, None) == 0
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
        ctx.sync()
    finally:
        ctx.hip.kf_set_scratch(ctx.h, None, 0)
    assert torch.equal(y, want)


def test_copies_whose_offsets_pass_32_bits(ctx):
    """gate | up of 65792 x 16384: the interleaved copy is 4 311 744 512 bytes long, rows from 65536 on lie past 2^32; every row against kf_dequant of its matrix"""
    dim, ffn, n = 16384, 65792, 2047
    gate, up = (ctx.quantize(torch.randn(ffn, dim, device=ctx.device, dtype=torch.bfloat16), L.Q4) for _ in range(2))
    small = [ctx.quantize((torch.randn(*s, device=ctx.device) * 0.05).bfloat16(), L.Q4) for s in ((256, dim), (256, dim), (256, dim), (dim, 256), (dim, 512))]   # (the last stands for down: widths are not compared)
    ws = small[:4] + [gate, up, small[4]]
    descs = [w.desc() for w in ws]
    try:
        need, scratch = _copies(ctx, descs, n)
        assert need > 2 ** 32
        off = sum(w.ne0 * w.ne1 * 2 for w in small[:4])
        rows = scratch[off:off + 4 * ffn * dim].view(torch.bfloat16).view(ffn // 16, 2, 16, dim)
        for i, w in enumerate((gate, up)):
            assert torch.equal(rows[:, i], ctx.dequant(w).view(ffn // 16, 16, dim))
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
    finally:
        ctx.sync()
        ctx.hip.kf_set_scratch(ctx.h, None, 0)


def test_swiglu_rows_whose_offsets_pass_32_bits(ctx):
    """gate | up with 2^23 + 65536 FFN rows: from token 254 of a tile on a row lies past 2^32 bytes; some columns of every token against fp32 on the dequantised values"""
    dim, ffn, n = 128, (1 << 23) + 65536, 320
    ws, descs = _layer(ctx, dim, 2048, 512, ffn)
    try:
        need, scratch = _copies(ctx, descs, n)
        assert need
        x = torch.randn(n, dim, device=ctx.device).bfloat16()
        act, up = (torch.zeros(n, ffn, device=ctx.device, dtype=torch.bfloat16) for _ in range(2))
        assert ctx.hip.kf_gateup_swiglu_batch(ctx.h, C.byref(descs[4]), C.byref(descs[5]), x.data_ptr(), act.data_ptr(), up.data_ptr(), n) == 0
        ctx.sync()
        at = torch.cat([torch.arange(64), torch.randint(0, ffn, (512,)), torch.arange(ffn - 64, ffn)]).to(ctx.device)
        g, u = (x.float() @ ctx.dequant(w)[at].float().t() for w in (ws[4], ws[5]))
        ref = torch.nn.functional.silu(g) * u
        assert float((act[:, at].float() - ref).abs().max()) <= 2.0 ** -6 * float(ref.abs().max())
        assert ctx.hip.kf_layer_copies_end(ctx.h) == 0
    finally:
        ctx.sync()
        ctx.hip.kf_set_scratch(ctx.h, None, 0)
