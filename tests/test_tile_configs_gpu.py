"""The layer GEMMs choose their tile by the number of rows. Every output takes its K blocks in the same order whatever
the tile, so a row's result must not depend on it: each kernel over `rows` rows, on both sides of every limit of the
rules (test_tile_rules.py checks on the host that the row counts here are), against the same rows taken in pieces of at
most 1025 (which run the smallest tiles, and which the parity tests check against the oracle), bit for bit. The pieces
go past `rows` and start elsewhere than the call's tiles, so every row sits in another place of another launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T, D, HIDP, PXH = 1025, 1024, 2816, 4736
F32, U8 = torch.float32, torch.uint8


def _codes(g, dev, *shape):
    return torch.randn(*shape, generator=g, device=dev).to(torch.float8_e4m3fn).view(U8)


class _W:
    """random weight codes [N][K] and block scales, or pack24 values and indices"""

    def __init__(self, g, dev, N, K, sp):
        self.s = torch.rand(N // 128, K // 128, generator=g, device=dev) * 0.01
        self.v = _codes(g, dev, N // 16, K // 128, 64, 16) if sp else _codes(g, dev, N, K)
        # index nibbles p0 | p1 << 2 with p0 < p1: 0x4 (0, 1), 0xe (2, 3), 0x9 (1, 2)
        self.x = torch.tensor([0x4E944E94, 0x4E9494E4, 0x44444444, -0x11111112], dtype=torch.int32, device=dev)
        self.x = self.x[torch.randint(0, 4, (N // 16, K // 128, 64), generator=g, device=dev)].contiguous() if sp else None

    def args(self, X):
        return (X.ptr(self.v),) + ((X.ptr(self.x),) if self.x is not None else ()) + (X.ptr(self.s),)


PAST = 129   # rows that the operands hold past `rows`


def _pieces(rows):
    """[0, 700) and then steps of 1025, to PAST rows past `rows`"""
    edges = [0, *range(700, rows + PAST, T), rows + PAST]
    return list(zip(edges[:-1], edges[1:]))


RES_ROWS = [1, 65, 1408, 1409, 2817, 4096, 4097, 4353, 8192, 8193, 8200, 8447, 8448, 10250, 16384, 16400]
TAIL_BASES, TAILS = [1280, 2048, 4224, 10240], [1, 8, 16, 17, 32, 33, 48, 49, 64]


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("rows", RES_ROWS)
def test_rows_do_not_depend_on_the_tile(dev, xt, rows, sparse):
    _check_rows(dev, xt, rows, sparse)


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("base", TAIL_BASES)
def test_partial_row_tiles_of_every_tile(dev, xt, base, sparse):
    """a last row tile with 1 to 64 rows below M (a wave runs only the 16-row tiles that hold such rows), at row counts
    that take fc1's smaller tile and each of the three tiles of the out-projection and fc2"""
    for tail in TAILS:
        _check_rows(dev, xt, base + tail, sparse)


def _check_rows(dev, xt, rows, sparse):
    print(f"tile configurations: {rows} rows, sparse {sparse}", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    sfx = "_sp" if sparse else ""
    g = torch.Generator(device=dev)
    g.manual_seed(rows)
    R = rows + PAST
    lds = R + 256                # a piece's last tile reads scales (of rows it drops) up to 127 rows past its own
    h8, hs = _codes(g, dev, R, D), torch.rand(8, lds, generator=g, device=dev) * 0.01
    m8, ms = _codes(g, dev, R, HIDP), torch.rand(22, lds, generator=g, device=dev) * 0.01
    stat = torch.rand(22, lds, 2, generator=g, device=dev) * 20
    x0 = torch.randn(R, D, generator=g, device=dev).half()
    cn, dn = torch.rand(D, generator=g, device=dev), torch.rand(D, generator=g, device=dev)
    wo, w1, w2 = (_W(g, dev, *s, sparse) for s in ((D, D), (2 * HIDP, D), (D, HIDP)))

    def run(bounds):
        xo, xf = x0.clone(), x0.clone()
        mo, so, to = (torch.zeros(R, HIDP, dtype=U8, device=dev), torch.zeros(22, lds, device=dev),
                      torch.zeros(22, lds, 2, device=dev))
        for a, b in bounds:
            n = b - a
            at = lambda t: P(t.reshape(-1)[a * t.stride(0):])           # row a of [rows][..]
            pl = lambda t: P(t.reshape(-1)[a * t.stride(1):])           # row a of every scale plane
            assert getattr(L, "eva_k_oproj" + sfx)(at(h8), pl(hs), lds, *wo.args(xt), at(xo), n, st) == 0
            assert getattr(L, "eva_k_fc1" + sfx)(at(h8), pl(hs), lds, *w1.args(xt), at(mo), pl(so), pl(to), n, st) == 0
            assert getattr(L, "eva_k_fc2" + sfx)(at(m8), pl(ms), lds, *w2.args(xt), pl(stat), P(cn), P(dn), at(xf), n, st) == 0
        torch.cuda.synchronize()
        return xo, xf, mo, so, to

    (xo, xf, mo, so, to), (rxo, rxf, rmo, rso, rto) = run([(0, rows)]), run(_pieces(rows))
    for got, ref, first in ((xo, rxo, x0), (xf, rxf, x0), (mo, rmo, torch.zeros_like(mo))):
        assert torch.equal(got[:rows], ref[:rows]) and torch.equal(got[rows:], first[rows:])   # nothing past the rows
    for got, ref in ((so, rso), (to, rto)):
        assert torch.equal(got[:, :rows], ref[:, :rows]) and not got[:, rows:].any()


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("nb", [2, 3, 5, 6, 7])
def test_qkv_rows_do_not_depend_on_the_tile(dev, xt, nb, sparse):
    print(f"qkv tile configurations: {nb} images, sparse {sparse}", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev)
    g.manual_seed(nb)
    rows = nb * T
    lds = rows + 256
    h8, hs = _codes(g, dev, rows, D), torch.rand(8, lds, generator=g, device=dev) * 0.01
    cs = torch.rand(1024, 32, 2, generator=g, device=dev)
    w = _W(g, dev, 3 * D, D, sparse)

    def run(step):
        q, k, v = (torch.zeros(nb, 16, 1088 * 64, dtype=torch.int16, device=dev) for _ in range(3))
        for b in range(0, nb, step):
            at = lambda t: P(t[b:])
            assert getattr(L, "eva_k_qkv" + ("_sp" if sparse else ""))(
                P(h8[b * T:]), P(hs.reshape(-1)[b * T:]), lds, *w.args(xt), P(cs), at(q), at(k), at(v), step * T, st) == 0
        torch.cuda.synchronize()
        return q, k, v

    for got, ref in zip(run(nb), run(1)):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("nb", [2, 3])
def test_patch_embedding_does_not_depend_on_the_tile(dev, xt, nb):
    """wd: nb images at once (64 x 64 tiles up to two, 128 x 128 from three) against each alone; PixAI: 128 nb 9 rows
    against pieces of 128."""
    print(f"patch embedding: {nb} images", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev)
    g.manual_seed(nb)
    x_in = torch.randn(nb * 1152, 592, generator=g, device=dev).half()
    pe, pos = (torch.randn(D, 592, generator=g, device=dev) * 0.05).half(), torch.randn(T, D, generator=g, device=dev)
    a, b = (torch.zeros(nb * T, D, dtype=torch.float16, device=dev) for _ in range(2))
    assert L.eva_k_pe(P(x_in), P(pe), P(pos), P(a), nb, st) == 0
    for i in range(nb):
        assert L.eva_k_pe(P(x_in[1024 * i:]), P(pe), P(pos), P(b[T * i:]), 1, st) == 0
    assert torch.equal(a, b) and a.abs().sum() > 0
    ref = (x_in[:1024].cpu().double() @ pe.cpu().double().T + pos[1:].cpu().double()).numpy()
    assert abs(a[1:T].cpu().double().numpy() - ref).max() <= 2.0 ** -11 * abs(ref).max() + 1e-4   # fp16 + fp32 sums
    rows = nb * 1152
    a, b = (torch.zeros(rows, D, dtype=torch.float16, device=dev) for _ in range(2))
    assert L.px_k_pe(P(x_in), P(pe), P(a), rows, st) == 0
    for r in range(0, rows, 128):
        assert L.px_k_pe(P(x_in[r:]), P(pe), P(b[r:]), 128, st) == 0
    assert torch.equal(a, b) and a.abs().sum() > 0


@pytest.mark.parametrize("nseq,T_,TP", [(3, 1025, 1088), (9, 576, 576), (40, 65, 128)])
def test_attention_does_not_depend_on_the_block(dev, xt, nseq, T_, TP):
    """sequences at once (128 queries a block) against each alone (64 queries a block)"""
    print(f"attention: {nseq} sequences of {T_}", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev)
    g.manual_seed(T_)
    q, k = (torch.randn(nseq, 16, TP, 64, generator=g, device=dev).bfloat16() for _ in range(2))
    v = torch.randn(nseq, 16, 64, TP, generator=g, device=dev).bfloat16()
    rows = nseq * T_

    def run(step):
        o8, s = torch.zeros(rows, D, dtype=U8, device=dev), torch.zeros(8, rows, device=dev)
        for i in range(0, nseq, step):
            assert L.eva_k_flash_seq(P(q[i:]), P(k[i:]), P(v[i:]), P(o8[i * T_:]), P(s.reshape(-1)[i * T_:]), rows, step,
                                     T_, TP, None, st) == 0
        torch.cuda.synchronize()
        return o8, s

    for got, ref in zip(run(nseq), run(1)):
        assert torch.equal(got, ref) and got.float().abs().sum() > 0


@pytest.mark.parametrize("rows", [1, 15, 17, 5184 + 5])
def test_hln_ragged_rows(dev, xt, orc, rows):
    """rows that do not fill the last block of 16: y bit for bit, scores within the order of 32-bit sums, nothing
    written past the last row"""
    import numpy as np

    print(f"px_k_hln: {rows} rows", flush=True)
    r = np.random.default_rng(rows)
    x = (r.standard_normal((rows, D)) * 1.5 + 0.2).astype(np.float16)
    gw, gb = (1 + 0.1 * r.standard_normal(D)).astype(np.float32), (0.1 * r.standard_normal(D)).astype(np.float32)
    hpos, U = (r.standard_normal((5184, D)) * 0.2).astype(np.float16), (r.standard_normal((16, D)) * 0.05).astype(np.float32)
    d = [torch.from_numpy(a).to(dev) for a in (x, gw, gb, hpos, U)]
    y, s = torch.full((rows + 16, D), 7, dtype=torch.int16, device=dev), torch.full((rows + 16, 16), 7.0, device=dev)
    P = xt.ptr
    assert xt.lib.px_k_hln(P(d[0]), P(d[1]), P(d[2]), P(d[3]), 5184, P(d[4]), P(y), P(s), rows,
                           torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    y_ref, s_ref = orc.px_hln(x.view(np.uint16), 5184, gw, gb, hpos.view(np.uint16), U)
    y, s = y.cpu().numpy(), s.cpu().numpy()
    assert (y[:rows].view(np.uint16) == y_ref).all() and (y[rows:] == 7).all() and (s[rows:] == 7).all()
    terms = np.abs(y_ref.view(np.float16).astype(np.float64)) @ np.abs(U.astype(np.float64)).T
    assert np.all(np.abs(s[:rows] - s_ref) <= 2e-6 * terms)   # 32-bit sums of 1024 terms in two orders


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("M,N,K,off,pad", [(1, 64, 128, 0, 0), (65, 207, 256, 1, 3), (1025, 3071, 1024, 0, 1),
                                            (1025, 1024, 512, 3, 0), (2050, 3088, 128, 0, 0), (4100, 3072, 256, 5, 2),
                                            (8200, 2000, 128, 0, 8), (1025, 13461, 128, 0, 0), (4100, 3072, 256, 0, 0),
                                            (3000, 4096, 2048, 8, 8), (2049, 3072, 256, 16, 16), (2050, 3088, 256, 3, 1)])
def test_gemm_any_alignment_and_tile(dev, xt, M, N, K, off, pad, sparse):
    """C at any element offset and row stride, N ragged: the same bits as the fp32 output of the aligned call row by
    row (in pieces of 64 rows: the smallest tiles), bf16 rounded to nearest even, nothing written outside C."""
    N = (N + 15) // 16 * 16 if sparse else N
    print(f"gemm {M} x {N} x {K}, offset {off}, pad {pad}, sparse {sparse}", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev)
    g.manual_seed(M + N)
    Np = (N + 127) // 128 * 128
    a, sa = _codes(g, dev, M, K), torch.rand(K // 128, M + 64, generator=g, device=dev) * 0.01
    w = _W(g, dev, Np, K, sparse)
    fn = L.eva_k_gemm_sp if sparse else L.eva_k_gemm
    ref = torch.zeros(M, Np, device=dev)
    for r in range(0, M, 64):
        assert fn(P(a[r:]), K, P(sa.reshape(-1)[r:]), M + 64, *w.args(xt), min(64, M - r), N, K, P(ref[r:]), Np, 1, st) == 0
    for kind, dt in ((1, torch.float32), (0, torch.bfloat16)):
        ldc = N + pad
        buf = torch.full((off + M * ldc + 64,), 7.0, dtype=dt, device=dev)
        assert fn(P(a), K, P(sa), M + 64, *w.args(xt), M, N, K, P(buf[off:]), ldc, kind, st) == 0
        torch.cuda.synchronize()
        want = torch.full_like(buf, 7.0)
        want[off:off + M * ldc].view(M, ldc)[:, :N] = ref[:, :N].to(dt)
        assert torch.equal(buf, want)


PX_FC1_ROWS = [2048, 2049, 3328, 3329, 12288, 12289]


@pytest.mark.parametrize("with_rs", [False, True])
@pytest.mark.parametrize("rows", PX_FC1_ROWS)
def test_px_fc1_rows_do_not_depend_on_the_tile(dev, xt, rows, with_rs):
    print(f"px fc1: {rows} rows, rs {with_rs}", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev)
    g.manual_seed(rows)
    lds = rows + 256
    h8, hs = _codes(g, dev, rows, D), torch.rand(8, lds, generator=g, device=dev) * 0.01
    w, bias = _W(g, dev, PXH, D, False), torch.randn(PXH, generator=g, device=dev)
    rs = torch.rand(PXH, generator=g, device=dev) + 0.5 if with_rs else None

    def run(step):
        m8, ms = torch.zeros(rows, PXH, dtype=U8, device=dev), torch.zeros(37, lds, device=dev)
        for r in range(0, rows, step):
            assert L.px_k_fc1(P(h8[r:]), P(hs.reshape(-1)[r:]), lds, *w.args(xt), P(bias), P(rs), P(m8[r:]),
                              P(ms.reshape(-1)[r:]), min(step, rows - r), st) == 0
        torch.cuda.synchronize()
        return m8, ms

    for got, ref in zip(run(rows), run(1000)):
        assert torch.equal(got, ref)


PX_ROWS = [1, 65, 4096, 4097, 8192, 8193, 8447, 8448, 10273, 16384]


@pytest.mark.parametrize("rows", PX_ROWS)
def test_px_residual_rows_do_not_depend_on_the_tile(dev, xt, rows):
    """PixAI's out-projection (K = 1024) and fc2 (K = 4736) on both sides of the limits of their tiles"""
    print(f"px residual GEMMs: {rows} rows", flush=True)
    L, P, st = xt.lib, xt.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev)
    g.manual_seed(rows)
    R = rows + PAST
    lds = R + 256
    for fn, K in ((L.px_k_proj, D), (L.px_k_fc2, PXH)):
        a8, as_ = _codes(g, dev, R, K), torch.rand(K // 128, lds, generator=g, device=dev) * 0.01
        w, bias = _W(g, dev, D, K, False), torch.randn(D, generator=g, device=dev)
        x0 = torch.randn(R, D, generator=g, device=dev).half()

        def run(bounds):
            x = x0.clone()
            for a, b in bounds:
                assert fn(P(a8[a:]), P(as_.reshape(-1)[a:]), lds, *w.args(xt), P(bias), P(x[a:]), b - a, st) == 0
            torch.cuda.synchronize()
            return x

        got, ref = run([(0, rows)]), run(_pieces(rows))
        assert torch.equal(got[:rows], ref[:rows]) and torch.equal(got[rows:], x0[rows:])
        assert not torch.equal(got[:rows], x0[:rows])
