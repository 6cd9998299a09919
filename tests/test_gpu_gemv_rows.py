"""The fp64-matrix GEMV for int8 batches of 3..15, and of 2 over long or large matrices (gemv_rows.hip),
at the edges of its tiles: rows that end inside a tile, K that ends inside a 256-wide chunk, odd and
single-scale runs, every group size from 16 up, one to four column groups, every tile height, one and
two steps in flight, work shared between wavefronts and not; and the batches beside it that stay on the
vector form. Every output is the correctly rounded bf16 of the exact value (fp64 accumulation is within
2^-40 of it), so the bar is bit equality with the fp64 oracle."""

import ctypes

import pytest
import torch

from iron_amd import _lib
from iron_amd.operators import GEMVInt8, SwiGLUMLPDataParallelOurs
from iron_amd.operators.wire import pack_wire
from oracle import blocks as oblk
from oracle import gemv as ogemv
from oracle import norms as onorm
from oracle.numerics import bf16_bits

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _weights(M, K, G, gen):
    q = torch.randint(-128, 128, (M, K), generator=gen, dtype=torch.int16)
    s = (torch.randn(M, K // G, generator=gen) * 0.02).to(torch.bfloat16)
    return q, s


def _same(got, want, what):
    bad = int((bf16_bits(got.cpu().reshape(-1)) != bf16_bits(want.reshape(-1))).sum())
    assert bad == 0, f"{what}: {bad} of {want.numel()} values differ from the exact oracle"


@pytest.mark.parametrize("M,K,G,tile,B,domain", [
    (8, 16, 16, 8, 2, "signed"),          # (a small pair: the vector form)
    (8, 16, 16, 8, 3, "signed"),          # one slice, two tiles, one scale a row
    (8, 16, 16, 8, 5, "biased"),
    (16, 272, 16, 8, 3, "biased"),        # 17 scales a row, one slice past a chunk
    (200, 1152, 128, 8, 5, "signed"),     # nine groups: the last chunk holds one scale
    (200, 1152, 128, 8, 4, "biased"),
    (96, 768, 256, 8, 7, "signed"),       # a group per chunk
    (72, 1536, 512, 8, 2, "signed"),      # (the vector form)
    (72, 1536, 512, 8, 3, "signed"),      # groups longer than a chunk
    (72, 1536, 512, 8, 6, "biased"),
    (1032, 320, 64, 8, 9, "signed"),      # five groups, rows eight past a tile of sixteen
    (2560, 2176, 32, 4, 3, "signed"),     # half a chunk at the end
    (2564, 4096, 32, 4, 3, "signed"),     # tiles of twelve rows, the last one of eight
    (4100, 12288, 128, 4, 9, "signed"),   # of sixteen, the last one of four
    (4100, 512, 32, 4, 13, "biased"),     # four column groups, tiles and chunks shared
    (8, 12288, 32, 4, 15, "signed"),      # one tile: every wavefront holds a share of it
    (40000, 128, 32, 16, 6, "signed"),    # many whole tiles per wavefront
    (64, 16384, 128, 8, 2, "biased"),     # the longest K
    (64, 16384, 128, 8, 13, "signed"),    # few tiles: a workgroup per column group, the last of one row
    (24, 512, 16, 8, 6, "biased"),
    (256, 1040, 16, 8, 15, "signed"),
    (1000, 512, 16, 8, 7, "signed"),      # groups of 16: tiles of four rows
    (4104, 1040, 16, 8, 3, "biased"),     # and of eight
])
def test_gemv(M, K, G, tile, B, domain):
    print(f"[case] gemv rows M={M} K={K} G={G} tile={tile} B={B} {domain}", flush=True)
    gen = torch.Generator().manual_seed(M + K + B)
    q, s = _weights(M, K, G, gen)
    x = (torch.randn(B, K, generator=gen) * torch.exp(torch.randn(B, K, generator=gen))).to(
        torch.bfloat16)
    op = GEMVInt8(M=M, K=K, tile_size_input=tile, group_size=G, batch_size=B,
                  kernel_vector_size=16,
                  kernel_source="mv_int8_signed.cc" if domain == "signed" else None)
    y = torch.zeros(B, M, dtype=torch.bfloat16, device=DEV)
    op.get_callable()(pack_wire(q, s, tile, domain).to(DEV), x.to(DEV), y)
    torch.cuda.synchronize()
    _same(y, ogemv.gemv_exact(q, s, x).float().to(torch.bfloat16), "gemv")


def _bits_or_nan(got, want, what):
    got, want = got.cpu().reshape(-1), want.cpu().reshape(-1)
    nan = torch.isnan(want.float())
    assert torch.equal(torch.isnan(got.float()), nan), f"{what}: NaN elsewhere"
    _same(got[~nan], want[~nan], what)
    return int(nan.sum()), int(torch.isinf(want.float()).sum())


def _infinite_scales(M, K, G, gen, stride=3):
    """Weights with an infinite scale in every `stride`-th row, in the first, a middle or the last
    group, of either sign or of both (two groups); half of the rows have positive weights only."""
    q, s = _weights(M, K, G, gen)
    q[::2] = q[::2].abs().clamp(1, 127)
    for i, row in enumerate(range(0, M, stride)):
        g = (0, K // G // 2, K // G - 1)[i % 3]
        s[row, g] = float("inf") if i % 2 else float("-inf")
        if i % 5 == 0:
            s[row, -1 - g] = float("inf")
    return q, s


@pytest.mark.parametrize("M,K,G,tile,B,domain", [
    (16, 272, 16, 8, 3, "signed"),       # the infinite group beside slices past K
    (200, 1152, 128, 8, 5, "biased"),
    (96, 1536, 512, 8, 4, "signed"),
    (2560, 2176, 32, 4, 3, "signed"),
    (4100, 512, 32, 4, 13, "biased"),
    (8, 12288, 32, 4, 15, "signed"),
])
def test_gemv_infinite_scales(M, K, G, tile, B, domain):
    """An infinite scale gives what the batch-1 kernel gives: the sign of the scaled slice sums, NaN
    where a slice sums to zero or two differ in sign; so do an infinite x and a NaN scale."""
    print(f"[case] infinite scales M={M} K={K} G={G} B={B} {domain}", flush=True)
    gen = torch.Generator().manual_seed(M + K + B)
    q, s = _infinite_scales(M, K, G, gen)
    x = torch.randn(B, K, generator=gen).to(torch.bfloat16)
    x[0] = x[0].abs() + 0.5            # with positive weights: slices of one sign
    x[1, K // 2:] = 0.0
    x[-1, 3] = float("inf")
    s[1, 0] = float("nan")
    op = lambda n: GEMVInt8(M=M, K=K, tile_size_input=tile, group_size=G, batch_size=n,  # noqa: E731
                            kernel_vector_size=16,
                            kernel_source="mv_int8_signed.cc" if domain == "signed" else None)
    w, xd = pack_wire(q, s, tile, domain).to(DEV), x.to(DEV)
    y = torch.zeros(B, M, dtype=torch.bfloat16, device=DEV)
    op(B).get_callable()(w, xd, y)
    want, one = torch.zeros_like(y), op(1).get_callable()
    for b in range(B):
        one(w, xd[b], want[b])
    torch.cuda.synchronize()
    slices = (q.double().reshape(M, -1, 16) * x.double().reshape(B, 1, -1, 16)).sum(-1)
    exact = (slices * s.double().repeat_interleave(G // 16, 1)).sum(-1).float().to(torch.bfloat16)
    nans, infs = _bits_or_nan(want, exact, "batch 1")
    assert nans and infs
    _bits_or_nan(y, exact, "gemv")


@pytest.mark.parametrize("B", [3, 5])
def test_fused_infinite_scales(B):
    """The same in the other forms: x staged by the RMSNorm prologue with the argmax epilogue, gate/up
    with two matrices, down from fp32 x, each against one row at a time."""
    print(f"[case] infinite scales in the fused forms, B={B}", flush=True)
    D, FF, G = 512, 1152, 32
    gen = torch.Generator().manual_seed(B)
    x, a = (torch.randn(B, D, generator=gen).abs().to(torch.bfloat16).to(DEV) for _ in range(2))
    nw = torch.ones(D, dtype=torch.bfloat16, device=DEV)
    w = pack_wire(*_infinite_scales(2000, D, G, gen), 8, "signed").to(DEV)

    def head(x):
        n = x.shape[0]
        logits = torch.zeros(n, 2000, dtype=torch.bfloat16, device=DEV)
        keys = torch.zeros(n, dtype=torch.int64, device=DEV)
        _lib.call("iron_lm_head", w.data_ptr(), _lib.IRON_WEIGHT_INT8, x.data_ptr(), nw.data_ptr(),
                  ctypes.c_float(1e-6), logits.data_ptr(), keys.data_ptr(), n, 2000, D, G, 8, 0,
                  torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return logits

    nans, infs = _bits_or_nan(head(x), torch.cat([head(x[b:b + 1]) for b in range(B)]), "logits")
    assert nans and infs

    def mlp(cur, a, wires):
        n = cur.shape[0]
        op = SwiGLUMLPDataParallelOurs(D=D, FF=FF, group_size=G, epsilon=1e-6, batch=n,
                                       kernel_source="mv_int8_signed.cc")
        ws = torch.zeros(op.workspace_bytes(), dtype=torch.uint8, device=DEV)
        nxt = torch.zeros(n, D, dtype=torch.bfloat16, device=DEV)
        tiles = (op.tile_rows_gu, op.tile_rows_gu, op.tile_rows_d)
        packed = [pack_wire(*w, t, "signed").to(DEV) for w, t in zip(wires, tiles)]
        op.get_callable()(cur, a, nw, *packed, ws, nxt)
        torch.cuda.synchronize()
        # gh follows the 16 KiB of counters at the front of the workspace
        return nxt, ws[16384:16384 + n * FF * 4].view(torch.float32).reshape(n, FF)

    plain = [_weights(M, K, G, gen) for M, K in ((FF, D), (FF, D), (D, FF))]
    wires = [_infinite_scales(FF, D, G, gen), plain[1], plain[2]]
    nxt, gh = mlp(x, a, wires)
    one = [mlp(x[b:b + 1], a[b:b + 1], wires) for b in range(B)]
    _bits_or_nan(nxt, torch.cat([r[0] for r in one]), "nxt of NaN")
    want = torch.cat([r[1] for r in one])
    assert torch.equal(torch.isnan(gh), torch.isnan(want))
    inf = torch.isinf(want)
    assert bool(inf.any()) and torch.equal(gh[inf], want[inf])
    wires = [plain[0], plain[1], _infinite_scales(D, FF, G, gen)]
    nxt = mlp(x, a, wires)[0]
    nans, infs = _bits_or_nan(
        nxt, torch.cat([mlp(x[b:b + 1], a[b:b + 1], wires)[0] for b in range(B)]), "nxt")
    assert nans and infs


@pytest.mark.parametrize("M,tile", [
    (294912, 294912),    # one row block of 4.8 GB
    (393216, 131072),    # three of 2.2 GB
])
def test_gemv_large_blocks(M, tile):
    """Row blocks past 32-bit offsets: the same bits as the batch-1 kernel."""
    print(f"[case] gemv rows large blocks M={M} tile={tile}", flush=True)
    K, G, B = 16384, 128, 4
    gen = torch.Generator(DEV).manual_seed(M)
    w = torch.empty(M // tile, tile * K + tile * (K // G) * 2, dtype=torch.uint8, device=DEV)
    for b in w:
        b[:tile * K].random_(0, 256, generator=gen)
        s = torch.randn(tile * (K // G), generator=gen, device=DEV) * 0.02
        b[tile * K:] = s.to(torch.bfloat16).view(torch.uint8)
    x = torch.randn(B, K, generator=gen, device=DEV).to(torch.bfloat16)
    op = lambda n: GEMVInt8(M=M, K=K, tile_size_input=tile, group_size=G, batch_size=n,  # noqa: E731
                            kernel_vector_size=16, kernel_source="mv_int8_signed.cc").get_callable()
    y = torch.zeros(B, M, dtype=torch.bfloat16, device=DEV)
    op(B)(w.reshape(-1), x, y)
    one = op(1)
    want = torch.zeros_like(y)
    for b in range(B):
        one(w.reshape(-1), x[b], want[b])
    torch.cuda.synchronize()
    _same(y, want.cpu(), "gemv")


@pytest.mark.parametrize("V,D,G,B", [
    (5000, 1024, 32, 3),
    (5000, 1152, 128, 12),     # ragged columns staged in LDS
    (1032, 4352, 64, 5),       # rows longer than the prologue's registers hold, one wavefront each
    (1032, 16384, 128, 4),     # staged rows that fit one at a time: a launch per batch row
    (256, 16384, 128, 4),      # few rows: the vector form in pairs of batch rows
    (512, 1024, 32, 15),       # (the last pair half empty)
    (1024, 4096, 64, 9),
    (1024, 1024, 64, 6),       # and here the fp64-matrix form again
])
def test_head_with_norm(V, D, G, B):
    """Staged RMSNorm prologue and the argmax epilogue (first index of the largest logit)."""
    print(f"[case] head V={V} D={D} G={G} B={B}", flush=True)
    gen = torch.Generator().manual_seed(V + D + B)
    q, s = _weights(V, D, G, gen)
    x = torch.randn(B, D, generator=gen).to(torch.bfloat16)
    nw = (torch.rand(D, generator=gen) + 0.5).to(torch.bfloat16)
    w, xd, nwd = pack_wire(q, s, 8, "signed").to(DEV), x.to(DEV), nw.to(DEV)
    logits = torch.zeros(B, V, dtype=torch.bfloat16, device=DEV)
    keys = torch.zeros(B, dtype=torch.int64, device=DEV)
    _lib.call("iron_lm_head", w.data_ptr(), _lib.IRON_WEIGHT_INT8, xd.data_ptr(), nwd.data_ptr(),
              ctypes.c_float(1e-6), logits.data_ptr(), keys.data_ptr(), B, V, D, G, 8, 0,
              torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    want = ogemv.gemv_exact(q, s, onorm.rms_norm(x, nw, 1e-6)).float().to(torch.bfloat16)
    _same(logits, want, "logits")
    idx = [(~k) & 0xFFFFFFFF for k in keys.cpu().tolist()]
    assert idx == [int(torch.argmax(r.float())) for r in want.reshape(B, V)]


@pytest.mark.parametrize("D,B,norm", [
    (1024, 3, False), (1056, 3, True), (1056, 5, False), (1024, 8, True),
])
def test_large_head(D, B, norm):
    """Two steps in flight (12 and more for each wavefront), ending on either half of the ring, with
    argmax keys: the same bits as one row at a time."""
    print(f"[case] large head D={D} B={B} norm={norm}", flush=True)
    V, G, tile = 100016, 32, 8
    gen = torch.Generator(DEV).manual_seed(D + B)
    w = torch.randint(0, 256, (V // tile, tile * D + tile * (D // G) * 2), generator=gen,
                      dtype=torch.uint8, device=DEV)
    s = torch.randn(V // tile, tile * (D // G), generator=gen, device=DEV) * 0.02
    w[:, tile * D:] = s.to(torch.bfloat16).view(torch.uint8)
    x = torch.randn(B, D, generator=gen, device=DEV).to(torch.bfloat16)
    nw = (torch.rand(D, generator=gen, device=DEV) + 0.5).to(torch.bfloat16)

    def head(x):
        n = x.shape[0]
        logits = torch.zeros(n, V, dtype=torch.bfloat16, device=DEV)
        keys = torch.zeros(n, dtype=torch.int64, device=DEV)
        _lib.call("iron_lm_head", w.data_ptr(), _lib.IRON_WEIGHT_INT8, x.data_ptr(),
                  nw.data_ptr() if norm else None, ctypes.c_float(1e-6), logits.data_ptr(),
                  keys.data_ptr(), n, V, D, G, tile, 0, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return logits, keys

    logits, keys = head(x)
    one = [head(x[b:b + 1]) for b in range(B)]
    _same(logits, torch.cat([r[0] for r in one]).cpu(), "logits")
    assert keys.tolist() == [int(r[1][0]) for r in one]


@pytest.mark.parametrize("D,FF,G,tile,B", [
    (1152, 2304, 128, 8, 2),   # (the vector form)
    (1152, 2304, 128, 8, 3),   # nine groups, half a chunk at the end of every row of gate/up
    (1152, 2304, 128, 8, 4),
    (2560, 1536, 32, 4, 4),    # down in tiles of twelve rows
    (1024, 12288, 128, 12, 2),  # a pair in down alone (its rows are long)
    (256, 768, 32, 12, 3),     # fewer tiles than CUs
    (4608, 512, 128, 4, 5),    # batches of 5..8: rows longer than the prologue's registers hold
])
def test_mlp(D, FF, G, tile, B):
    """gate/up (two matrices, residual RMSNorm, SwiGLU) and down (fp32 x, residual)."""
    print(f"[case] mlp D={D} FF={FF} G={G} B={B}", flush=True)
    gen = torch.Generator().manual_seed(D + FF + B)
    op = SwiGLUMLPDataParallelOurs(D=D, FF=FF, group_size=G, epsilon=1e-6, batch=B,
                                   tile_rows_gu=tile, kernel_source="mv_int8_signed.cc")
    lin = lambda M, K: ogemv.rtn_quantize(torch.randn(M, K, generator=gen) * 0.05, G)  # noqa: E731
    wg, wu, wd = lin(FF, D), lin(FF, D), lin(D, FF)
    cur, a = (torch.randn(B, D, generator=gen).to(torch.bfloat16) for _ in range(2))
    n_pf = (torch.rand(D, generator=gen) + 0.5).to(torch.bfloat16)
    ws = torch.zeros(op.workspace_bytes(), dtype=torch.uint8, device=DEV)
    nxt = torch.zeros(B, D, dtype=torch.bfloat16, device=DEV)
    wires = [pack_wire(*w, t, "signed").to(DEV)
             for w, t in ((wg, tile), (wu, tile), (wd, op.tile_rows_d))]
    op.get_callable()(cur.to(DEV), a.to(DEV), n_pf.to(DEV), *wires, ws, nxt)
    torch.cuda.synchronize()
    want, _ = oblk.swiglu_mlp(cur, a, n_pf, wg, wu, wd, 1e-6)
    _same(nxt, want, "nxt")


@pytest.mark.parametrize("D,FF,QD,G,B", [
    (512, 1536, 1024, 32, 5),
    (512, 1536, 1024, 32, 8),
    (1024, 8192, 1024, 128, 7),     # gemv_mlp's tallest gate/up
    (2048, 2048, 4096, 64, 6),      # and longest
    (2048, 6144, 2048, 32, 5),      # with G = 32 and the output projection
])
def test_mlp_small_batch(D, FF, QD, G, B):
    """Batches of 5..8 over small matrices take the GEMV kernels inside the fused MLP: two column
    groups in gate/up and, from fp32, in down; with the output projection."""
    print(f"[case] mlp on the GEMV path, D={D} FF={FF} QD={QD} G={G} B={B}", flush=True)
    gen = torch.Generator().manual_seed(B)
    op = SwiGLUMLPDataParallelOurs(D=D, FF=FF, QD=QD, fuse_o=True, group_size=G, epsilon=1e-6,
                                   batch=B, tile_rows_gu=4 * max(1, FF // D),
                                   kernel_source="mv_int8_signed.cc")
    lin = lambda M, K: ogemv.rtn_quantize(torch.randn(M, K, generator=gen) * 0.05, G)  # noqa: E731
    wo, wg, wu, wd = lin(D, QD), lin(FF, D), lin(FF, D), lin(D, FF)
    cur = torch.randn(B, D, generator=gen).to(torch.bfloat16)
    cx = torch.randn(B, QD, generator=gen).to(torch.bfloat16)
    n_pf = (torch.rand(D, generator=gen) + 0.5).to(torch.bfloat16)
    ws = torch.zeros(op.workspace_bytes(), dtype=torch.uint8, device=DEV)
    a, nxt = (torch.zeros(B, D, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    wires = [pack_wire(*w, t, "signed").to(DEV)
             for w, t in ((wo, op.tile_rows_o), (wg, op.tile_rows_gu), (wu, op.tile_rows_gu),
                          (wd, op.tile_rows_d))]
    op.get_callable()(cur.to(DEV), cx.to(DEV), n_pf.to(DEV), *wires, ws, a, nxt)
    torch.cuda.synchronize()
    want, want_a = oblk.swiglu_mlp(cur, cx, n_pf, wg, wu, wd, 1e-6, wo=wo)
    _same(a, want_a, "a")
    _same(nxt, want, "nxt")
