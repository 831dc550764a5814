"""GPU parity at the sizes where a launch shape can go wrong: edges of tiles, remainders, the smallest
and largest of a kernel's range, against the CPU oracle (bars: tests/util.py)."""
import numpy as np
import pytest

import lastengine_amd as le
import oracle
from tests.util import acts, check_close, wbytes

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def absmag(ty, q, rows, cols, xs):
    w = oracle.dequant_rows(ty, q, rows, cols).astype(np.float64)
    return np.abs(np.atleast_2d(xs).astype(np.float64)) @ np.abs(w).T


# super-blocks that do not divide over the waves: one item or fewer than waves, 4 waves (more row
# tiles than CUs), 8 and 16 waves, items of two, and a K whose images need fewer waves
@pytest.mark.parametrize("name", list(le.MV_TYPES))
@pytest.mark.parametrize("rows,nsb", [(37, 1), (4112, 3), (100, 7), (4100, 18), (64, 27), (48, 43), (17, 54), (16, 200)])
def test_matvec_ragged_split(engine, name, rows, nsb):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, rows, cols, seed=rows + nsb)
    x = acts(cols, 5 + nsb)
    mag = absmag(ty, q, rows, cols, x)[0]
    y = torch.full((rows,), float("nan"), device="cuda")
    print("ragged split", name, rows, cols, flush=True)
    engine.mv(ty, dev(q), dev(x), y, rows, cols)
    check_close(y.cpu().numpy(), oracle.matvec(ty, q, rows, cols, x), mag)
    # int8 mode: exact integer products, only the fp32 sums differ (as tests/test_gpu_formats.py)
    xq, xd, xs = oracle.quant_x(x)
    y.fill_(float("nan"))
    engine.mv_q8(ty, None, dev(xq), dev(xd), dev(xs), y, rows, cols, 0, 1, w=dev(q))
    want = oracle.matvec_q8(ty, q, rows, cols, xq, xd, xs).astype(np.float64)
    assert np.all(np.abs(y.cpu().numpy() - want) <= 1e-5 * mag + 1e-30)


# an item size can be handed back to the automatic choice, and the GEMM knobs take the values that the header names
def test_options_automatic(fresh_engine):
    import torch
    opts = {"Q4_K": "ms_p", "Q6_K": "ms_p6", "Q8_0": "ms_p80", "Q4_0": "ms_p40", "Q5_K": "ms_p5k", "Q3_K": "ms_p3k", "IQ2_S": "ms_p2s",
            "IQ2_XXS": "ms_piq", "IQ3_XXS": "ms_piq"}
    rows, cols = 4112, 8192
    for name, opt in opts.items():
        ty = le.MV_TYPES[name]
        dq, dx = dev(wbytes(ty, 257, cols, seed=ty)).reshape(-1).repeat(16), dev(acts(cols, 1))
        outs = []
        for v in (None, 1, 2, 0):
            if v is not None:
                fresh_engine.set_option(opt, v)
            outs.append(torch.empty(rows, device="cuda"))
            fresh_engine.mv(ty, dq, dx, outs[-1], rows, cols)
        assert torch.equal(outs[0].view(torch.int32), outs[3].view(torch.int32)), opt
        assert not torch.equal(outs[1].view(torch.int32), outs[2].view(torch.int32)), opt
        for bad in (3, -1):
            with pytest.raises(le.LeError) as e:
                fresh_engine.set_option(opt, bad)
            assert e.value.code == -1, opt
    for k, v in [("mt", 0), ("mt", 1), ("mmg_mt", 0), ("mmg_mt", 1), ("mmg_gp", 0), ("mmg_gp", 1), ("gq_cfg", 21), ("gq_cfg", 22), ("gq_cfg", 0)]:
        fresh_engine.set_option(k, v)
    for v in (20, 23, -1):
        with pytest.raises(le.LeError):
            fresh_engine.set_option("gq_cfg", v)


# the pipelined GEMM: its 64- and 128-token blocks (the latter where the former overfill the chip), first and last
# token count, ragged last row tile (moved back to be whole), one super-block, K slices, super-blocks whose scale is
# zero (offsets only) between ones whose scales differ by 2^20
@pytest.mark.parametrize("name", ["Q4_K", "Q5_K"])
@pytest.mark.parametrize("rows,nsb,m", [(256, 1, 33), (257, 2, 64), (511, 3, 65), (300, 4, 129), (8448, 2, 513)])
def test_gemm_pipelined(engine, name, rows, nsb, m):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, rows, cols, seed=rows + m).reshape(rows, nsb, -1).copy()
    rng = np.random.default_rng(m)
    scale = rng.choice(np.float16([0.0, 2.0 ** -14, 0.01, 64.0]), size=(rows, nsb)).astype(np.float16)
    some = rng.random((rows, nsb)) < 0.3
    d = q[:, :, 0:2].copy().view(np.float16)[:, :, 0]
    q[:, :, 0:2] = np.where(some, scale, d)[:, :, None].view(np.uint8).reshape(rows, nsb, 2)
    x = acts(m * cols, 7 + m).reshape(m, cols)
    pick = np.unique(np.r_[0:8, rows - 264:rows - 248, rows - 8:rows].clip(0, rows - 1))  # oracle rows
    y = torch.full((m, rows), float("nan"), device="cuda")
    print("pipelined GEMM", name, rows, cols, m, flush=True)
    try:
        engine.set_option("gq_cfg", 21 if m > 512 else 22)  # less work than the pipelined kernel is chosen for
        engine.gemm(ty, dev(q), dev(x), m, y, rows, cols)
    finally:
        engine.set_option("gq_cfg", 0)
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    sel = np.ascontiguousarray(q[pick])
    check_close(got[:, pick], oracle.matmat(ty, sel, len(pick), cols, x), absmag(ty, sel, len(pick), cols, x))


# the few-token kernel: its three token counts (4, 8, 16) and their edges, fewer rows than a tile and a ragged last one,
# one super-block, waves without a super-block, K in slices summed through the workspace (56 super-blocks), and more
# row tiles than one round of blocks
@pytest.mark.parametrize("name", list(le.MV_TYPES))
@pytest.mark.parametrize("rows,nsb,m", [(5, 1, 2), (37, 3, 4), (300, 9, 5), (40, 56, 3), (40, 56, 8), (130, 7, 9), (40, 43, 16), (33000, 1, 3)])
def test_gemm_few_tokens(engine, name, rows, nsb, m):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, rows, cols, seed=rows + nsb)
    x = acts(m * cols, 3 + m).reshape(m, cols)
    x[m - 1] *= np.float32(1e-20)  # a token of another magnitude
    x[0, :256] = 0.0
    y = torch.full((m, rows), float("nan"), device="cuda")
    print("few tokens", name, rows, cols, m, flush=True)
    engine.gemm(ty, dev(q), dev(x), m, y, rows, cols)
    w = oracle.dequant_rows(ty, q, rows, cols).astype(np.float64)
    want, mag = x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T
    # two fp16 halves: 2^-22 a value, fp32 sums of 8 products' chains and nsb super-blocks (2^-24 each); one half
    # (9 tokens and more, and Q4_K's own kernel): 2^-11; 15-bit activations (Q4_K, 2 tokens): 3.1e-5 of a block's maximum
    tol = 1e-5 if m <= 8 and ty != le.Q4_K else 1e-3
    assert np.all(np.abs(y.cpu().numpy() - want) <= tol * mag + 1e-30), float(np.max(np.abs(y.cpu().numpy() - want) / (mag + 1e-30)))


# ... an output head's rows with K in slices, on the workspace that le_gemm_workspace_size_rows states (by default) and on
# the one without room for the slices' sums, below nine tokens none at all: the vector kernels' 15-bit activations there
@pytest.mark.parametrize("name", ["Q6_K", "IQ2_S"])
def test_gemm_few_tokens_head(engine, name):
    import torch
    ty, rows, cols, m = le.MV_TYPES[name], 70000, 4096, 8
    q = wbytes(ty, 64, cols, seed=3)
    dw = dev(q).reshape(-1).repeat(-(-rows // 64))[:rows * le.row_bytes(ty, cols)].clone()
    x = acts(m * cols, 4).reshape(m, cols)
    w = oracle.dequant_rows(ty, q, 64, cols).astype(np.float64)
    want, mag = x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T
    small = torch.empty(engine.gemm_workspace_size(ty, m, cols), dtype=torch.uint8, device="cuda")
    for kw, tol in (({}, 1e-5), ({"ws": small}, 1e-3), ({"ws": 0, "ws_bytes": 0}, 1e-3)):
        y = torch.full((m, rows), float("nan"), device="cuda")
        print("few tokens head", name, list(kw), flush=True)
        engine.gemm(ty, dw, dev(x), m, y, rows, cols, **kw)
        for r in (0, 64 * 500, rows - rows % 64):
            got = y[:, r:r + 64].cpu().numpy()
            n = got.shape[1]
            assert np.all(np.abs(got - want[:, :n]) <= tol * mag[:, :n])


# grouped few-pair form: a tile's edges (8 and 9 pairs at 8 a pass, 16 and 17 at 16), empty slots at both ends,
# one super-block and one row tile (one wave), waves sharing a tile, a K whose images do not fit the LDS, every pair to one
# slot (few tiles, each shared by more blocks), tiles past the first 256 slots
@pytest.mark.parametrize("name", list(le.MV_TYPES))
@pytest.mark.parametrize("rows,nsb,counts", [(16, 1, (0, 1, 0)), (37, 3, (0, 8, 0, 9, 0, 0, 0, 0, 1, 0)), (272, 7, (16, 0, 17, 1, 2)),
                                             (2064, 4, (0, 3, 9, 0, 0, 0, 0)), (50, 17, (12, 5, 0, 0)), (40, 30, (2, 1)),
                                             (40, 13, (12, 5, 0, 0)), (40, 14, (12, 5, 0, 0)), (40, 16, (12, 5, 0, 0)),
                                             (1300, 3, (0,) * 9 + (70,) + (0,) * 7), (33, 2, (1, 9) + (0,) * 260 + (700, 0, 17, 1))])
def test_grouped_few_pairs(engine, name, rows, nsb, counts):
    import torch
    ty, cols, nslot = le.MV_TYPES[name], 256 * nsb, len(counts)
    q = wbytes(ty, nslot * rows, cols, seed=rows + nsb)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    npair = int(off[-1])
    x = acts(npair * cols, 9 + nsb).reshape(npair, cols)
    x[npair - 1] *= np.float32(1e-20)  # a row of another magnitude
    rng = np.random.default_rng(nsb)
    in_idx, out_idx = rng.permutation(npair).astype(np.int32), rng.permutation(npair).astype(np.int32)
    y = torch.full((npair, rows), float("nan"), device="cuda")
    print("grouped few pairs", name, rows, cols, counts, flush=True)
    engine.mm_grouped(ty, dev(off), dev(in_idx), dev(out_idx), nslot, npair, dev(x), y, rows, cols, w=dev(q))
    got = y.cpu().numpy()[out_idx]
    w = oracle.dequant_rows(ty, q, nslot * rows, cols).astype(np.float64).reshape(nslot, rows, cols)
    for s in range(nslot):
        xs = x[in_idx[off[s]:off[s + 1]]].astype(np.float64)
        # activations rounded to fp16 (2^-11 each), fp32 sums far below it
        assert np.all(np.abs(got[off[s]:off[s + 1]] - xs @ w[s].T) <= 1e-3 * (np.abs(xs) @ np.abs(w[s]).T) + 1e-30)


# grouped tiles of 32, 64 and 128 pairs past the first 256 slots (the blocks' walk takes 256 at a time), some slots empty,
# tiles with one pair of their last
@pytest.mark.parametrize("name", ["Q4_K", "Q6_K", "Q5_K"])
@pytest.mark.parametrize("mean,bm", [(8, 32), (20, 64), (70, 128)])
def test_grouped_tiles_many_slots(engine, name, mean, bm):
    import torch
    ty, rows, cols, nslot = le.MV_TYPES[name], 300, 256, 270
    counts = np.random.default_rng(mean).poisson(mean, nslot)
    counts[[0, 7, 255, 256, 269]] = (0, 2 * bm + 1, bm + 1, 0, bm)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    npair = int(off[-1])
    assert 6 * nslot < npair and (npair <= 16 * nslot) == (bm == 32) and (npair > 64 * nslot) == (bm == 128)
    q = wbytes(ty, nslot * rows, cols, seed=mean).reshape(nslot, -1)
    x, perm = acts(npair * cols, mean).reshape(npair, cols), np.random.default_rng(2).permutation(npair).astype(np.int32)
    y = torch.full((npair, rows), float("nan"), device="cuda")
    print("grouped tiles, many slots", name, npair, flush=True)
    engine.mm_grouped(ty, dev(off), dev(perm), dev(perm), nslot, npair, dev(x), y, rows, cols, w=dev(q))
    got = y.cpu().numpy()
    assert np.isfinite(got).all()
    for s in (1, 7, 63, 64, 254, 255, 257, 269):
        p = perm[off[s]:off[s + 1]]
        if len(p):
            check_close(got[p], oracle.matmat(ty, q[s], rows, cols, x[p]), absmag(ty, q[s], rows, cols, x[p]))


# dequantization: waves of 64 units: a part of one, exactly one, one unit more, several grid strides (256 CUs x 16 blocks)
@pytest.mark.parametrize("name", list(le.MV_TYPES))
@pytest.mark.parametrize("rows,nsb", [(1, 1), (8, 1), (3, 3), (64, 16), (16500, 8)])
def test_dequant_units(engine, name, rows, nsb):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, min(rows, 64), cols, seed=rows + nsb)
    reps = -(-rows // len(q))
    w = torch.cat([dev(np.zeros(2, np.uint8)), dev(q).reshape(-1).repeat(reps)])[2:2 + rows * le.row_bytes(ty, cols)]  # 2-byte aligned
    out = torch.full((rows * cols + 64,), 7.0, device="cuda")
    print("dequant", name, rows, cols, flush=True)
    engine.dequant_rows(ty, w, out, rows, cols)
    want = np.tile(oracle.dequant_rows(ty, q, len(q), cols).reshape(len(q), cols), (reps, 1))[:rows]
    got = out.cpu().numpy()
    assert np.array_equal(got[:rows * cols].view(np.uint32), want.reshape(-1).view(np.uint32))
    assert (got[rows * cols:] == 7.0).all()


@pytest.mark.parametrize("name", ["Q8_0", "Q4_0"])
def test_dequant_units_single_blocks(engine, name):
    import torch
    ty = le.MV_TYPES[name]
    for rows, cols in ((1, 32), (65, 32), (13, 160)):
        q = wbytes(ty, rows, cols, seed=rows)
        out = torch.full((rows * cols + 64,), 7.0, device="cuda")
        print("dequant", name, rows, cols, flush=True)
        engine.dequant_rows(ty, dev(q), out, rows, cols)
        got, want = out.cpu().numpy(), oracle.dequant_rows(ty, q, rows, cols)
        assert np.array_equal(got[:rows * cols].view(np.uint32), np.asarray(want, np.float32).reshape(-1).view(np.uint32))
        assert (got[rows * cols:] == 7.0).all()


# small GEMMs: the first token count, token tiles with one row of their last, a ragged last row tile, K slices (even
# counts) and none (odd ones), both block shapes and the first sizes past each
@pytest.mark.parametrize("name", list(le.MV_TYPES))
@pytest.mark.parametrize("rows,nsb,m", [(1, 1, 33), (130, 3, 65), (1000, 4, 33), (640, 8, 225), (2049, 12, 100), (2176, 16, 129), (4100, 16, 193)])
def test_gemm_small(engine, name, rows, nsb, m):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, rows, cols, seed=rows + m)
    x = acts(m * cols, 7 + m).reshape(m, cols)
    pick = np.unique(np.r_[0:8, rows // 2:rows // 2 + 8, rows - 8:rows].clip(0, rows - 1))  # oracle rows
    y = torch.full((m, rows), float("nan"), device="cuda")
    print("small GEMM", name, rows, cols, m, flush=True)
    engine.gemm(ty, dev(q), dev(x), m, y, rows, cols)
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    sel = np.ascontiguousarray(q.reshape(rows, -1)[pick])
    check_close(got[:, pick], oracle.matmat(ty, sel, len(pick), cols, x), absmag(ty, sel, len(pick), cols, x))


# long K on 4 waves: items of one where only they leave room for two blocks a CU (112 super-blocks; Q6_K 88), of two
# otherwise; two super-blocks an item for IQ2_XXS on 8 waves: the same bits as with the item size set
@pytest.mark.parametrize("name,opt,rows,nsb,p", [("Q5_K", "ms_p5k", 4112, 112, 1), ("Q4_K", "ms_p", 4112, 112, 1), ("Q6_K", "ms_p6", 4112, 88, 1),
                                                 ("Q6_K", "ms_p6", 4112, 112, 2), ("Q5_K", "ms_p5k", 4112, 88, 2), ("IQ2_XXS", "ms_piq", 2048, 32, 2)])
def test_matvec_item_size(engine, fresh_engine, name, opt, rows, nsb, p):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    dq = dev(wbytes(ty, 64, cols, seed=nsb)).reshape(-1).repeat(-(-rows // 64))[:rows * le.row_bytes(ty, cols)].clone()
    dx = dev(acts(cols, nsb))
    fresh_engine.set_option(opt, p)
    print("item size", name, rows, cols, p, flush=True)
    a, b = torch.empty(rows, device="cuda"), torch.empty(rows, device="cuda")
    engine.mv(ty, dq, dx, a, rows, cols)
    fresh_engine.mv(ty, dq, dx, b, rows, cols)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    fresh_engine.set_option(opt, 3 - p)
    fresh_engine.mv(ty, dq, dx, b, rows, cols)
    assert not torch.equal(a.view(torch.int32), b.view(torch.int32))  # the item sizes sum in different orders


# weights that are not 16-byte aligned (a tensor inside a file image): tiles loaded straight to LDS are not taken for
# them, in a pointer table slot by slot
@pytest.mark.parametrize("name", ["Q4_K", "Q5_K"])
@pytest.mark.parametrize("shift", [2, 8])
@pytest.mark.parametrize("rows,nsb,m", [(300, 3, 40), (4096, 8, 300), (256, 1, 3)])
def test_gemm_unaligned_weights(engine, fresh_engine, name, shift, rows, nsb, m):
    import torch
    ty, cols = le.MV_TYPES[name], 256 * nsb
    q = wbytes(ty, rows, cols, seed=rows)
    x = acts(m * cols, m).reshape(m, cols)
    at = torch.zeros(q.size + 32, dtype=torch.uint8, device="cuda")
    at[shift:shift + q.size] = dev(q).reshape(-1)
    dw, dx, y = at[shift:shift + q.size], dev(x), torch.full((m, rows), float("nan"), device="cuda")
    assert dw.data_ptr() % 16 == shift
    print("unaligned GEMM", name, shift, rows, cols, m, flush=True)
    for cfg in (0, 21, 22) if m > 32 else (0,):
        fresh_engine.set_option("gq_cfg", cfg)
        y.fill_(float("nan"))
        fresh_engine.gemm(ty, dw, dx, m, y, rows, cols)
        pick = np.unique(np.r_[0:8, rows - 8:rows])
        sel = np.ascontiguousarray(q.reshape(rows, -1)[pick])
        check_close(y.cpu().numpy()[:, pick], oracle.matmat(ty, sel, len(pick), cols, x), absmag(ty, sel, len(pick), cols, x))


@pytest.mark.parametrize("name", ["Q4_K", "Q5_K"])
@pytest.mark.parametrize("counts", [(20, 70, 0, 45), (150, 3, 200, 64), (3, 1, 0, 2)])  # tiles of 64, 128 and few pairs
def test_grouped_unaligned_tables(engine, name, counts):
    import torch
    ty, rows, cols, nslot = le.MV_TYPES[name], 600, 768, len(counts)
    q = wbytes(ty, nslot * rows, cols, seed=70).reshape(nslot, -1)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    npair = int(off[-1])
    x, perm = acts(npair * cols, 9).reshape(npair, cols), np.random.default_rng(1).permutation(npair).astype(np.int32)
    dx, idx = dev(x), dev(perm)
    rb = q.shape[1] + 64
    outs = []
    for shifts in ((0, 0, 0, 0), (2, 0, 8, 6)):
        arena = torch.zeros(nslot * rb, dtype=torch.uint8, device="cuda")
        for s, sh in enumerate(shifts):
            arena[s * rb + sh:s * rb + sh + q.shape[1]] = dev(q[s])
        ptrs = dev(np.array([arena.data_ptr() + s * rb + sh for s, sh in enumerate(shifts)], dtype=np.uint64))
        y = torch.full((npair, rows), float("nan"), device="cuda")
        print("unaligned tables", name, counts, shifts, flush=True)
        engine.mm_grouped(ty, dev(off), idx, idx, nslot, npair, dx, y, rows, cols, ptrs=ptrs)
        outs.append(y.cpu().numpy())
    # the same codes and activations in both kernels, fp32 sums in another order: 2^-24 for each of K / 16 + K / 256 additions
    for s in range(nslot):
        p = perm[off[s]:off[s + 1]]
        mag = absmag(ty, q[s], rows, cols, x[p])
        assert np.all(np.abs(outs[0][p] - outs[1][p]) <= 6e-6 * mag)
