"""The grouped int8-MFMA product (MUL_MAT_ID of batches and prefill) at the
edges of its tiling: buckets around 16, 32 and 64 pairs, rows off the 16- and
64-row tiles, one to seventeen K blocks, weights that do not start on a dword, and
the pair count from which it is taken.

Bar: 2e-5 of sum_i |w x| per output.  The integer block sums are exact; what is
left is f32 rounding of at most 17 block terms and of the two products each is
the difference of (2^-24 each, the terms up to a few times the sum): below
2e-6 of the bound, and as much in the oracle."""
import numpy as np
import pytest
import torch

import zm_oracle as O
from moe_cases import CONFIGS, IQ2, IQ3, IQ4, Q2, Q3, Q4, Q5, Q6, Built, assert_close_layer, reduced

pytestmark = pytest.mark.gpu

TYPES = [Q2, Q3, Q4, Q5, Q6, IQ2, IQ3, IQ4]
TOL = 2e-5


@pytest.fixture(scope="module", autouse=True)
def _init():
    import zeromoe_amd as Z

    assert torch.cuda.is_available(), "GPU tests need a device"
    Z.init()
    yield


def _place(W, offset):
    """W on the device, starting `offset` bytes past an aligned address."""
    buf = torch.zeros(W.size + 16, dtype=torch.uint8, device="cuda")
    v = buf[offset:offset + W.size].view(W.shape)
    v.copy_(torch.from_numpy(W))
    return v


def _check(t, I, rows, sizes, offset=0, extra=()):
    import zeromoe_amd as Z

    E = len(sizes)
    ids = np.concatenate([np.full(n, e) for e, n in enumerate(sizes)] + [np.array(extra, int)]).astype(np.int32)
    ids = np.random.default_rng(I + rows).permutation(ids).reshape(-1, 1)
    S = len(ids)
    print(f"mmq t={t} I={I} O={rows} sizes={sizes} offset={offset}", flush=True)
    W = O.random_blocks(t, E * rows, I, seed=t + I).reshape(E, rows, -1)
    x = np.random.default_rng(S).standard_normal((S, 1, I)).astype(np.float32)
    out = torch.full((S, 1, rows), 7.0, device="cuda")
    Z.mul_mat_id(_place(W, offset), t, I, torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda(), out=out)
    got = out.cpu().numpy()[:, 0]
    ok = (ids[:, 0] >= 0) & (ids[:, 0] < E)
    assert not got[ids[:, 0] < 0].any() and np.isnan(got[ids[:, 0] >= E]).all()
    ref = O.mul_mat_id(t, W, x, np.where(ok[:, None], ids, 0).astype(np.int32), nthreads=8)[:, 0]
    for e in range(E):
        m = ok & (ids[:, 0] == e)
        if m.any():
            bound = O.f32_matmul_absbound(t, W[e], x[m, 0])
            err = np.abs(got[m].astype(np.float64) - ref[m])
            assert (err <= TOL * bound + 1e-30).all(), (e, float((err / (bound + 1e-30)).max()))


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("I,rows", [(256, 16), (512, 37), (768, 130), (1280, 64), (1792, 1)])
def test_bucket_and_row_edges(t, I, rows):
    _check(t, I, rows, [1, 15, 16, 17, 31, 32, 33, 0, 2])                      # 32-pair items
    _check(t, I, rows, [1, 0, 2, 15, 16, 3, 17, 7, 5, 9, 6], extra=(-1, 11))      # 16-pair items
    _check(t, I, rows, [1, 16, 33, 47, 48, 49, 63, 64, 65, 129], extra=(-1, 10, 99))  # 64-pair items


@pytest.mark.parametrize("tiles", ["1", "2", "4"])
@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("I,rows", [(256, 16), (512, 37), (2304, 130), (4352, 50)])
def test_every_item_size(t, I, rows, tiles, monkeypatch):
    """The same edges with items of 16, 32 and 64 pairs whatever the rule takes
    for these few rows; 9 and 17 K blocks: odd, and one past the runs of 8."""
    monkeypatch.setenv("ZEROMOE_MMQ_TILES", tiles)
    _check(t, I, rows, [1, 15, 16, 17, 31, 32, 33, 0, 47, 48, 49, 63, 64, 65, 129], extra=(-1, 15, 99))


@pytest.mark.parametrize("tiles", ["1", "2", "4"])
@pytest.mark.parametrize("t", [Q4, Q3, Q6, IQ2, IQ3, IQ4])
@pytest.mark.parametrize("offset", [2, 4, 6])
def test_every_item_size_off_a_dword(t, offset, tiles, monkeypatch):
    monkeypatch.setenv("ZEROMOE_MMQ_TILES", tiles)
    _check(t, 2304, 33, [20, 5, 55, 1], offset=offset)


def _is_mfma(t, I, rows, sizes, monkeypatch):
    """Whether the call with these bucket sizes ran on another kernel than the GEMV:
    the two add the K blocks in another order."""
    import zeromoe_amd as Z

    E = len(sizes)
    ids = torch.from_numpy(np.repeat(np.arange(E, dtype=np.int32), sizes).reshape(-1, 1)).cuda()
    W = torch.from_numpy(O.random_blocks(t, E * rows, I, seed=t).reshape(E, rows, -1)).cuda()
    x = torch.randn((len(ids), 1, I), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    got = Z.mul_mat_id(W, t, I, x, ids)
    with monkeypatch.context() as m:
        m.setenv("ZEROMOE_MMQ", "0")
        return not torch.equal(got, Z.mul_mat_id(W, t, I, x, ids))


@pytest.mark.parametrize("t,I,rows,least", [(Q3, 1024, 512, 64), (Q6, 1024, 512, 64), (IQ3, 1024, 512, 80),
                                            (IQ2, 1024, 512, 80), (IQ4, 1024, 512, 64), (Q3, 2560, 1000, 40),
                                            (IQ3, 2560, 1000, 40)])
def test_pairs_spread_over_experts(t, I, rows, least, monkeypatch):
    """From `least` pairs on, one or two per expert."""
    n = least // 2 if least > 40 else 39
    below, at = ([2] * (n - 1) + [1], [2] * n) if least > 40 else ([1] * 39, [1] * 40)
    assert sum(below) == least - 1 and sum(at) == least
    assert not _is_mfma(t, I, rows, below, monkeypatch)
    assert _is_mfma(t, I, rows, at, monkeypatch)


@pytest.mark.parametrize("t,below,sizes", [
    (Q4, [15], [16]), (Q4, [7, 16], [8, 16]), (Q6, [4] * 5, [4] * 6), (Q3, [23], [32]),
    (Q2, [2] * 7, [2] * 8), (Q2, [15], [16]), (IQ4, [23], [24]), (IQ3, [7] * 4, [8] * 4), (IQ2, [4] * 15, [4] * 16),
])
def test_pairs_of_few_experts(t, below, sizes, monkeypatch):
    """Several pairs per expert take the MFMA kernel at fewer pairs in all."""
    if t != Q3:
        assert not _is_mfma(t, 1024, 512, below, monkeypatch)
    assert _is_mfma(t, 1024, 512, sizes, monkeypatch)
    _check(t, 1024, 512, sizes)


@pytest.mark.parametrize("t", [Q4, Q3, Q6, IQ2, IQ3, IQ4])
@pytest.mark.parametrize("offset", [1, 2, 3, 4, 6])
def test_weights_off_a_dword(t, offset):
    """Odd row counts of 110-, 210-, 66- and 98-byte blocks put experts and rows
    on either half of a dword; other alignments take the GEMV."""
    _check(t, 768, 33, [20, 5, 55, 1], offset=offset)


@pytest.mark.parametrize("t,I,rows,least", [(Q3, 512, 48, 64), (IQ3, 512, 48, 80), (Q3, 2560, 1000, 40)])
def test_smallest_pair_count(t, I, rows, least):
    for pairs in (least - 1, least, least + 1):
        _check(t, I, rows, [pairs - 3, 2, 1])


@pytest.mark.parametrize("tg,off_g,off_u", [(Q3, 0, 2), (Q3, 2, 2), (Q4, 0, 4), (Q4, 2, 0), (IQ2, 2, 0)])
def test_gate_and_up_on_different_halves(tg, off_g, off_u):
    """The layer with gate and up weights shifted against each other: bit-equal
    where the same kernel runs, else within 1e-4 of the token's largest output
    but for re-quantization ties, which either kernel may round its own way."""
    c = reduced(CONFIGS["c3"], tg=tg, td=Q4, S=48, H=512, F=256, E=8)
    b = Built(c, seed=3)
    x, lg = torch.from_numpy(b.x).cuda(), torch.from_numpy(b.logits).cuda()
    ref, ids, w = (v.cpu().numpy() for v in b.layer().forward(x, lg))
    b.wg = _place(b.wg.cpu().numpy(), off_g)
    b.wu = _place(b.wu.cpu().numpy(), off_u)
    out = b.layer().forward(x, lg)[0].cpu().numpy()
    if off_g % 4 == off_u % 4 and off_g % (2 if tg != Q4 else 4) == 0:
        np.testing.assert_array_equal(out, ref)
    else:
        assert_close_layer(out, ref, rtol=1e-4, slack=lambda: 2 * b.requant_slack(ids, w))


@pytest.mark.parametrize("S,n_ids", [(600_001, 1), (1 << 20, 16)])
def test_bucket_of_more_than_half_a_million_pairs(S, n_ids):
    """All pairs of a long call in one bucket, up to the most the op takes
    (2^24): every part of the result is bit for bit that of a call on these
    tokens alone (a pair's sums do not depend on its place in the bucket)."""
    import zeromoe_amd as Z

    I, rows = 256, 16
    W = torch.from_numpy(O.random_blocks(Q4, 2 * rows, I, seed=5).reshape(2, rows, -1)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(S)
    x = torch.randn((S, 1, I), device="cuda", generator=gen)
    ids = torch.ones((S, n_ids), dtype=torch.int32, device="cuda")
    out = Z.mul_mat_id(W, Q4, I, x, ids)
    first = (1 << 19) // n_ids  # the token of pair 2^19
    for a, b in [(0, 512), (first - 256, first + 256), (S // 2, S // 2 + 512), (S - 512, S)]:
        part = Z.mul_mat_id(W, Q4, I, x[a:b].contiguous(), ids[a:b].contiguous())
        assert torch.equal(out[a:b], part), (a, b)


def test_matrix_of_eight_million_rows():
    """Row tiles times work items past the 2^32 threads of one grid (nearly all
    of the 128 experts without pairs, their weights never touched): the product
    goes out in several launches, bit for bit what slices of the rows give."""
    import zeromoe_amd as Z

    E, rows, S, I = 128, 7_900_001, 128, 256
    if torch.cuda.mem_get_info()[0] < 90 << 30:
        pytest.skip("needs 71 GB of weights and outputs")
    W = torch.empty((E, rows, 66), dtype=torch.uint8, device="cuda")
    part = torch.from_numpy(O.random_blocks(IQ2, 99_991, I, seed=9)).cuda()
    for e in (3, 100):
        for a in range(0, rows, len(part)):
            W[e, a:a + len(part)] = part[:rows - a].roll(e, 0)[:rows - a]
    x = torch.randn((S, 1, I), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    ids = torch.where(torch.arange(S) % 2 == 0, 3, 100).to(torch.int32).view(S, 1).cuda()
    out = Z.mul_mat_id(W, IQ2, I, x, ids)
    for a in (0, 1_234_567, 4_194_303, rows - 2000):
        assert torch.equal(out[:, :, a:a + 2000], Z.mul_mat_id(W[:, a:a + 2000], IQ2, I, x, ids)), a
    # no part of the whole was left out
    assert out.isfinite().all() and (out != 0).float().mean() > 0.99
    del W, out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("over", ["src1", "ids"])
@pytest.mark.parametrize("S,n_ids", [(5, 4), (150, 4)])
def test_result_lying_over_an_input(over, S, n_ids):
    """dst over src1 (a few rows further on) or over the ids, with skipped
    routes: src1 and the ids are taken in before any row is written."""
    import zeromoe_amd as Z

    I = rows = 512
    W = torch.from_numpy(O.random_blocks(Q4, 6 * rows, I, seed=2).reshape(6, rows, -1)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(S)
    x = torch.randn((S, n_ids, I), device="cuda", generator=gen)
    ids = torch.randint(-1, 7, (S, n_ids), dtype=torch.int32, device="cuda", generator=gen)
    ref = Z.mul_mat_id(W, Q4, I, x, ids)
    buf = torch.empty(2 * x.numel(), device="cuda")
    for shift in (0, 3 * I, 16 * I):  # dst so many floats after the input, or over the start of the ids
        for _ in range(3):
            xs, ids_ = x, ids
            if over == "src1":
                xs = buf[:x.numel()].view(x.shape).copy_(x)
            else:
                ids_ = buf[shift:shift + ids.numel()].view(torch.int32).view(ids.shape).copy_(ids)
            out = buf[shift if over == "src1" else 0:][:x.numel()].view(ref.shape)
            Z.mul_mat_id(W, Q4, I, xs, ids_, out=out)
            assert torch.equal(out.nan_to_num(7.0), ref.nan_to_num(7.0)), shift


def test_records_past_two_gibibytes(monkeypatch):
    """Records of src1 beyond 2^31 bytes (Q8_K rows of these tokens are not):
    bit for bit the same kernel's results for a few of the tokens, which are
    not bit for bit the GEMV's."""
    import zeromoe_amd as Z

    S, I, rows = 114_000, 16384, 32
    assert S * (I // 256) * 292 < 1 << 31 < S * (I // 256) * 304
    W = torch.from_numpy(O.random_blocks(Q6, 2 * rows, I, seed=4).reshape(2, rows, -1)).cuda()
    x = torch.randn((S, 1, I), device="cuda", generator=torch.Generator(device="cuda").manual_seed(2))
    ids = (torch.arange(S, device="cuda") % 2).to(torch.int32).view(S, 1)
    out = Z.mul_mat_id(W, Q6, I, x, ids)
    for a in (0, S // 2, S - 20_000):  # enough tokens for items of the same size
        part = Z.mul_mat_id(W, Q6, I, x[a:a + 20_000], ids[a:a + 20_000])
        assert torch.equal(out[a:a + 20_000], part), a
    monkeypatch.setenv("ZEROMOE_MMQ", "0")
    assert not torch.equal(out[-256:], Z.mul_mat_id(W, Q6, I, x[-256:], ids[-256:]))
    del x, out
    torch.cuda.empty_cache()


def _forward(b, monkeypatch=None):
    """The layer's output, ids and weights; with monkeypatch, on the GEMV."""
    L = b.layer()
    x = torch.from_numpy(b.x).cuda()
    lg = None if b.c.router_gemv else torch.from_numpy(b.logits).cuda()
    if monkeypatch is None:
        return [v.cpu().numpy() for v in L.forward(x, lg)]
    with monkeypatch.context() as m:
        m.setenv("ZEROMOE_MMQ", "0")
        return [v.cpu().numpy() for v in L.forward(x, lg)]


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("S,tiles", [(32, None), (160, None), (160, "1"), (160, "4")])
def test_layer_of_every_type(t, S, tiles, monkeypatch):
    """Gate and up together, at 4 and 20 pairs per expert (items of 16 and 32
    pairs by the rule) and 9 blocks of K, against the oracle."""
    if tiles:
        monkeypatch.setenv("ZEROMOE_MMQ_TILES", tiles)
    b = Built(reduced(CONFIGS["c3"], tg=t, td=Q4, S=S, H=2304, F=512, E=32, K=4, logit_bias_sd=0.0), seed=S)
    out, ids, w = _forward(b)
    assert not np.array_equal(out, _forward(b, monkeypatch)[0]), "not on the MFMA kernel"
    assert_close_layer(out, b.oracle_forward(ids, w), slack=lambda: b.requant_slack(ids, w))


@pytest.mark.parametrize("off_gu,off_d", [(1, 0), (0, 1)])
def test_list_for_one_of_two_products(off_gu, off_d, monkeypatch):
    """One work list serves gate/up and down; here only one of them runs on the
    MFMA kernel (weights off their alignment take the GEMV)."""
    b = Built(reduced(CONFIGS["c3"], tg=Q4, td=Q6, S=96, H=1024, F=512, E=16), seed=8)
    ref, ids, w = _forward(b)
    gemv = _forward(b, monkeypatch)[0]
    b.wg, b.wu = _place(b.wg.cpu().numpy(), off_gu), _place(b.wu.cpu().numpy(), off_gu)
    b.wd = _place(b.wd.cpu().numpy(), off_d)
    out = _forward(b)[0]
    assert not np.array_equal(out, ref) and not np.array_equal(out, gemv)
    for r in (ref, gemv):
        assert_close_layer(out, r, rtol=1e-4, slack=lambda: 2 * b.requant_slack(ids, w))


def _tie_slack(b, ids, w):
    """Per token, what re-quantization ties can change: those of the routed act
    rows (Built.requant_slack) and, counted the same way, of the shared expert's."""
    c, tie = b.c, 2e-4
    x, one = b.x[:, None, :], np.zeros((c.S, 1), np.int32)
    g, u = (O.mul_mat_id(c.t_shared, v.cpu().numpy()[None], x, one, nthreads=8) for v in (b.sg, b.su))
    act = O.swiglu(g, u).reshape(c.S, c.F_shared // 256, 256).astype(np.float64)
    d = np.abs(act).max(-1, keepdims=True) / 127.0
    v = act / np.where(d > 0, d, 1.0)
    tied = np.abs(np.abs(v - np.floor(v)) - 0.5) < tie
    cols = np.abs(O.dequantize(c.t_shared, b.sd.cpu().numpy(), c.F_shared)).max(0).reshape(1, -1, 256)
    return b.requant_slack(ids, w, tie) + (tied * d * cols).sum(axis=(1, 2))


@pytest.mark.parametrize("ts", TYPES)
@pytest.mark.parametrize("S", [8, 17, 64])
def test_shared_expert_of_every_type(ts, S, monkeypatch):
    """Few tokens through a dense shared expert (one-wave workgroups), against
    the oracle."""
    monkeypatch.setenv("ZEROMOE_FUSED_DECODE", "0")
    b = Built(reduced(CONFIGS["c5"], S=S, H=1280, F=512, F_shared=768, t_shared=ts, router_gemv=False), seed=S)
    out, ids, w = _forward(b)
    assert not np.array_equal(out, _forward(b, monkeypatch)[0]), "not on the MFMA kernel"
    assert_close_layer(out, b.oracle_forward(ids, w), rtol=1e-4, slack=lambda: _tie_slack(b, ids, w))


@pytest.mark.parametrize("ts", [Q4, Q6, IQ2])
@pytest.mark.parametrize("S", [256, 1024])
def test_shared_expert_of_many_tokens(ts, S, monkeypatch):
    """Enough tokens for workgroups of several waves, items of 16 to 64 pairs,
    against the GEMV (ties of either path)."""
    b = Built(reduced(CONFIGS["c5"], S=S, H=2048, F=256, E=8, n_slots=4, K=1, groups=0, groups_used=0,
                      F_shared=2048, t_shared=ts, router_gemv=False), seed=S)
    out, ids, w = _forward(b)
    gemv = _forward(b, monkeypatch)[0]
    assert not np.array_equal(out, gemv), "not on the MFMA kernel"
    assert_close_layer(out, gemv, rtol=1e-4, slack=lambda: 2 * _tie_slack(b, ids, w))


@pytest.mark.parametrize("t", [Q3, Q4])
@pytest.mark.parametrize("S,ne11", [(3, 4), (60, 1), (60, 4)])
@pytest.mark.parametrize("layout", ["token", "row", "ids", "out", "all", "one_token"])
def test_strided_tensors(t, S, ne11, layout):
    """src1 with padded tokens or rows (or one token for all), ids and dst with
    padded rows: bit for bit the result of dense tensors."""
    import zeromoe_amd as Z

    I, rows, E, n_ids = 768, 40, 6, 4
    gen = torch.Generator(device="cuda").manual_seed(S)
    W = torch.from_numpy(O.random_blocks(t, E * rows, I, seed=1).reshape(E, rows, -1)).cuda()
    x = torch.randn((S, ne11, I), device="cuda", generator=gen)
    ids = torch.randint(-1, E + 1, (S, n_ids), dtype=torch.int32, device="cuda", generator=gen)
    if layout == "one_token":
        x = x[:1].expand(S, ne11, I)
    ref = Z.mul_mat_id(W, t, I, x.contiguous(), ids)
    wide = lambda v, *shape: torch.full(shape, 3, dtype=v.dtype, device="cuda")  # noqa: E731
    out = torch.empty_like(ref)
    if layout in ("token", "all"):
        x = wide(x, S, ne11 + 2, I)[:, :ne11].copy_(x)
    if layout in ("row", "all"):
        x = wide(x, S, ne11, I + 64)[:, :, :I].copy_(x)
    if layout in ("ids", "all"):
        ids = wide(ids, S, n_ids + 3)[:, :n_ids].copy_(ids)
    whole = wide(ref, S, n_ids + 1, rows + 8)
    if layout in ("out", "all"):
        out = whole[:, :n_ids, :rows]
    Z.mul_mat_id(W, t, I, x, ids, out=out)
    assert torch.equal(out.nan_to_num(7.0), ref.nan_to_num(7.0))
    if layout in ("out", "all"):
        assert (whole[:, n_ids:] == 3).all() and (whole[:, :, rows:] == 3).all()
