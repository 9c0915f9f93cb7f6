"""The workspace sizes with which MUL_MAT_ID shapes are accepted, and that an
accepted workspace is never written past its end."""
import ctypes as C

import numpy as np
import pytest
import torch

import zm_oracle as O
from moe_cases import IQ3, Q3, Q4, Q6
from zeromoe_amd._lib import ZmTensor, lib

STATIC = 16 << 20


def _up(n):
    return (n + 255) // 256 * 256


def least(I, E, S, n_ids, ne11):
    """Q8_K rows, a copy of the ids, the bucket arrays and a list of 32-pair items."""
    row, pairs = (I // 256 * 292 + 15) // 16 * 16, S * n_ids
    arrays = [S * ne11 * row, pairs * 4, E * 4, (E + 1) * 4, pairs * 4, E * 4, 4,
              ((pairs + 31) // 32 + min(pairs, E)) * 4]
    return sum(_up(a) for a in arrays) + 4 + 256


def _descs(t, I, O_, E, S, n_ids, ne11, data=(0, 0, 0, 0)):
    row = I // 256 * O.BLOCK_BYTES[t]

    def tensor(type_, ne, nb, p):
        T = ZmTensor()
        T.type, T.data = type_, p
        for i in range(4):
            T.ne[i], T.nb[i] = (*ne, 1)[i], (*nb, nb[2] * ne[2])[i]
        return T

    return [tensor(t, (I, O_, E), (O.BLOCK_BYTES[t], row, row * O_), data[0]),
            tensor(0, (I, ne11, S), (4, 4 * I, 4 * I * ne11), data[1]),
            tensor(26, (n_ids, S, 1), (4, 4 * n_ids, 4 * n_ids * S), data[2]),
            tensor(0, (O_, n_ids, S), (4, 4 * O_, 4 * O_ * n_ids), data[3])]


@pytest.mark.parametrize("t,I,E,n_ids,ne11", [(Q4, 4096, 128, 8, 1), (Q3, 2048, 8, 8, 8), (IQ3, 256, 512, 2, 1),
                                              (Q6, 16384, 4, 6, 1), (Q4, 1024, 60, 64, 1)])
def test_static_scratch_accepts_up_to_its_size(t, I, E, n_ids, ne11):
    """The largest token count that the fixed scratch array is accepted for."""
    L = lib()

    def ok(S):
        d = _descs(t, I, 64, E, S, n_ids, ne11)
        return L.zm_mul_mat_id_static(*[C.byref(v) for v in d], None, 0) == 1

    S = next(s for s in range(1, 1 << 16) if least(I, E, s + 1, n_ids, ne11) > STATIC)
    assert ok(S) and not ok(S + 1)
    for s in (1, 2, 7, S // 2):
        d = _descs(t, I, 64, E, s, n_ids, ne11)
        assert L.zm_mul_mat_id_workspace_size(*[C.byref(v) for v in d]) >= least(I, E, s, n_ids, ne11)
        assert ok(s)


@pytest.mark.gpu
@pytest.mark.parametrize("t,I,rows,E,S,n_ids,ne11", [
    (Q4, 4096, 64, 8, 401, 8, 1),   # records for half the tokens at a time
    (Q6, 1024, 48, 4, 300, 2, 2),
    (IQ3, 512, 32, 5, 77, 4, 1),
    (Q3, 1024, 64, 3, 1, 100, 1),   # one token: no half, planar rows
    (Q4, 2048, 64, 8, 2, 4, 4),     # planar rows anyway
])
def test_least_workspace_is_enough(t, I, rows, E, S, n_ids, ne11):
    """A bound workspace of the accepted size: the result is the one that a
    workspace of the asked-for size gives (up to the order of f32 sums where
    another kernel runs), and the bytes after it stay as they were."""
    import zeromoe_amd as Z

    Z.init()
    L = lib()
    rng = np.random.default_rng(S)
    W = torch.from_numpy(O.random_blocks(t, E * rows, I, seed=S).reshape(E, rows, -1)).cuda()
    x = torch.from_numpy(rng.standard_normal((S, ne11, I)).astype(np.float32)).cuda()
    ids = torch.from_numpy(rng.integers(-1, E, (S, n_ids)).astype(np.int32)).cuda()
    ref = Z.mul_mat_id(W, t, I, x, ids)
    n = least(I, E, S, n_ids, ne11)
    buf = torch.full((n + (1 << 16),), 0xA5, dtype=torch.uint8, device="cuda")
    y = torch.full_like(ref, float("nan"))
    d = [C.byref(v) for v in _descs(t, I, rows, E, S, n_ids, ne11,
                                    [v.data_ptr() for v in (W, x, ids, y)])]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    count = L.zm_mul_mat_id_launches()
    try:
        assert L.zm_mul_mat_id_set_workspace(s.cuda_stream, buf.data_ptr(), n - 1) == 0
        assert L.zm_mul_mat_id(*d, s.cuda_stream, 1) == 0
        assert L.zm_mul_mat_id_set_workspace(s.cuda_stream, buf.data_ptr(), n) == 0
        assert L.zm_mul_mat_id(*d, s.cuda_stream, 1) == 1, L.zm_last_error()
        torch.cuda.synchronize()
    finally:
        L.zm_mul_mat_id_set_workspace(s.cuda_stream, None, 0)
    assert (buf[n:] == 0xA5).all()
    assert L.zm_mul_mat_id_launches() == count + 1
    # f32 rounding of I / 256 block terms in another order (2^-24 each, against
    # the bound sum |w x| of about 10 times the result's scale)
    scale = ref.abs().max()
    assert (y - ref).abs().max() <= 2e-5 * scale
    assert not y[ids < 0].any()


@pytest.mark.gpu
def test_static_scratch_at_its_limit():
    """The longest call that the scratch array takes (its records would not fit
    it at once) against the bound workspace."""
    import zeromoe_amd as Z

    Z.init()
    L = lib()
    t, I, rows, E, n_ids = Q4, 4096, 256, 8, 8
    S = next(s for s in range(1, 1 << 16) if least(I, E, s + 1, n_ids, 1) > STATIC)
    W = torch.from_numpy(O.random_blocks(t, E * rows, I, seed=1).reshape(E, rows, -1)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((S, 1, I), device="cuda", generator=gen)
    ids = torch.randint(-1, E, (S, n_ids), dtype=torch.int32, device="cuda", generator=gen)
    ref = Z.mul_mat_id(W, t, I, x, ids)
    y = torch.full_like(ref, float("nan"))
    d = [C.byref(v) for v in _descs(t, I, rows, E, S, n_ids, 1, [v.data_ptr() for v in (W, x, ids, y)])]
    assert L.zm_mul_mat_id_workspace_size(*d) > STATIC
    assert L.zm_mul_mat_id_static(*d, torch.cuda.current_stream().cuda_stream, 1) == 1, L.zm_last_error()
    assert torch.equal(y, ref)  # the same kernel on halves: a pair's sums do not depend on its place
