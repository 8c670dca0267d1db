"""The wide-wave prepared-X kernel (csrc/mm_int4.hip, RK_MM_WIDE128) over its block shapes: 3 or 4 tiles of 32 rows, one
or two K ways, whole and split K, odd step counts, ragged rows and columns; against the CPU oracle.
Bar: max relative error <= 1e-2 with the per-output floor max(2^-14, 256 u32 sum_k |X_mk w_nk|), cosine >= 0.9999."""
import pytest
import torch

import synth
import _hiplib as H
from oracle import int4 as O

pytestmark = pytest.mark.gpu
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


@pytest.mark.parametrize("M,N,K,xdt,ydt", [
    (65, 17409, 512, F16, F32),      # 3 row tiles (the last half absent), two K ways of 2 steps, one column in a block
    (96, 17500, 768, BF16, BF16),    # two K ways of 3 steps
    (97, 17420, 1280, F16, F16),     # 4 row tiles with 15 of the last 31 rows absent, two K ways of 5 steps
    (129, 9000, 1024, BF16, F32),    # two row blocks of 3 tiles
    (131, 17401, 768, BF16, BF16),   # odd N: rows of Y off the 16-byte pieces, one K way
    (170, 17000, 512, F16, BF16),    # more blocks than CUs: one K way, 3 row tiles, the fewest groups (4)
    (250, 1030, 8448, BF16, F16),    # split over K, two K ways of 2 and 3 steps
    (260, 2048, 4608, BF16, F16),    # split, row blocks of 3 tiles, two K ways of 3 and 4 steps
    (250, 1030, 11008, F16, F32),    # split, N % 4 != 0 (the scalar sum over splits)
    (300, 5000, 3328, F16, F16),     # split, one K way
])
def test_wide_kernel_block_shapes(M, N, K, xdt, ydt, dev):
    kernel, splits = H.mm_plan(M, N, K)
    assert kernel == H.MM_WIDE128 and (splits > 1) == (K > 2048)
    X, q, s, m = synth.prefill_case(M, N, K, 70 + M)
    Xw = torch.zeros(M, K + 64, dtype=xdt)  # rows with a stride beyond K
    Xw[:, :K] = X.to(xdt)
    Xd, qd, sd, md = Xw.to(dev), q.to(dev), s.to(dev), m.to(dev)
    nws = H.lib().rk_mm_int4_workspace_bytes(M, N, K)
    ws = torch.full((nws + 64,), 0xFF, device=dev, dtype=torch.uint8)  # stale contents must not matter
    Yw = torch.full((M + 1, N + 8), 7.0, device=dev, dtype=ydt)       # one guard row, eight guard columns
    for _ in range(2):
        H.check(H.lib().rk_mm_int4_g128_ws(H.ptr(Xd), H.dt(Xd), K + 64, H.ptr(qd), H.ptr(sd), H.ptr(md), H.ptr(Yw),
                                           H.dt(Yw), N + 8, M, N, K, H.ptr(ws), nws, H.stream(dev)), "mm_int4")
        torch.cuda.synchronize()
    a = (Xw[:, :K].float().numpy(), q.numpy(), s.numpy(), m.numpy())
    rep = O.parity_report(Yw[:M, :N].float().cpu().numpy(), O.mm_int4(*a), O.cond_floor(O.mm_int4_abs(*a)))
    assert rep["max_rel"] <= 1e-2 and rep["cosine"] >= 0.9999, rep
    assert torch.all(Yw[M] == 7.0) and torch.all(Yw[:, N:] == 7.0)
    assert torch.all(ws[nws:] == 0xFF)
