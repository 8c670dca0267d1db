"""Rounding of the int4 prefill product (csrc/mm_int4.hip), fp32 outputs against 64 bits: a kernel that adds the groups'
min terms apart from their scaled products must be no further off than the group-by-group order of the reference
(kernels/mm_int4.py:24-46: acc += scale * dot + min * rowsum, all fp32), also for activations with a mean, where the
two sums cancel."""
import numpy as np
import pytest
import torch

import synth
import _hiplib as H
from oracle import int4 as O

pytestmark = pytest.mark.gpu


def _group_by_group(X, q, s, m):
    """the reference's order: dot and rowsum rounded to fp32 once per group, then two fused multiply-adds"""
    codes = O.unpack_int4(q).astype(np.float64)
    s, m = s.astype(np.float64), m.astype(np.float64)
    acc = np.zeros((X.shape[0], q.shape[0]))
    f32 = lambda a: a.astype(np.float32).astype(np.float64)  # noqa: E731
    for g in range(s.shape[1]):
        x = X[:, 128 * g:128 * g + 128].astype(np.float64)
        dot, xs = f32(x @ codes[:, 128 * g:128 * g + 128].T), f32(x.sum(1, keepdims=True))
        acc = f32(dot * s[:, g] + f32(xs * m[:, g] + acc))
    return acc


@pytest.mark.parametrize("M,N,K,kernel", [
    (69, 2048, 2048, H.MM_TILE64),    # 16 columns per block, eight waves
    (34, 1030, 11008, H.MM_TILE64),   # split over K
    (512, 3072, 2048, H.MM_TILE64),   # 64 columns, four waves
    (80, 17500, 2048, H.MM_WIDE128),  # two K ways
    (512, 22016, 1024, H.MM_WIDE128),  # one K way
    (300, 2048, 11008, H.MM_WIDE128),  # split over K
])
@pytest.mark.parametrize("mean", [0.0, 1.0, 8.0])
def test_no_further_off_than_group_by_group(M, N, K, kernel, mean, dev):
    assert H.mm_plan(M, N, K)[0] == kernel
    X, q, s, m = synth.prefill_case(M, N, K, 5)
    X = (X.float() + mean).half()
    Xd, qd, sd, md = (t.to(dev) for t in (X, q, s, m))
    Y = torch.empty(M, N, device=dev, dtype=torch.float32)
    nws = H.lib().rk_mm_int4_workspace_bytes(M, N, K)
    ws = torch.empty(max(nws, 16), device=dev, dtype=torch.uint8)
    H.check(H.lib().rk_mm_int4_g128_ws(H.ptr(Xd), H.dt(Xd), K, H.ptr(qd), H.ptr(sd), H.ptr(md), H.ptr(Y), H.dt(Y), N, M,
                                       N, K, H.ptr(ws), nws, H.stream(dev)), "mm_int4")
    rows = np.unique(np.linspace(0, M - 1, 48).astype(int))  # rows across every row block
    cols = np.unique(np.linspace(0, N - 1, 512).astype(int))
    a = (X.numpy()[rows], q.numpy()[cols], s.numpy()[cols], m.numpy()[cols])
    ref = O.mm_int4_f64(*a)
    off = lambda y: np.linalg.norm(y - ref) / np.linalg.norm(ref)  # noqa: E731
    got = off(Y.cpu().numpy()[np.ix_(rows, cols)].astype(np.float64))
    assert got <= off(_group_by_group(*a)), got
