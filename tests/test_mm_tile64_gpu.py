"""The 64 x 64 tile kernel (csrc/mm_int4.hip, RK_MM_TILE64) over its block shapes: 1 .. 4 m tiles, 16 / 32 / 64 columns,
eight or four waves, whole and split K, waves without a group, the LDS-staged form, ragged rows and columns; against
the CPU oracle.
Bar: max relative error <= 1e-2 with the per-output floor max(2^-14, 256 u32 sum_k |X_mk w_nk|), cosine >= 0.9999."""
import pytest
import torch

import synth
import _hiplib as H
from oracle import int4 as O

pytestmark = pytest.mark.gpu
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


@pytest.mark.parametrize("M,N,K,xdt,ydt", [
    (49, 70, 128, F16, F32),          # one group: seven waves without one; 16 columns, 4 m tiles, the last with 1 row
    (65, 1001, 640, BF16, BF16),      # 3 m tiles of the last row block partly past M, 5 groups
    (81, 2050, 1920, F16, F16),       # 15 groups: one wave with one group less
    (200, 2040, 2048, BF16, F32),     # 32 columns
    (130, 3100, 1152, F16, F16),      # 64 columns by eight waves, 9 groups
    (150, 3100, 896, BF16, F16),      # 64 columns, fewer groups than eight waves
    (150, 3100, 768, F16, F32),       # the fewest groups the waves share in one round
    (150, 3100, 640, BF16, F32),      # LDS-staged: one round, five groups
    (300, 6000, 384, F16, BF16),      # LDS-staged: more blocks than CUs
    (300, 5701, 1280, BF16, F32),     # LDS-staged: ten groups
    (300, 5701, 1408, F16, F16),      # 64 columns by four waves, the fewest groups (11)
    (300, 3400, 8320, BF16, F32),     # more blocks than CUs, 65 groups: tables too long for two four-wave blocks a CU
    (1, 40, 2176, F16, F32),          # 1 m tile, one row, split
    (20, 130, 6400, BF16, F16),       # 2 m tiles, split into narrow columns, N % 4 != 0
    (40, 2052, 11008, F16, F32),      # 3 m tiles, eight splits of 64 columns
    (5, 40, 50048, F16, F32),         # K beyond one block's scale table: split by the plan
])
def test_tile64_block_shapes(M, N, K, xdt, ydt, dev):
    assert H.mm_plan(M, N, K)[0] == H.MM_TILE64
    X, q, s, m = synth.prefill_case(M, N, K, 90 + M)
    Xw = torch.zeros(M, K + 64, dtype=xdt)  # rows with a stride beyond K
    Xw[:, :K] = X.to(xdt)
    Xd, qd, sd, md = Xw.to(dev), q.to(dev), s.to(dev), m.to(dev)
    L = H.lib()
    nws = L.rk_mm_int4_workspace_bytes(M, N, K)
    ws = torch.full((nws + 64,), 0xFF, device=dev, dtype=torch.uint8)  # stale contents must not matter
    a = (Xw[:, :K].float().numpy(), q.numpy(), s.numpy(), m.numpy())
    ref, floor = O.mm_int4(*a), O.cond_floor(O.mm_int4_abs(*a))
    outs = []
    for entry in ("ws", "noalloc", "plain"):
        Yw = torch.full((M + 1, N + 8), 7.0, device=dev, dtype=ydt)  # one guard row, eight guard columns
        args = [H.ptr(Xd), H.dt(Xd), K + 64, H.ptr(qd), H.ptr(sd), H.ptr(md), H.ptr(Yw), H.dt(Yw), N + 8, M, N, K]
        if entry == "ws":
            H.check(L.rk_mm_int4_g128_ws(*args, H.ptr(ws), nws, H.stream(dev)), entry)
        elif entry == "noalloc":
            H.check(L.rk_mm_int4_g128_noalloc(*args, H.stream(dev)), entry)
        else:
            H.check(L.rk_mm_int4_g128(*args, H.stream(dev)), entry)
        torch.cuda.synchronize()
        rep = O.parity_report(Yw[:M, :N].float().cpu().numpy(), ref, floor)
        assert rep["max_rel"] <= 1e-2 and rep["cosine"] >= 0.9999, (entry, rep)
        assert torch.all(Yw[M] == 7.0) and torch.all(Yw[:, N:] == 7.0), entry
        outs.append(Yw)
    assert torch.equal(outs[0], outs[1])  # the same plan and order of sums
    assert torch.all(ws[nws:] == 0xFF)


@pytest.mark.parametrize("M,N,K,ldx", [
    (2, 70, 82048, 2 ** 25 + 8),           # rows 64 MiB apart, more groups than one block's tables hold
    (3, 40, 2048 + 128, 2 ** 25 + 8),      # the same stride, few groups, split
    (1, 3, 2 ** 25 + 128, 2 ** 25 + 128),  # K itself past the 32-bit row offsets
])
def test_tile64_wide_strides(M, N, K, ldx, dev):
    """X rows or code rows further apart than the 32-bit offsets of the wave-split kernel reach"""
    assert H.mm_plan(M, N, K)[0] == H.MM_TILE64
    g = torch.Generator(device=dev).manual_seed(K)
    X = torch.zeros((M - 1) * ldx + K, device=dev, dtype=F16).as_strided((M, K), (ldx, 1))
    X.copy_(torch.randn(M, K, generator=g, device=dev))
    q = torch.randint(0, 256, (N, K // 2), generator=g, device=dev, dtype=torch.uint8)
    s = (torch.rand(N, K // 128, generator=g, device=dev) * 1.9e-2 + 1e-3).half()
    m = ((torch.randn(N, K // 128, generator=g, device=dev) - 7.5) * s.float()).half()
    ref, mag = torch.zeros(M, N, device=dev, dtype=torch.float64), torch.zeros(M, N, device=dev, dtype=torch.float64)
    step = 1 << 20
    for k in range(0, K, step):
        c = q[:, k // 2:(k + step) // 2]
        w = torch.stack((c & 15, c >> 4), -1).reshape(N, -1, 128).double()
        gs = slice(k // 128, (k + step) // 128)
        w = (w * s[:, gs].double()[..., None] + m[:, gs].double()[..., None]).reshape(N, -1)
        x = X[:, k:k + step].double()
        ref += (x[:, None] * w).sum(-1)
        mag += (x[:, None] * w).abs().sum(-1)
    floor = (256 * 2.0 ** -24 * mag).clamp_min(2.0 ** -14)
    L = H.lib()
    nws = L.rk_mm_int4_workspace_bytes(M, N, K)
    ws = torch.empty(max(nws, 16), device=dev, dtype=torch.uint8)
    for entry in ("ws", "noalloc"):
        Y = torch.full((M, N), 7.0, device=dev, dtype=F32)
        args = [H.ptr(X), H.dt(X), ldx, H.ptr(q), H.ptr(s), H.ptr(m), H.ptr(Y), H.dt(Y), N, M, N, K]
        st = L.rk_mm_int4_g128_ws(*args, H.ptr(ws), nws, H.stream(dev)) if entry == "ws" else \
            L.rk_mm_int4_g128_noalloc(*args, H.stream(dev))
        H.check(st, entry)
        err = ((Y.double() - ref).abs() / torch.maximum(ref.abs(), floor)).max().item()
        assert err <= 1e-2, (entry, err)
