"""Decode attention at the edges of its launch shapes: every heads-per-KV-head count, split lengths around the 16 slots
a block has in flight, more splits than the combine's first pass holds, pointers without 16-byte alignment, head dims
that are no multiple of four."""
import numpy as np
import pytest
import torch

import fused
from oracle import glue as OG

pytestmark = pytest.mark.gpu
HD = 128


def _off(t, dev, shift):
    """t on the device, `shift` elements past an aligned address"""
    buf = torch.empty(t.numel() + shift, dtype=t.dtype, device=dev)
    buf[shift:] = t.reshape(-1).to(dev)
    return buf[shift:].view(t.shape)


@pytest.mark.parametrize("nkv", [2, 4, 8, 16])
@pytest.mark.parametrize("pos,nsplit", [(0, 64), (14, 1), (15, 1), (16, 1), (1023, 64), (1024, 64), (299, 100),
                                        (255, 7)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])
def test_split_and_combine(nkv, pos, nsplit, dt, shift, dev):
    NH, S = 16, 1100
    g = torch.Generator().manual_seed(1000 * pos + nsplit)
    kc, vc = (torch.randn(nkv, S, HD, generator=g).to(dt) for _ in range(2))
    q = torch.randn(NH * HD, generator=g).to(dt)
    kc[:, pos + 1:], vc[:, pos + 1:] = float("nan"), float("nan")  # slots past pos are never used
    po = torch.full((NH, nsplit, HD), float("nan"), device=dev)
    pm, pl = (torch.full((NH, nsplit), float("nan"), device=dev) for _ in range(2))
    out = torch.empty(NH * HD, device=dev, dtype=dt)
    p = torch.tensor([pos], device=dev)
    fused.attn_split[(nkv, nsplit)](_off(q, dev, shift), _off(kc, dev, shift), _off(vc, dev, shift), p, po, pm, pl, S,
                                    HD ** -0.5, REP=NH // nkv, HD=HD, NSPLIT=nsplit)
    fused.attn_combine[(NH,)](po, pm, pl, p, out, HD=HD, NSPLIT=nsplit)
    K, V = kc[:, :pos + 1].float().numpy(), vc[:, :pos + 1].float().numpy()
    ref = OG.attend(q.float().numpy().reshape(NH, HD), K, V)
    ch = (-(-(pos + 1) // nsplit) + 7) // 8 * 8
    racc, rm, rl = OG.attend_split(q.float().numpy().reshape(NH, HD), K, V, nsplit, ch)[0:3]
    # the output is rounded once: half an ulp per value, 2^-11 (fp16) or 2^-8 (bf16) of it
    got = out.float().cpu().numpy().reshape(NH, HD)
    assert np.linalg.norm(got - ref) <= (2 ** -11 if dt == torch.float16 else 2 ** -8) * np.linalg.norm(ref)
    used = np.arange(nsplit) * ch < pos + 1
    m, l = pm.cpu().numpy(), pl.cpu().numpy()
    # fp32 scores of 128 products and sums of at most ch weights: a few hundred ulps at most
    np.testing.assert_allclose(m[:, used], rm[:, used], rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(l[:, used], rl[:, used], rtol=1e-3)
    assert np.all(np.isneginf(m[:, ~used])) and np.all(l[:, ~used] == 0) and np.all(po.cpu().numpy()[:, ~used] == 0)


def test_masked_scores(dev):
    """a score of -inf has weight zero wherever it stands in the split"""
    NH, nkv, S, pos, nsplit = 16, 4, 64, 40, 2
    q = torch.ones(NH * HD, dtype=torch.bfloat16)
    kc = torch.zeros(nkv, S, HD).bfloat16()
    vc = torch.randn(nkv, S, HD, generator=torch.Generator().manual_seed(1)).bfloat16()
    kc[:, 0, 0], kc[:, 17, 0], kc[:, 30, 5] = float("-inf"), float("-inf"), float("-inf")
    po, pm, pl = torch.empty(NH, nsplit, HD, device=dev), *(torch.empty(NH, nsplit, device=dev) for _ in range(2))
    out = torch.empty(NH * HD, device=dev, dtype=torch.bfloat16)
    p = torch.tensor([pos], device=dev)
    fused.attn_split(q.to(dev), kc.to(dev), vc.to(dev), p, po, pm, pl, S, HD ** -0.5, REP=4, HD=HD, NSPLIT=nsplit)
    fused.attn_combine(po, pm, pl, p, out, HD=HD, NSPLIT=nsplit)
    keep = [t for t in range(pos + 1) if t not in (0, 17, 30)]
    ref = vc[:, keep].float().mean(1).repeat_interleave(NH // nkv, 0).numpy()  # the others' scores are all 0
    got = out.float().cpu().numpy().reshape(NH, HD)
    assert np.linalg.norm(got - ref) <= 2 ** -8 * np.linalg.norm(ref)


@pytest.mark.parametrize("hd,nsplit", [(1, 3), (30, 64), (33, 65), (128, 1), (130, 200)])
def test_combine_any_shape(hd, nsplit, dev):
    NH = 5
    g = torch.Generator().manual_seed(hd)
    po, pm, pl = torch.randn(NH, nsplit, hd, generator=g), torch.randn(NH, nsplit, generator=g) * 4, None
    pl = torch.rand(NH, nsplit, generator=g) + 0.5
    pm[:, 1::3] = float("-inf")
    out = torch.empty(NH * hd, device=dev, dtype=torch.float16)
    fused.attn_combine(po.to(dev), pm.to(dev), pl.to(dev), torch.zeros(1, dtype=torch.int64, device=dev), out, HD=hd,
                       NSPLIT=nsplit)
    w = torch.exp(pm.double() - pm.double().amax(1, keepdim=True))
    ref = (w[..., None] * po.double()).sum(1) / (w * pl.double()).sum(1, keepdim=True)
    got = out.double().cpu().reshape(NH, hd)
    # one fp16 rounding plus fp32 sums of nsplit terms that can cancel: 2^-11 of the value, 1e-6 of the terms
    terms = (w[..., None] * po.double().abs()).sum(1) / (w * pl.double()).sum(1, keepdim=True)
    assert bool(((got - ref).abs() <= 2 ** -11 * ref.abs() + 1e-6 * terms + 2 ** -25).all())
