"""prefill_attn (csrc/prefill.hip) where its layouts can go wrong: every share of heads per KV head, tiles of 16
queries and blocks of 32 keys with remainders, past 512 keys, and outputs that lie off an 8-byte boundary."""
import numpy as np
import pytest
import torch

import prefill as PF
from oracle import glue as OG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,p0,NKV,off,qs", [(1, 0, 16, 0, 1), (33, 31, 16, 1, 1), (47, 0, 8, 2, 1), (65, 352, 8, 0, 6),
                                             (31, 1, 2, 3, 1), (417, 0, 2, 0, 6), (17, 367, 4, 1, 1), (17, 368, 4, 2, 1),
                                             (1, 1022, 4, 0, 1), (1023, 1, 4, 0, 6)])
def test_prefill_attn_layouts(T, p0, NKV, off, qs):
    """Against the fp32 oracle: P and the result are rounded to fp16 once each (2^-11 of a value, P's errors averaging
    over the keys), so a row is within 2^-10 of its norm."""
    NH, HD, S = 16, 128, 1024
    g = torch.Generator().manual_seed(T + 7 * p0 + NKV)
    q = (torch.randn(T, NH * HD, generator=g) * qs).half()
    kc, vc = (torch.randn(NKV, S, HD, generator=g).half() for _ in range(2))
    buf = torch.full((T * NH * HD + 8,), 7.0, dtype=torch.float16, device="cuda")
    o = buf[off:off + T * NH * HD].view(T, NH * HD)
    PF.prefill_attn(q.cuda(), kc.cuda(), vc.cuda(), o, T, p0, NH, NKV, HD, S, HD ** -0.5)
    torch.cuda.synchronize()
    ref = OG.causal_attend(q.float().numpy().reshape(T, NH, HD), kc.numpy(), vc.numpy(), p0)
    got = o.float().cpu().numpy().reshape(T, NH, HD)
    ref = ref.reshape(got.shape)
    worst = float((np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)).max())
    assert worst <= 2.0 ** -10, worst
    assert (buf[:off] == 7).all() and (buf[off + T * NH * HD:] == 7).all()
