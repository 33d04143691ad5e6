"""The key split of the D = 512 attention with 64 query rows per workgroup:
ragged query blocks, ranges and key tiles, K and V as strided views (rows of
a wider matrix, NaN behind them: bytes of no key reach a result), bitwise the
32-row workgroups' result, and against the oracle."""
import numpy as np
import pytest
import torch

import kd_fa
import kd_oracle as orc
from fa_common import assert_parity, gather_rows, randn, sample_rows

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
D = 512

# B, H, Lq, Lk, K/V type, Q type: each with more 32-row workgroups than CUs
# and at least 17 tenths as many rounds of them as of 64-row ones
CASES = [
    (1, 1, 2100, 2011, torch.bfloat16, torch.float32),
    (1, 1, 4095, 161, torch.float16, torch.float32),
    (2, 3, 1300, 130, torch.float16, torch.float16),
    (1, 2, 2600, 193, torch.bfloat16, torch.bfloat16),
]
# too many 32-row blocks for a split: the unsplit call, ragged in rows and keys
UNSPLIT = (1, 2, 4097, 129, torch.bfloat16, torch.bfloat16)


def _wide(x):
    """x's values as a view into rows with 16 NaN elements behind each."""
    w = torch.full(x.shape[:-1] + (D + 16,), float("nan"), dtype=x.dtype, device=DEV)
    w[..., :D] = x.to(DEV)
    return w[..., :D]


@pytest.mark.parametrize("case", CASES + [UNSPLIT], ids=lambda c: f"B{c[0]}H{c[1]}q{c[2]}k{c[3]}{str(c[4])[-4:]}")
def test_split_64_rows(case):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    B, H, Lq, Lk, kt, qt = case
    print(f"[case] d512 split 64 rows {case}", flush=True)
    q, k, v = randn((B, H, Lq, D), qt, 1), randn((B, H, Lk, D), kt, 2), randn((B, H, Lk, D), kt, 3)
    qd, kd, vd = q.to(DEV), _wide(k), _wide(v)
    outs = [torch.empty((B, Lq, H, D), dtype=torch.float32, device=DEV) for _ in range(2)]
    descs = [kd_fa.make_desc(qd, kd, vd, None, o, D ** -0.5) for o in outs]
    size = kd_fa.workspace_size_full(descs[0])
    assert (size > 0) == (case != UNSPLIT)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV).fill_(0x7F)
    assert kd_fa.run_desc(descs[0], workspace=ws) == kd_fa.OK
    with kd_fa.routing(kd_fa.ROUTE_D512_R1):
        assert kd_fa.run_desc(descs[1], workspace=ws) == kd_fa.OK
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    rows = sample_rows(B, H, Lq, 64, seed=9)
    rows = np.unique(np.concatenate([rows, [0, B * H * Lq - 1]]))
    ref = orc.fa_f64(q, k, v, scale=D ** -0.5, rows=rows)
    assert_parity(gather_rows(outs[0], rows, H, Lq), ref, f"d512 split 64 rows {case}")


@pytest.mark.parametrize("shape", [(1, 256, 32, 256), (4, 64, 31, 520), (2, 128, 17, 130)], ids=lambda s: "x".join(map(str, s)))
def test_many_short_heads_are_not_split(shape):
    """One 64-row workgroup per CU or more: the workspace stays untouched and
    the result is the call's without one."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    B, H, Lq, Lk = shape
    print(f"[case] d512 short heads {shape}", flush=True)
    q, k, v = (randn(s, t, i).to(DEV) for i, (s, t) in
               enumerate([((B, H, Lq, D), torch.float32), ((B, H, Lk, D), torch.float16), ((B, H, Lk, D), torch.float16)]))
    outs = [torch.empty((B, Lq, H, D), dtype=torch.float32, device=DEV) for _ in range(2)]
    descs = [kd_fa.make_desc(q, k, v, None, o, D ** -0.5) for o in outs]
    size = kd_fa.workspace_size_full(descs[0])
    assert size > 0
    ws = torch.full((size,), 0x7F, dtype=torch.uint8, device=DEV)
    assert kd_fa.run_desc(descs[0], workspace=ws) == kd_fa.OK
    assert kd_fa.run_desc(descs[1]) == kd_fa.OK
    torch.cuda.synchronize()
    assert bool((ws == 0x7F).all())
    assert torch.equal(outs[0], outs[1])
