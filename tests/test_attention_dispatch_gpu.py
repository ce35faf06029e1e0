"""Attention launches that AUTO sends to a kernel for reasons of size: query counts that are not whole blocks, few query
blocks. Against the oracle on sampled heads, with a guard region behind the output.

Tolerance: queries times scale, probabilities and outputs are each rounded to f16 (2^-11); logits of N(0, 1) data stay
below 6 and |v| below 5, so an output is within 5 * 2^-11 * (6 + 1 + 1) = 2e-2 of the exact one if every rounding goes the
same way, and half of that bounds sums of many."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ABS_TOL = 1e-2


def _run(tcu, oracle, device, call, batch, M, N, D, heads):
    import torch

    q = oracle.fill_normal(batch * M * D, 31).reshape(batch, M, D)
    k = oracle.fill_normal(batch * N * D, 32).reshape(batch, N, D)
    v = oracle.fill_normal(batch * N * D, 33).reshape(batch, N, D)
    buf = torch.full((batch * M * D + 256 * D,), 7.0, dtype=torch.float16, device=device)
    out = buf[:batch * M * D].view(batch, M, D)
    dq, dk, dv = (torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in (q, k, v))
    call(dq, dk, dv, out)
    torch.cuda.synchronize()
    for b in heads:
        ref = oracle.attention(q[b:b + 1], k[b:b + 1], v[b:b + 1], 1.0 / math.sqrt(D))
        assert oracle.max_abs_err(out[b:b + 1].float().cpu().numpy(), ref) <= ABS_TOL
    assert bool((buf[batch * M * D:] == 7.0).all())
    return dq, dk, dv, out


@pytest.mark.parametrize("algo", ["mfma32", "mfma32_fused"])
@pytest.mark.parametrize("batch,M,N,D", [(200, 192, 128, 128), (300, 64, 64, 128), (101, 320, 192, 128), (96, 576, 64, 64),
                                         (100, 448, 128, 64), (258, 128, 64, 64)])
def test_query_counts_that_are_not_whole_blocks(tcu, oracle, device, batch, M, N, D, algo):
    """The 32-queries-per-wavefront kernels with 2, 4 or 8 wavefronts by the number of rounds a launch takes, the last
    block of a head partly beyond M (its wavefronts there store nothing); head counts that are not multiples of 8."""
    print(f"attention partial blocks b{batch} {M}x{N} D{D} {algo}", flush=True)
    _run(tcu, oracle, device, lambda q, k, v, o: tcu.flash_attention(q, k, v, out=o, algo=algo), batch, M, N, D,
         (0, batch // 2, batch - 1))
