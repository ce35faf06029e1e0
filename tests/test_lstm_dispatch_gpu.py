"""The LSTM step kernel AUTO runs, at the sizes where its tiles and its division of the columns end: every tile shape,
batches that are not whole tiles, last chunks of 16, 32 and 48 columns in either part, wavefronts without a chunk. Against
the oracle, in the tolerance of the layer (outputs below 1, gates' sums rounded once to f16 by the inputs: 1e-2)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ABS_TOL = 1e-2


@pytest.mark.parametrize("T,B,I,H", [(2, 16, 1024, 1024),   # 4 units x 16 rows
                                     (2, 32, 480, 992),     # 4 x 32
                                     (3, 48, 80, 112),      # 4 x 16, fewer chunks than wavefronts
                                     (2, 80, 336, 656),     # 8 x 32: rows 16 of 32 in the last tile
                                     (2, 16, 64, 2048),     # 8 x 16
                                     (1, 16, 96, 3056),     # 16 x 16
                                     (2, 112, 80, 1008),    # 16 x 32, rows 16 of 32
                                     (2, 240, 368, 592),    # 16 x 64, rows 48 of 64
                                     (3, 16, 16, 16), (2, 64, 144, 272)])
@pytest.mark.parametrize("with_state", [False, True])
def test_lstm_step_tiles(tcu, oracle, device, T, B, I, H, with_state):
    import torch

    print(f"lstm tiles T{T} B{B} I{I} H{H} state={with_state}", flush=True)
    x = oracle.fill_normal(T * B * I, 61, 0, 0.5).reshape(T, B, I)
    W = oracle.fill_normal(4 * H * (I + H), 62, 0, 0.05).reshape(4 * H, I + H)
    b = oracle.fill_normal(4 * H, 63, 0, 0.1)
    h0 = oracle.fill_normal(B * H, 64, 0, 0.5).reshape(B, H) if with_state else None
    c0 = oracle.fill_normal(B * H, 65, 0, 0.5).reshape(B, H).astype(np.float32) if with_state else None
    to = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(device)
    h_buf = torch.full((T * B * H + 4096,), 7.0, dtype=torch.float16, device=device)
    c_buf = torch.full((B * H + 4096,), 7.0, dtype=torch.float32, device=device)
    out = (h_buf[:T * B * H].view(T, B, H), c_buf[:B * H].view(B, H))
    h_all, c_T = tcu.lstm(to(x), to(W), to(b), to(h0), to(c0), out=out)
    torch.cuda.synchronize()
    h_ref, c_ref = oracle.lstm(x, W, b, h0, c0)
    assert oracle.max_abs_err(h_all.float().cpu().numpy(), h_ref) <= ABS_TOL
    assert oracle.max_abs_err(c_T.cpu().numpy(), c_ref) <= ABS_TOL
    assert bool((h_buf[T * B * H:] == 7.0).all()) and bool((c_buf[B * H:] == 7.0).all())
