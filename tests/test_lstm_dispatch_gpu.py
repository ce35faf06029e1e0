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


@pytest.mark.parametrize("T,B,I,H", [(16, 256, 4096, 1024), (8, 1024, 4096, 512), (16, 64, 2048, 512), (8, 64, 8192, 2048)])
def test_lstm_projects_long_inputs_beforehand(tcu, device, T, B, I, H):
    """Long inputs: AUTO and the torch op compute the input half of the gates in one GEMM (bit for bit ``algo="hoisted"``), in a
    workspace of the caller's as well, and run one fused kernel per step with ``workspace=False``. The two differ by the
    order of f32 sums before h is rounded to f16 (2^-11, outputs below 1, carried over T steps)."""
    import torch

    import tiledcuda_amd.torch_ops  # noqa: F401

    print(f"lstm projection T{T} B{B} I{I} H{H}", flush=True)
    gen = torch.Generator(device=device)
    gen.manual_seed(T + I)
    normal = lambda *shape, std=1.0: torch.randn(*shape, generator=gen, device=device).mul_(std).half()
    x, W, b = normal(T, B, I, std=0.5), normal(4 * H, I + H, std=0.02), normal(4 * H, std=0.1)
    assert tcu.lib().tcu_lstm_uses_workspace(T, B, I, H) == 1
    need = tcu.lstm_workspace_bytes(T, B, I, H)
    want, fused = tcu.lstm(x, W, b, algo="hoisted"), tcu.lstm(x, W, b, workspace=False)
    ws = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=device)
    for got in (tcu.lstm(x, W, b), tcu.lstm(x, W, b, workspace=ws), torch.ops.tiledcuda.lstm(x, W, b, None, None)):
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert bool((ws[need:] == 0x5A).all()) and not bool((ws[:need] == 0x5A).all())
    assert not torch.equal(fused[1], want[1])
    assert float((fused[0].float() - want[0].float()).abs().max()) <= ABS_TOL


def test_lstm_fuses_short_inputs(tcu, device):
    """The sizes at which a fused kernel per step is the faster plan, and shapes the projection does not take."""
    uses = tcu.lib().tcu_lstm_uses_workspace
    for shape in ((16, 256, 1024, 1024), (8, 512, 512, 1024), (24, 80, 336, 656), (16, 80, 4096, 1024), (3, 256, 8192, 1024), (0, 1, 1, 1)):
        assert uses(*shape) == 0, shape
