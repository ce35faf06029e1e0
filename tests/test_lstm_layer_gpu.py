"""The LSTM layer whose time loop is one launch (``algo="layer"``): every instantiation, sizes where its slices, row tiles and columns
end, more groups of rows than XCDs, and launches with fewer workgroups than slices. Against the oracle, in the tolerance of the
layer (outputs below 1, h rounded to f16 every step: 1e-2), and against the step kernels, which differ by the order of f32 sums
before that rounding (2^-11 per step, carried over T steps: 4e-3)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ABS_TOL, STEP_TOL = 1e-2, 4e-3


def operands(tcu, device, T, B, I, H, state=True):
    import torch

    gen = torch.Generator(device=device)
    gen.manual_seed(T * B + I + H)
    normal = lambda *shape, std=1.0: torch.randn(*shape, generator=gen, device=device).mul_(std)
    return (normal(T, B, I, std=0.5).half(), normal(4 * H, I + H, std=0.05).half(), normal(4 * H, std=0.1).half(),
            normal(B, H, std=0.5).half() if state else None, normal(B, H, std=0.5) if state else None)


def close(got, want, tol=STEP_TOL):
    return all(float((g.float() - w.float()).abs().max()) <= tol for g, w in zip(got, want))


def limited(tcu, args, workgroups, takeover_us=30, max_tries=1 << 24):
    """The layer in a launch of at most ``workgroups`` workgroups."""
    import torch

    x, W, b, h0, c0 = args
    T, B, I = x.shape
    H = b.numel() // 4
    need = int(tcu.lib().tcu_lstm_layer_workspace_bytes(T, B, I, H))
    ws = torch.full((need,), 0x5A, dtype=torch.uint8, device=x.device)
    h_all = torch.full((T, B, H), 7.0, dtype=torch.float16, device=x.device)
    c_T = torch.full((B, H), 7.0, dtype=torch.float32, device=x.device)
    ptr = lambda t: 0 if t is None else t.data_ptr()
    tcu._check(tcu.lib().tcu_lstm_f16_layer_limited(*map(ptr, (x, W, b, h0, c0, h_all, c_T)), T, B, I, H, ptr(ws), need, workgroups,
                                                    takeover_us, max_tries, tcu._stream()))
    return h_all, c_T


@pytest.mark.parametrize("T,B,I,H", [(2, 16, 16, 16), (3, 48, 64, 112), (5, 128, 80, 128),    # 16 units, 128 columns
                                     (4, 144, 64, 64), (3, 240, 96, 128),                     # ... 32 rows, 16 of 32 in the last group
                                     (4, 80, 128, 144), (3, 160, 64, 256),                    # 256 columns
                                     (3, 16, 48, 272), (3, 128, 64, 512), (3, 208, 64, 496),  # 512
                                     (4, 80, 336, 656), (3, 144, 64, 528), (3, 256, 64, 768),  # 32 units, 768
                                     (3, 32, 64, 784), (3, 16, 64, 1024), (3, 240, 64, 1008), (3, 256, 128, 1024),
                                     (4, 336, 64, 112), (3, 1040, 16, 80)])                    # more groups than XCDs
@pytest.mark.parametrize("state", [False, True])
def test_lstm_layer_matches_the_steps(tcu, device, T, B, I, H, state):
    import torch

    print(f"lstm layer T{T} B{B} I{I} H{H} state={state}", flush=True)
    args = operands(tcu, device, T, B, I, H, state)
    want = tcu.lstm(*args, workspace=False)
    h_buf = torch.full((T * B * H + 4096,), 7.0, dtype=torch.float16, device=device)
    c_buf = torch.full((B * H + 4096,), 7.0, dtype=torch.float32, device=device)
    need = int(tcu.lib().tcu_lstm_layer_workspace_bytes(T, B, I, H))
    ws = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=device)
    for _ in range(2):  # (the synchronisation words of the first call are in the workspace of the second)
        out = (h_buf[:T * B * H].view(T, B, H), c_buf[:B * H].view(B, H))
        assert close(tcu.lstm(*args, algo="layer", workspace=ws, out=out), want)
    assert bool((h_buf[T * B * H:] == 7.0).all()) and bool((c_buf[B * H:] == 7.0).all()) and bool((ws[need:] == 0x5A).all())


@pytest.mark.parametrize("T,B,I,H", [(2, 16, 16, 16), (3, 144, 64, 128), (2, 80, 64, 656),                         # two buffers of pre-activations
                                     (2, 144, 48, 272), (3, 256, 64, 512), (2, 208, 48, 656), (2, 16, 64, 784),      # one: H > 768, or
                                     (3, 80, 48, 1024), (2, 512, 48, 1008)])                                          # more than 128 rows and H > 256
def test_lstm_layer_without_an_initial_state(tcu, device, T, B, I, H):
    """No h0 is an h0 of zeros, bit for bit: the products of zeros add nothing to the pre-activations, whichever way step 0 takes them."""
    import torch

    print(f"lstm layer no h0 T{T} B{B} I{I} H{H}", flush=True)
    x, W, b, h0, c0 = operands(tcu, device, T, B, I, H)
    want = tcu.lstm(x, W, b, torch.zeros_like(h0), c0, algo="layer")
    assert close(want, tcu.lstm(x, W, b, None, c0, workspace=False))
    for _ in range(8):
        got = tcu.lstm(x, W, b, None, c0, algo="layer")
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def ran(tcu, name, back=0):
    """Whether the kernel of the last launch but ``back`` is ``name`` (an instantiation of the template)."""
    return f"{len(name)}{name}I" in tcu.lib().tcu_recent_kernel(back).decode()


@pytest.mark.parametrize("T,B,I,H,projection", [(7, 16, 16, 16, "gemm_direct"),
                                                # K-splitting: rows and gates partial, rows whole, both whole; K tails with the same
                                                (23, 208, 384, 112, "gemm_w128k"), (19, 256, 384, 112, "gemm_w128k"), (17, 128, 384, 256, "gemm_w128k"),
                                                (23, 208, 704, 112, "gemm_w128k"), (17, 128, 704, 256, "gemm_w128k"), (9, 224, 704, 464, "gemm_w128k"),
                                                # 256 x 256 tiles: partial, whole; K tails; the layer with odd multiples of 16
                                                (23, 208, 64, 64, "gemm_w128"), (19, 256, 64, 64, "gemm_w128"), (24, 240, 16, 64, "gemm_w128"),
                                                (23, 256, 16, 64, "gemm_w128"), (24, 80, 336, 656, "gemm_w128"),
                                                # the pipelined kernel's ring and its 64 x 64 tiles, with K tails and without
                                                (9, 96, 16, 16, "gemm_pipelined"), (8, 48, 64, 64, "gemm_pipelined"),
                                                (10, 208, 336, 256, "gemm_pipelined"), (12, 112, 1024, 768, "gemm_pipelined")])
def test_lstm_layer_projections(tcu, device, T, B, I, H, projection):
    """Every kernel that computes the input half of the gates, with W's row distance and the synchronisation words to clear: twice in one
    workspace whose words hold something else before each call. AUTO takes the same."""
    import torch

    print(f"lstm layer projection T{T} B{B} I{I} H{H} {projection}", flush=True)
    args = operands(tcu, device, T, B, I, H)
    want = tcu.lstm(*args, workspace=False)
    need = int(tcu.lib().tcu_lstm_layer_workspace_bytes(T, B, I, H))
    ws = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=device)
    for _ in range(2):
        got = tcu.lstm(*args, algo="layer", workspace=ws)
        assert ran(tcu, "lstm_layer_xcd") and ran(tcu, projection, 1)
        assert close(got, want)
        ws[:4096] = 0x5A
    assert bool((ws[need:] == 0x5A).all()) and tcu.lib().tcu_lstm_uses_layer(T, B, I, H) == 1
    auto = tcu.lstm(*args)
    assert ran(tcu, "lstm_layer_xcd") and ran(tcu, projection, 1) and torch.equal(auto[0], got[0]) and torch.equal(auto[1], got[1])


def test_lstm_layer_against_the_oracle(tcu, oracle, device):
    import torch

    T, B, I, H = 6, 80, 336, 656
    x = oracle.fill_normal(T * B * I, 61, 0, 0.5).reshape(T, B, I)
    W = oracle.fill_normal(4 * H * (I + H), 62, 0, 0.05).reshape(4 * H, I + H)
    b = oracle.fill_normal(4 * H, 63, 0, 0.1)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)
    h_all, c_T = tcu.lstm(to(x), to(W), to(b), algo="layer")
    h_ref, c_ref = oracle.lstm(x, W, b)
    assert oracle.max_abs_err(h_all.float().cpu().numpy(), h_ref) <= ABS_TOL
    assert oracle.max_abs_err(c_T.cpu().numpy(), c_ref) <= ABS_TOL


@pytest.mark.parametrize("T,B,I,H,grid", [(5, 80, 64, 112, 1), (5, 80, 64, 112, 8), (5, 80, 64, 112, 40), (4, 144, 96, 656, 9),
                                          (4, 256, 64, 1024, 100), (4, 336, 64, 320, 24), (3, 16, 64, 784, 5), (3, 160, 64, 272, 9)])
@pytest.mark.parametrize("state", [False, True])
def test_lstm_layer_with_few_workgroups(tcu, device, T, B, I, H, grid, state):
    """Slices without a workgroup are taken over by those that run, groups of rows by XCDs that are done; at the smallest, one
    workgroup does everything."""
    import torch

    print(f"lstm layer T{T} B{B} I{I} H{H} grid {grid} state={state}", flush=True)
    args = operands(tcu, device, T, B, I, H, state)
    want = tcu.lstm(*args, workspace=False)
    layer = tcu.lstm(*args, algo="layer")
    assert close(layer, want)
    got = limited(tcu, args, grid)
    assert torch.equal(got[0], layer[0]) and torch.equal(got[1], layer[1])


def test_lstm_layer_limits_are_checked(tcu, device):
    args = operands(tcu, device, 2, 16, 16, 16)
    for limits in ((0, 30), (-1, 30), (8, -1), (8, 1000001), (8, 30, -1)):
        with pytest.raises(RuntimeError, match="workgroup"):
            limited(tcu, args, *limits)


@pytest.mark.parametrize("T,B,I,H,units", [(4, 16, 64, 656, 32), (3, 48, 64, 272, 16), (3, 160, 64, 1024, 32)])
def test_lstm_layer_gives_up_with_nan(tcu, device, T, B, I, H, units):
    """A wait that does not end: one workgroup, told not to take over the other slices and to poll once. The launch ends, and what the
    workgroup computes from then on is NaN; the next call is not affected."""
    import torch

    print(f"lstm layer gives up T{T} B{B} I{I} H{H}", flush=True)
    args = operands(tcu, device, T, B, I, H)
    h_all, c_T = limited(tcu, args, 1, 1000000, 0)
    assert bool(torch.isnan(h_all[1:, :, :units]).all()) and bool(torch.isnan(c_T[:, :units]).all())
    assert bool((c_T[:, units:] == 7.0).all()) and bool((h_all[:, :, units:] == 7.0).all())
    assert close(tcu.lstm(*args, algo="layer"), tcu.lstm(*args, workspace=False))


def test_lstm_layer_two_streams_and_nan(tcu, device):
    """Calls that overlap on two streams, each with a workspace of its own; NaN inputs stay NaNs of their rows (and end no wait
    early or late), infinite initial states saturate."""
    import torch

    T, B, I, H = 12, 80, 96, 528
    args = operands(tcu, device, T, B, I, H)
    want = tcu.lstm(*args, workspace=False)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for k in range(6):
        with torch.cuda.stream(streams[k % 2]):
            got.append(tcu.lstm(*args, algo="layer"))
    torch.cuda.synchronize()
    assert all(close(g, want) for g in got)
    x, W, b, h0, c0 = (t.clone() for t in args)
    x.view(torch.int16)[2, 17, 3] = -1  # 0xffff
    x.view(torch.int16)[5, 40, :] = -1
    h0[3, 5] = float("inf")
    want, got = tcu.lstm(x, W, b, h0, c0, workspace=False), tcu.lstm(x, W, b, h0, c0, algo="layer")
    for w, g in zip(want, got):
        assert torch.equal(torch.isnan(w), torch.isnan(g))
        assert close((torch.nan_to_num(g),), (torch.nan_to_num(w),))


@pytest.mark.parametrize("T,B,I,H,parts", [(9, 2048, 16, 1024, 2), (65, 256, 64, 1024, 2), (135, 256, 16, 1008, 3), (64, 256, 64, 1024, 1)])
def test_lstm_layer_in_parts(tcu, device, T, B, I, H, parts):
    """Layers whose pre-activations would take more than 256 MiB: bit for bit what the parts give by themselves, in a workspace of the
    stated size and no more, with an initial state and without."""
    import torch

    print(f"lstm layer in parts T{T} B{B} I{I} H{H}", flush=True)
    x, W, b, h0, c0 = operands(tcu, device, T, B, I, H)
    need = int(tcu.lib().tcu_lstm_layer_workspace_bytes(T, B, I, H))
    assert need == 4096 + -(-T // parts) * B * H * 16 <= 4096 + 2 ** 28
    ws = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=device)
    for state in ((h0, c0), (None, None)):
        got = tcu.lstm(x, W, b, *state, algo="layer", workspace=ws)
        h, c = state
        for k in range(parts):
            first, last = T * k // parts, T * (k + 1) // parts
            h_part, c = tcu.lstm(x[first:last], W, b, h, c, algo="layer")
            assert torch.equal(got[0][first:last], h_part)
            h = h_part[-1]
        assert torch.equal(got[1], c)
        assert close(got, tcu.lstm(x, W, b, *state, workspace=False), 8e-3)  # (up to 135 steps: twice the bound of the short layers)
    assert bool((ws[need:] == 0x5A).all())


def test_lstm_layer_fed_with_its_own_outputs(tcu, device):
    """Inputs that are the outputs a step before, in the same memory: what a launch per step gives, and what feeding them one call at a
    time gives."""
    import torch

    T, B, H = 12, 48, 272
    assert tcu.lib().tcu_lstm_uses_layer(T, B, H, H) == 1
    x, W, b, h0, c0 = operands(tcu, device, T, B, H, H)
    want = [x[0]]
    h, c = h0, c0
    for _ in range(T):
        h_all, c = tcu.lstm(want[-1][None], W, b, h, c)
        h = h_all[0]
        want.append(h)
    for kwargs in ({}, {"algo": "layer"}, {"workspace": False}):
        buf, c_T = torch.zeros(T + 1, B, H, dtype=torch.float16, device=device), torch.empty(B, H, device=device)
        buf[0] = x[0]
        tcu.lstm(buf[:-1], W, b, h0, c0, out=(buf[1:], c_T), **kwargs)
        assert torch.equal(buf, torch.stack(want)) and torch.equal(c_T, c), kwargs


def test_lstm_auto_with_a_workspace_the_layer_cannot_use(tcu, device):
    """A size whose AUTO was a launch per step and never looked at the workspace: one on the host, with gaps, misaligned, too small or
    no tensor at all is left alone, and the steps run; ``algo="layer"`` refuses it."""
    import torch

    T, B, I, H = 24, 48, 64, 272
    args = operands(tcu, device, T, B, I, H)
    steps = tcu.lstm(*args, workspace=False)
    need = int(tcu.lib().tcu_lstm_layer_workspace_bytes(T, B, I, H))
    assert tcu.lib().tcu_lstm_uses_layer(T, B, I, H) == 1 and tcu.lib().tcu_lstm_uses_workspace(T, B, I, H) == 0
    room = torch.full((2 * need,), 0x5A, dtype=torch.uint8, device=device)
    for ws in (torch.empty(need, dtype=torch.uint8), room[::2], room[4:need + 4], room[:need - 1]):
        got = tcu.lstm(*args, workspace=ws)
        assert torch.equal(got[0], steps[0]) and torch.equal(got[1], steps[1])
        with pytest.raises((ValueError, RuntimeError)):
            tcu.lstm(*args, algo="layer", workspace=ws)
    got = tcu.lstm(*args, workspace=True)
    assert torch.equal(got[0], steps[0]) and torch.equal(got[1], steps[1]) and bool((room == 0x5A).all())


@pytest.mark.parametrize("entry", ["python", "calls", "op"])
def test_lstm_auto_without_memory_for_a_workspace(tcu, device, entry):
    """AUTO needs no memory beside its outputs: where the allocator has none for the layer's workspace the steps run."""
    import torch

    import tiledcuda_amd.torch_ops  # noqa: F401

    T, B, I, H = 64, 256, 64, 1024  # h_all 32 MiB, the workspace 256
    assert tcu.lib().tcu_lstm_uses_layer(T, B, I, H) == 1
    args = operands(tcu, device, T, B, I, H)
    steps = tcu.lstm(*args, workspace=False)
    out = tuple(torch.empty_like(t) for t in steps)
    call = {"python": lambda: tcu.lstm(*args, out=out), "calls": lambda: tcu.lstm(*args), "op": lambda: torch.ops.tiledcuda.lstm(*args)}[entry]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (128 << 20)) / total)
    try:
        got = call()
        with pytest.raises(torch.OutOfMemoryError):
            tcu.lstm(*args, algo="layer")
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got[0], steps[0]) and torch.equal(got[1], steps[1])
    assert not torch.equal(tcu.lstm(*args)[0], steps[0])


def test_lstm_layers_beside_each_other(tcu, device):
    """Two layers on two streams whose workgroups do not all fit at once: the later one waits for CUs rather than run its slices two to
    a workgroup, which took three times as long as one layer after the other. (Both orders of streams, best of several: a third more
    than in turn is allowed.)"""
    import time

    import torch

    T, B, I, H = 64, 80, 336, 656
    args = operands(tcu, device, T, B, I, H)
    want = tcu.lstm(*args, algo="layer")
    ws = [torch.empty(int(tcu.lib().tcu_lstm_layer_workspace_bytes(T, B, I, H)), dtype=torch.uint8, device=device) for _ in range(2)]
    outs = [tuple(torch.empty_like(t) for t in want) for _ in range(2)]
    two = [torch.cuda.Stream() for _ in range(2)]

    def us(streams, calls=6):
        torch.cuda.synchronize()
        start = time.perf_counter()
        for _ in range(calls):
            for s, w, o in zip(streams, ws, outs):
                with torch.cuda.stream(s):
                    tcu.lstm(*args, algo="layer", workspace=w, out=o)
        torch.cuda.synchronize()
        return (time.perf_counter() - start) * 1e6 / calls

    in_turn, together = min(us(two[:1] * 2) for _ in range(4)), min(us(two) for _ in range(4))
    print(f"lstm layers in turn {in_turn:.0f} us, on two streams {together:.0f} us", flush=True)
    assert all(torch.equal(a, b) for o in outs for a, b in zip(o, want))
    assert together <= 1.33 * in_turn


def test_lstm_layer_route(tcu, device):
    """Where AUTO takes it, where not, and what it does with a caller's workspace, an h0 inside h_all and a captured stream."""
    import torch

    import tiledcuda_amd.torch_ops  # noqa: F401

    uses, need = tcu.lib().tcu_lstm_uses_layer, tcu.lib().tcu_lstm_layer_workspace_bytes
    for shape in ((16, 256, 1024, 1024), (24, 80, 336, 656), (20, 16, 416, 80), (12, 144, 80, 208)):
        assert uses(*shape) == 1, shape
    for shape in ((3, 16, 64, 64), (16, 256, 4096, 1024), (31, 4096, 96, 160), (16, 64, 64, 1040), (16, 24, 64, 64), (0, 1, 1, 1),
                  (14, 480, 288, 288), (20, 464, 128, 448), (5, 368, 144, 768), (13, 464, 128, 432), (16, 448, 240, 384)):  # measured slower than the steps
        assert uses(*shape) == 0, shape
    assert need(1, 16, 64, 64) == 0 and need(2, 16, 64, 1040) == 0 and need(2, 2064, 64, 64) == 0 and need(2, 16, 64, 64) == 4096 + 2 * 16 * 256 * 4
    T, B, I, H = 24, 48, 64, 272
    args = operands(tcu, device, T, B, I, H)
    steps, layer = tcu.lstm(*args, workspace=False), tcu.lstm(*args, algo="layer")
    same = lambda a, b: torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    assert uses(T, B, I, H) == 1 and not same(steps, layer)
    ws = torch.full((need(T, B, I, H),), 0x5A, dtype=torch.uint8, device=device)
    assert same(tcu.lstm(*args), layer) and same(torch.ops.tiledcuda.lstm(*args), layer)
    assert same(tcu.lstm(*args, workspace=ws[:-1]), steps) and bool((ws == 0x5A).all())
    assert same(tcu.lstm(*args, workspace=ws), layer) and not bool((ws == 0x5A).all())
    # an initial state that is a step of the output
    out = (torch.empty(T, B, H, dtype=torch.float16, device=device), torch.empty(B, H, device=device))
    out[0][5].copy_(args[3])
    assert same(tcu.lstm(*args[:3], out[0][5], args[4], workspace=ws, out=out), steps)
    # captured: the steps, or the layer in the caller's workspace, replayed with work in between
    for workspace, want in ((None, steps), (ws, layer)):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            tcu.lstm(*args, workspace=workspace, out=out)
        for _ in range(3):
            out[0].zero_(), out[1].zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert same(out, want)
