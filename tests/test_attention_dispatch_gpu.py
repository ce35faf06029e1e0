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


@pytest.mark.parametrize("v_layout", ["row", "col"])
@pytest.mark.parametrize("batch,M,N,D", [(1, 64, 64, 128), (1, 64, 128, 128), (3, 192, 320, 128), (2, 128, 576, 128),
                                         (5, 64, 1024, 128), (1, 64, 64, 64), (3, 192, 320, 64), (9, 128, 832, 64)])
def test_wavefronts_split_the_keys(tcu, oracle, device, batch, M, N, D, v_layout):
    """The key-splitting kernel by name: 1 to 8 blocks of 32 keys per wavefront (even and odd counts take different ways
    out of its unrolled loop), wavefronts with no block at all (64 keys) and with one less than the others, head counts
    that are not multiples of 8; both V layouts at head size 128."""
    if v_layout == "col" and D != 128:
        pytest.skip("a column-major V is instantiated for head size 128")
    print(f"attention keys b{batch} {M}x{N} D{D} V {v_layout}", flush=True)

    def call(q, k, v, o):
        if v_layout == "row":
            tcu.flash_attention(q, k, v, out=o, algo="keys")
        else:
            tcu.flash_attention_fwd(q.flatten(), k.flatten(), v.transpose(1, 2).contiguous().flatten(), o.view(-1), M, N, D, D,
                                    scale=1.0 / math.sqrt(D), batch=batch, algo="keys")

    _run(tcu, oracle, device, call, batch, M, N, D, range(batch))


@pytest.mark.parametrize("batch,M,N,D,v_layout", [(1, 64, 8192, 128, "row"), (1, 64, 8192, 128, "col"), (32, 64, 4096, 128, "row"),
                                                  (3, 192, 2112, 128, "row"), (2, 64, 4096, 64, "row")])
def test_workgroups_split_the_keys_through_a_workspace(tcu, oracle, device, batch, M, N, D, v_layout):
    """Few queries against many keys: AUTO splits the keys over workgroups when it has a workspace (one of the caller's,
    whose bytes past the stated size stay untouched, or one it takes itself) and gives the same result without one, up to
    rounding; splits of unequal length (66 blocks of 32 keys)."""
    import torch

    code = tcu.TCU_V_ROW_MAJOR if v_layout == "row" else tcu.TCU_V_COL_MAJOR
    need = tcu.attention_workspace_bytes(batch, M, N, D, D, code)
    print(f"attention split keys b{batch} {M}x{N} D{D} V {v_layout}: {need} bytes", flush=True)
    assert need > 0 and need % (batch * M * (D + 2) * 4) == 0
    ws = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=device)

    def call(workspace):
        def go(q, k, v, o):
            if v_layout == "row":
                tcu.flash_attention(q, k, v, out=o, workspace=workspace)
            else:
                tcu.flash_attention_fwd(q.flatten(), k.flatten(), v.transpose(1, 2).contiguous().flatten(), o.view(-1), M, N, D,
                                        D, scale=1.0 / math.sqrt(D), batch=batch, workspace=workspace)
        return go

    q, k, v, out = _run(tcu, oracle, device, call(ws), batch, M, N, D, {0, batch - 1})
    assert bool((ws[need:] == 0x5A).all())
    own, unsplit = torch.empty_like(out), torch.empty_like(out)
    call(None)(q, k, v, own)
    call(False)(q, k, v, unsplit)
    torch.cuda.synchronize()
    assert torch.equal(own, out)
    assert float((unsplit.float() - out.float()).abs().max()) <= 2 * ABS_TOL


@pytest.mark.parametrize("N,splits", [(512, 1), (4096, 4)])
def test_keys_kernel_moves_its_maxima(tcu, oracle, device, N, splits):
    """Keys whose norm grows along the sequence and large queries: the maxima move in many blocks, and the splits of the
    keys differ in theirs by far. Logits reach 30 here, where rounding the scaled queries to f16 alone costs
    30 * 2^-11 * 5 / 2 = 4e-2 at most."""
    import torch

    batch, M, D = 2, 64, 128
    q = (oracle.fill_normal(batch * M * D, 41).reshape(batch, M, D).astype(np.float32) * 2).astype(np.float16)
    k = oracle.fill_normal(batch * N * D, 42).reshape(batch, N, D).astype(np.float32)
    k = (k * np.linspace(0.2, 3.0, N, dtype=np.float32)[None, :, None]).astype(np.float16)
    v = oracle.fill_normal(batch * N * D, 43).reshape(batch, N, D)
    assert (tcu.attention_workspace_bytes(batch, M, N, D, D) > 0) == (splits > 1)
    dq, dk, dv = (torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in (q, k, v))
    out = tcu.flash_attention(dq, dk, dv) if splits > 1 else tcu.flash_attention(dq, dk, dv, algo="keys")
    torch.cuda.synchronize()
    assert oracle.max_abs_err(out.float().cpu().numpy(), oracle.attention(q, k, v, 1.0 / math.sqrt(D))) <= 4e-2


def _masked(oracle, batch, M, N, D, masked, level):
    """N(0, 1) operands whose feature 0 masks keys: 1 in every query, -infinity in the masked keys and `level` in the others."""
    q = oracle.fill_normal(batch * M * D, 51).reshape(batch, M, D)
    k = oracle.fill_normal(batch * N * D, 52).reshape(batch, N, D)
    v = oracle.fill_normal(batch * N * D, 53).reshape(batch, N, D)
    q[..., 0] = 1.0
    k[..., 0] = level
    k[:, masked, 0] = -np.inf
    return q, k, v


@pytest.mark.parametrize("D,v_layout", [(128, "row"), (128, "col"), (64, "row")])
@pytest.mark.parametrize("N,masked", [(512, slice(32, 64)), (512, slice(0, 128)), (512, slice(192, 512)), (512, slice(1, 512)),
                                      (4096, slice(0, 1024)), (4096, slice(1024, 2048)), (4096, slice(1000, 4096)),
                                      (4096, slice(0, 4032))])
@pytest.mark.parametrize("level", [0.0, -600.0])
def test_masked_keys(tcu, oracle, device, N, masked, D, v_layout, level):
    """Scores of -infinity: over one wavefront's first block of 32 keys, over every wavefront's, over a whole split of the keys,
    over their tail, over all but one. level = -600 puts the scores that are left near -53 (-75 at head size 64), far below a
    maximum of 0, where 2^s itself is far below the least f16. By name and through AUTO with its workspace and without. The
    tolerance is that of the other tests with N(0, 1) logits: the level adds the same rounded number to all scores of a row
    (its product with q's rounded scale enters every score alike), and f32 scores of magnitude 110 in the log2 domain are
    off by 110 * 2^-24 each: nothing beside f16's 2^-11."""
    import torch

    batch, M = 2, 64
    q, k, v = _masked(oracle, batch, M, N, D, masked, level)
    print(f"attention masked keys {N} {masked} D{D} V {v_layout} level {level}", flush=True)
    dq, dk, dv = (torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in (q, k, v))
    ref = oracle.attention(q, k, v, 1.0 / math.sqrt(D))
    assert np.isfinite(ref).all()
    calls = [dict(algo="keys"), dict(workspace=False), dict()]
    for kw in calls:
        if v_layout == "row":
            out = tcu.flash_attention(dq, dk, dv, **kw)
        else:
            out = torch.empty_like(dq)
            tcu.flash_attention_fwd(dq.flatten(), dk.flatten(), dv.transpose(1, 2).contiguous().flatten(), out.view(-1), M, N, D, D,
                                    scale=1.0 / math.sqrt(D), batch=batch, **kw)
        torch.cuda.synchronize()
        assert oracle.max_abs_err(out.float().cpu().numpy(), ref) <= ABS_TOL, kw


@pytest.mark.parametrize("N", [64, 512, 4096])
def test_all_keys_masked_stay_undefined(tcu, oracle, device, N):
    """A row of nothing but -infinity has no softmax: NaN, as before the keys were split, in the masked head only."""
    import torch

    q, k, v = _masked(oracle, 2, 64, N, 128, slice(0, 0), 0.0)
    k[1, :, 0] = -np.inf
    out = tcu.flash_attention(*(torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in (q, k, v)), algo="auto")
    torch.cuda.synchronize()
    assert bool(out[1].isnan().all()) and not bool(out[0].isnan().any())


def test_infinite_value_keeps_its_sign(tcu, oracle, device):
    """One infinite value, at a key with a weight of about 1/N: its column is infinite, not NaN, also where fewer workgroups
    than the combining kernel has slots for split the keys."""
    import torch

    q, k, v = _masked(oracle, 3, 192, 2112, 128, slice(0, 0), 0.0)
    v[:, -1, 7] = np.inf  # (the last split: what unused slots would repeat)
    dq, dk, dv = (torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in (q, k, v))
    need = tcu.attention_workspace_bytes(3, 192, 2112, 128, 128)
    assert need // (3 * 192 * 130 * 4) == 12
    out = tcu.flash_attention(dq, dk, dv)
    torch.cuda.synchronize()
    assert bool((out[..., 7] == float("inf")).all())
    assert bool(out[..., :7].isfinite().all()) and bool(out[..., 8:].isfinite().all())


@pytest.mark.parametrize("entry", ["python", "torch_op"])
def test_captured_calls_allocate_nothing(tcu, oracle, device, entry):
    """A call that would split its keys through a workspace from the allocator takes none while it is captured (it runs unsplit);
    a workspace of the caller's is used at every replay. Replays with eager work between them, each against the eager call."""
    import torch

    import tiledcuda_amd.torch_ops  # noqa: F401

    M, N, D = 64, 8192, 128
    q, k, v = (torch.from_numpy(oracle.fill_normal(rows * D, seed)).to(device) for rows, seed in ((M, 71), (N, 72), (N, 73)))
    need = tcu.attention_workspace_bytes(1, M, N, D, D, tcu.TCU_V_COL_MAJOR)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    own, plain = (torch.empty(M * D, dtype=torch.float16, device=device) for _ in range(2))

    def call(out, workspace):
        if entry == "python":
            tcu.flash_attention_fwd(q, k, v, out, M, N, D, D, workspace=workspace)
        else:
            torch.ops.tiledcuda.flash_attention_fwd(q, k, v, out, M, N, D, D)

    split, unsplit = torch.empty_like(own), torch.empty_like(own)
    tcu.flash_attention_fwd(q, k, v, split, M, N, D, D)
    tcu.flash_attention_fwd(q, k, v, unsplit, M, N, D, D, workspace=False)
    call(own, None)
    torch.cuda.synchronize()
    assert torch.equal(own, split) and not torch.equal(split, unsplit)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        call(plain, None)
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
        if entry == "python":
            call(own, ws)
    for _ in range(3):
        own.zero_(), plain.zero_(), ws.fill_(0x5A)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(plain, unsplit)
        assert entry != "python" or torch.equal(own, split)


@pytest.mark.parametrize("batch,N,algo", [(85, 2368, "keys"), (88, 1600, "keys"), (88, 4160, "wave64"), (96, 2368, "wave64")])
def test_192_queries_and_a_column_major_v(tcu, device, batch, N, algo):
    """Three workgroups per head split the keys until they need a second round of any size; then AUTO takes blocks of 256
    queries, one per head. Bit for bit the kernel by name, which the other differs from by the order of its sums."""
    import torch

    print(f"attention b{batch} 192x{N} D128 V col {algo}", flush=True)
    gen = torch.Generator(device=device)
    gen.manual_seed(N)
    q, k, v = (torch.randn(batch * n * 128, generator=gen, device=device).half() for n in (192, N, N))
    outs = {}
    for name in ("auto", "keys", "wave64"):
        outs[name] = torch.empty_like(q)
        tcu.flash_attention_fwd(q, k, v, outs[name], 192, N, 128, 128, scale=128 ** -0.5, batch=batch, algo=name)
    assert torch.equal(outs["auto"], outs[algo])
    assert not torch.equal(outs["keys"], outs["wave64"])


def _auto_is(tcu, device, batch, M, N, algo):
    import torch

    print(f"attention auto b{batch} {M}x{N} D64 {algo}", flush=True)
    gen = torch.Generator(device=device)
    gen.manual_seed(M)
    q, k, v = (torch.randn(batch, n, 64, generator=gen, device=device).half() for n in (M, N, N))
    named = {name: tcu.flash_attention(q, k, v, algo=name) for name in ("keys", "mfma32_fused", "wave64_k32")}
    got = tcu.flash_attention(q, k, v)
    assert [name for name, out in named.items() if torch.equal(got, out)] == [algo]


@pytest.mark.parametrize("batch,M,N,algo", [(84, 576, 2688, "keys"), (104, 448, 2560, "keys"), (62, 640, 704, "mfma32_fused")])
def test_blocks_partly_beyond_the_queries_against_split_keys(tcu, device, batch, M, N, algo):
    """One block of 256 queries per CU, the last of a head partly empty: AUTO counts what that costs when it looks at the
    key-splitting kernel. Bit for bit the kernel by name."""
    _auto_is(tcu, device, batch, M, N, algo)


@pytest.mark.parametrize("batch,M,N,algo", [(142, 3392, 448, "wave64_k32"), (134, 1856, 384, "mfma32_fused")])
def test_many_rounds_of_query_blocks(tcu, device, batch, M, N, algo):
    """More than three rounds of blocks of 256 queries that are not whole: AUTO runs the 16x16x32 kernel unless its estimate is
    far behind. Bit for bit the kernel by name."""
    _auto_is(tcu, device, batch, M, N, algo)


@pytest.mark.parametrize("D,v_layout,batches", [(128, "row", (1, 128, 129)), (128, "col", (3, 128, 129)), (64, "row", (2, 128, 129))])
@pytest.mark.parametrize("M,N", [(64, 64), (64, 192), (64, 320)])
def test_keys_kernel_with_32_and_64_queries(tcu, device, D, v_layout, batches, M, N):
    """The largest launches of workgroups of 32 queries and the smallest of 64 beyond them, with one to three blocks per wavefront
    and wavefronts without one, against f32 (f16 probabilities and output: 2^-11 each, 1.5e-3 as everywhere)."""
    import torch

    for batch in batches:
        print(f"attention keys rows b{batch} {M}x{N} D{D} V {v_layout}", flush=True)
        gen = torch.Generator(device=device)
        gen.manual_seed(batch + N)
        q, k, v = (torch.randn(batch, n, D, generator=gen, device=device).half() for n in (M, N, N))
        scale = 1.0 / math.sqrt(D)
        if v_layout == "row":
            out = tcu.flash_attention(q, k, v, algo="keys")
        else:
            out = torch.full_like(q, 7.0)
            tcu.flash_attention_fwd(q.flatten(), k.flatten(), v.transpose(1, 2).contiguous().flatten(), out.view(-1), M, N, D, D,
                                    scale=scale, batch=batch, algo="keys")
        want = torch.matmul(torch.softmax(torch.matmul(q.float(), k.float().transpose(1, 2).contiguous()) * scale, -1), v.float())
        assert float((out.float() - want).norm() / want.norm()) <= 1.5e-3
