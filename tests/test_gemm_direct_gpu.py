"""The GEMM kernel whose wavefronts split K without barriers (algo "direct", AUTO's choice for few output tiles), at the sizes
where its tiles, its chunks of K and its rings end. Against the oracle; relative tolerance of the layer's other tests (1e-3 of
a result rounded to f16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
REL_TOL = 1e-3


@pytest.mark.parametrize("M,N,K", [(16, 16, 16), (16, 16, 64), (16, 48, 80), (48, 16, 496), (32, 4080, 512), (16, 4096, 528),  # 1 wide
                                   (16, 64, 4096), (32, 2064, 2096), (48, 4112, 1040), (64, 4096, 1552),  # rings of 2 to 4 chunks
                                   (112, 4096, 576), (4112, 48, 592), (272, 400, 1088), (528, 1040, 608), (256, 4096, 1072),
                                   (2064, 48, 304), (16, 8208, 48), (208, 464, 1008)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_gemm_direct(tcu, oracle, device, M, N, K, out_dtype):
    import torch

    print(f"gemm direct {M}x{N}x{K} {out_dtype}", flush=True)
    dt = torch.float32 if out_dtype == "f32" else torch.float16
    A = oracle.fill_uniform(M * K, 31 + M).reshape(M, K)
    Bt = oracle.fill_uniform(N * K, 37 + N).reshape(N, K)
    # rows beyond the operands hold NaN: a product that took one in would show it
    a = torch.full((M + 64, K), float("nan"), dtype=torch.float16, device=device)
    b = torch.full((N + 64, K), float("nan"), dtype=torch.float16, device=device)
    a[:M], b[:N] = torch.from_numpy(A).to(device), torch.from_numpy(Bt).to(device)
    guard = torch.full((M + 2, N), -7.0, dtype=dt, device=device)
    tcu.gemm(a[:M], b[:N], out=guard[1:M + 1], algo="direct")
    torch.cuda.synchronize()
    assert oracle.max_rel_err(guard[1:M + 1].float().cpu().numpy(), oracle.gemm(A, Bt)) <= REL_TOL
    assert torch.all(guard[0] == -7.0) and torch.all(guard[M + 1] == -7.0)


def test_gemm_direct_leaves_the_workspace(tcu, device):
    """A short product that could be split: AUTO runs this kernel, with or without a workspace, which stays untouched."""
    import torch

    M, N, K = 256, 256, 8192
    a = torch.randn(M, K, device=device).half()
    b = torch.randn(N, K, device=device).half()
    assert not tcu.lib().tcu_gemm_uses_workspace(M, N, K)
    ws = torch.full((tcu.gemm_workspace_bytes(M, N, K),), 0xFF, dtype=torch.uint8, device=device)
    want = tcu.gemm(a, b, algo="direct")
    assert torch.equal(tcu.gemm(a, b, workspace=ws), want) and torch.equal(tcu.gemm(a, b), want)
    assert bool((ws == 0xFF).all())


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 1040), (1808, 1808, 1552), (2064, 1040, 1072), (1552, 1552, 1600),
                                   (1536, 1536, 1648), (1296, 1296, 4112), (1040, 1040, 8304), (1936, 1984, 1136)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_gemm_tail_of_the_k_splitting_kernel(tcu, oracle, device, M, N, K, out_dtype):
    """AUTO's choice for one round of 128 x 128 (or 128 x 96) tiles where K is not a multiple of 128: tails of 16 to 112 columns, odd
    and even numbers of steps, whole and edge tiles; what lies behind the operands' last rows is NaN."""
    import torch

    print(f"gemm k tail {M}x{N}x{K} {out_dtype}", flush=True)
    dt = torch.float32 if out_dtype == "f32" else torch.float16
    A = oracle.fill_uniform(M * K, 31 + M).reshape(M, K)
    Bt = oracle.fill_uniform(N * K, 37 + N).reshape(N, K)
    a = torch.full((M + 16, K), float("nan"), dtype=torch.float16, device=device)
    b = torch.full((N + 16, K), float("nan"), dtype=torch.float16, device=device)
    a[:M], b[:N] = torch.from_numpy(A).to(device), torch.from_numpy(Bt).to(device)
    guard = torch.full((M + 2, N), -7.0, dtype=dt, device=device)
    tcu.gemm(a[:M], b[:N], out=guard[1:M + 1])
    torch.cuda.synchronize()
    rows = sorted(set(list(range(0, 32)) + list(range(M - 32, M))))
    assert oracle.max_rel_err(guard[1:M + 1].float().cpu().numpy()[rows], oracle.gemm(A[rows], Bt)) <= REL_TOL
    want = tcu.gemm(a[:M], b[:N], out_dtype=torch.float32, algo="pipelined").cpu().numpy()
    assert oracle.max_rel_err(guard[1:M + 1].float().cpu().numpy(), want) <= REL_TOL
    assert torch.all(guard[0] == -7.0) and torch.all(guard[M + 1] == -7.0)


@pytest.mark.parametrize("M,N,batch", [(32, 512, 520), (96, 1024, 260), (2080, 768, 16), (65536, 512, 1), (1600, 1024, 16), (288, 2048, 150)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_b2b_streamed_weights(tcu, device, M, N, batch, out_dtype):
    """AUTO for long N (its choice is the streaming kernel with (2080, 768, 16), (65536, 512, 1) and (1600, 1024, 16), the resident
    one with the others): 8 to 32 blocks of columns, many and few items. Against the kernel with 32 rows per workgroup: the same f16
    intermediate up to the order of its f32 sums (an ulp of f16, 2^-11, in few elements), then f32 sums of N terms; a tenth of
    that for the whole."""
    import torch

    print(f"b2b stream {M}x{N} batch {batch} {out_dtype}", flush=True)
    dt = torch.float32 if out_dtype == "f32" else torch.float16
    gen = torch.Generator(device=device)
    gen.manual_seed(M + N)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=device).mul_(0.1).half()
    a, b, c = normal(batch, M, 128), normal(batch, N, 128), normal(batch, 128, N)
    guard = torch.full((batch * M + 2, 128), -7.0, dtype=dt, device=device)
    out = tcu.b2b_gemm(a, b, c, out=guard[1:-1].view(batch, M, 128))
    want = tcu.b2b_gemm(a, b, c, out_dtype=dt, algo="resident").float()
    assert ((out.float() - want).norm() / want.norm()).item() <= (5e-5 if dt == torch.float32 else 2.0 ** -12)
    assert torch.all(guard[0] == -7.0) and torch.all(guard[-1] == -7.0)


@pytest.mark.parametrize("M,N", [(16, 16), (48, 80)])
def test_gemm_auto_takes_every_k(tcu, device, M, N):
    """AUTO accepts a K beyond the 32-bit offsets of the tiled kernels where it has one that counts in 64 bits (outputs below
    64 x 64): operands of zeros with a few small integers, some in the last columns, whose products are exact."""
    import torch

    K = (1 << 24) + 16
    print(f"gemm {M}x{N}x{K}", flush=True)
    gen = torch.Generator(device=device)
    gen.manual_seed(M)
    cols = torch.cat((torch.randint(K, (500,), generator=gen, device=device), torch.arange(K - 12, K, device=device))).unique()
    a, b = (torch.zeros(rows, K, dtype=torch.float16, device=device) for rows in (M, N))
    for t in (a, b):
        t[:, cols] = torch.randint(-3, 4, (t.shape[0], cols.numel()), generator=gen, device=device).half()
    want = a[:, cols].float() @ b[:, cols].float().t()
    got = tcu.gemm(a, b, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and bool(want.any())


@pytest.mark.parametrize("M,N,batch,auto", [(32, 512, 520, False), (96, 1024, 260, False), (288, 2048, 150, False), (32, 512, 1, False),
                                            (160, 4096, 3, False), (2080, 768, 16, True), (65536, 512, 1, True), (1600, 1024, 16, True),
                                            (8128, 2048, 5, True)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_b2b_stream_by_name(tcu, oracle, device, M, N, batch, auto, out_dtype):
    """The weight-streaming kernel by name with workgroups of 128 rows (the first five, and 1600 x 16) and of 256, most or part of which
    lie beyond M, rings of 8 to 64 blocks; against the oracle on the first and last rows of the first and last item, in the
    tolerance of the other kernels' tests, with guard rows around the output. `auto`: this is AUTO's choice, bit for bit."""
    import torch

    print(f"b2b stream by name {M}x{N} batch {batch} {out_dtype}", flush=True)
    dt = torch.float32 if out_dtype == "f32" else torch.float16
    gen = torch.Generator(device=device)
    gen.manual_seed(M + N)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device=device).mul_(0.1).half()
    a, b, c = normal(batch, M, 128), normal(batch, N, 128), normal(batch, 128, N)
    guard = torch.full((batch * M + 2, 128), -7.0, dtype=dt, device=device)
    out = tcu.b2b_gemm(a, b, c, out=guard[1:-1].view(batch, M, 128), algo="stream")
    torch.cuda.synchronize()
    rows, items = sorted({*range(min(M, 40)), *range(max(0, M - 40), M)}), sorted({0, batch - 1})
    pick = lambda t: np.ascontiguousarray(t[items].cpu().numpy())
    want = oracle.b2b_gemm(np.ascontiguousarray(pick(a)[:, rows]), pick(b), pick(c))
    assert oracle.max_rel_err(out[items][:, rows].float().cpu().numpy(), want, eps=1.0) <= REL_TOL
    assert torch.all(guard[0] == -7.0) and torch.all(guard[-1] == -7.0)
    if auto:
        assert torch.equal(out, tcu.b2b_gemm(a, b, c, out_dtype=dt))


@pytest.mark.parametrize("M,N,K", [(48, 2064, 304), (112, 1040, 80), (80, 4112, 592), (208, 2064, 1040)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_gemm_direct_wide_tiles(tcu, oracle, device, M, N, K, out_dtype):
    """The tiles of 32 x 16 (first two) and 64 x 32, which the shapes of the first test do not select, with partial last tiles."""
    test_gemm_direct(tcu, oracle, device, M, N, K, out_dtype)


@pytest.mark.parametrize("M,N,K", [(384, 448, 128), (112, 1600, 144), (3664, 640, 1472), (48, 11968, 1296), (2064, 48, 8208)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_gemm_auto_around_the_direct_kernel(tcu, oracle, device, M, N, K, out_dtype):
    """AUTO where its choice lies close to another kernel's: short K, one more round of tiles, tails of K with most of a tile beyond
    M or N. Against the oracle on the first and last rows, and everywhere against the kernel without LDS."""
    import torch

    print(f"gemm auto {M}x{N}x{K} {out_dtype}", flush=True)
    dt = torch.float32 if out_dtype == "f32" else torch.float16
    A = oracle.fill_uniform(M * K, 31 + M).reshape(M, K)
    Bt = oracle.fill_uniform(N * K, 37 + N).reshape(N, K)
    a, b = torch.from_numpy(A).to(device), torch.from_numpy(Bt).to(device)
    got = tcu.gemm(a, b, out_dtype=dt).float().cpu().numpy()
    rows = sorted({*range(24), *range(M - 24, M)})
    assert oracle.max_rel_err(got[rows], oracle.gemm(A[rows], Bt)) <= REL_TOL
    assert oracle.max_rel_err(got, tcu.gemm(a, b, out_dtype=torch.float32, algo="ragged").cpu().numpy()) <= REL_TOL


@pytest.mark.parametrize("M,N,K,splits", [(224, 352, 16384, 16), (192, 384, 16384, 32), (16, 32, 32768, 64), (464, 592, 8192, 8)])
@pytest.mark.parametrize("out_dtype", ["f32", "f16"])
def test_gemm_split_k_in_many_ranges(tcu, oracle, device, M, N, K, splits, out_dtype):
    """Products that are split over K into 8 to 64 ranges rather than sent to the kernel of this file: the workspace's bytes past
    the stated size stay untouched, those before it do not; against the oracle on 32 rows and the unsplit call."""
    import torch

    print(f"gemm split-K {M}x{N}x{K} {splits} {out_dtype}", flush=True)
    dt = torch.float32 if out_dtype == "f32" else torch.float16
    need = tcu.gemm_workspace_bytes(M, N, K)
    assert need == splits * M * N * 4 and tcu.lib().tcu_gemm_uses_workspace(M, N, K)
    A = oracle.fill_uniform(M * K, 131 + M).reshape(M, K)
    Bt = oracle.fill_uniform(N * K, 137 + N).reshape(N, K)
    a, b = torch.from_numpy(A).to(device), torch.from_numpy(Bt).to(device)
    ws = torch.full((need + 4096,), 0xFF, dtype=torch.uint8, device=device)
    got = tcu.gemm(a, b, out_dtype=dt, workspace=ws).float().cpu().numpy()
    assert bool((ws[need:] == 0xFF).all()) and not bool((ws[:need] == 0xFF).all())
    rows = sorted({*range(min(M, 16)), *range(M - 16, M)})
    assert oracle.max_rel_err(got[rows], oracle.gemm(A[rows], Bt)) <= REL_TOL
    assert oracle.max_rel_err(got, tcu.gemm(a, b, out_dtype=torch.float32, workspace=False).cpu().numpy()) <= REL_TOL


@pytest.mark.parametrize("M,N,K,tile,whole", [(1040, 1040, 1040, (96, 64), False),   # rows 80 of 96, columns 16 of 64, K 16 of 64
                                              (1040, 1024, 1088, (96, 64), False), (1312, 784, 624, (96, 64), False),
                                              (1312, 832, 272, (96, 64), False), (288, 3328, 256, (96, 64), True),
                                              (2064, 1040, 1072, (96, 96), False),   # rows 48 of 96, columns 80, K 48 of 64
                                              (1424, 1552, 1040, (96, 96), False), (1056, 1824, 1600, (96, 96), True)])
@pytest.mark.parametrize("out_dtype", ["float16", "float32"])
def test_ring_tiles_with_96_rows(tcu, device, M, N, K, tile, whole, out_dtype):
    """Products that AUTO gives the ring with 96 x 64 or 96 x 96 tiles where the results are f16, and other tiles where they are f32:
    every element of the output and what lies behind it, f32 sums in another order (1e-6 of the norm), rounded to f16 (2^-11) where
    the output is."""
    import torch

    print(f"gemm ring 96 {M}x{N}x{K} {out_dtype}", flush=True)
    gen = torch.Generator(device=device)
    gen.manual_seed(M + K)
    a, b = (torch.rand(*s, generator=gen, device=device).mul_(2).sub_(1).half() for s in ((M, K), (N, K)))
    dtype = getattr(torch, out_dtype)
    buf = torch.full((M * N + 4096,), 7.0, dtype=dtype, device=device)
    tcu.gemm(a, b, out=buf[:M * N].view(M, N), workspace=False)
    kernel = tcu.lib().tcu_recent_kernel(0).decode()
    assert (f"PipelinedGemmTraitsILi{tile[0]}ELi{tile[1]}E" in kernel) == (out_dtype == "float16"), kernel
    assert out_dtype == "float32" or (f"__halfLb{int(not whole)}E" in kernel), kernel  # (with edges or without)
    want = a.double() @ b.double().t()
    err = float((buf[:M * N].view(M, N).double() - want).norm() / want.norm())
    assert err <= (1e-6 if dtype == torch.float32 else 2 ** -11)
    assert bool((buf[M * N:] == 7.0).all())
