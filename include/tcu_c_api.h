/*
 * C-ABI of the MI355X tile-kernel library: the boundary a host program (C, C++, Python
 * ctypes, a torch op) binds to. Plain pointers and sizes only; every pointer is a device
 * pointer owned by the caller and 16-byte aligned (the kernels move 16 bytes per lane);
 * nothing is allocated, freed or synchronised by the library;
 * work is enqueued on the hipStream_t passed as `stream` (NULL = the default stream).
 * Every function returns 0 on success or a negative tcu_status; tcu_last_error() gives the
 * message of the last failure on the calling thread. No function ever calls exit().
 *
 * Precedent in the reference: `extern "C" int kernel_entry(__half*, __half*, float*)` loaded
 * with ctypes (examples/python/gemm/entry.py:56-67, compile.py:129-137).
 */
#ifndef TCU_C_API_H_
#define TCU_C_API_H_

#ifdef __cplusplus
extern "C" {
#endif

typedef enum {
    TCU_OK = 0,
    TCU_ERR_INVALID_ARGUMENT = -1,  /* null or misaligned pointer, non-positive size, bad enum value */
    TCU_ERR_UNSUPPORTED_SHAPE = -2, /* shape not divisible by the tile / not instantiated */
    TCU_ERR_HIP = -3,               /* a HIP runtime call failed (message has the HIP error) */
    TCU_ERR_NO_DEVICE = -4,         /* no HIP device is available to this process */
    TCU_ERR_INCOMPLETE = -5         /* a single-launch kernel gave up a bounded wait; its outputs are invalid */
} tcu_status;

typedef enum { TCU_DTYPE_F32 = 0, TCU_DTYPE_F16 = 1 } tcu_dtype;

/* Which GEMM kernel to run. AUTO picks WAVE128 when M and N are multiples of 256 with more than 128 tiles of 256 x 256;
 * WAVE128 on the leading block of whole tiles plus PIPELINED on the remaining columns and rows (three launches on
 * disjoint parts of C, bit for bit the result of one launch) when M or N lie a little above such multiples and that
 * saves a round of workgroups; WAVE128 on the leading rows or columns that fill whole rounds of 256 workgroups plus a
 * kernel with smaller tiles (WAVE128_KSPLIT, WAVE128_NARROW or PIPELINED) on the rest of C when the last round would be
 * far from full (2560 x 8192: 320 tiles); WAVE128_KSPLIT and WAVE128_NARROW as described below; DIRECT wherever a cost model
 * expects it to be the shorter launch (few output tiles); RAGGED for outputs below 64 x 64 with K <= 48 or K >= 2^24; else
 * PIPELINED. Every shape made of whole 16 x 16
 * BaseTiles (M, N, K multiples of 16), the granularity of the reference's tile types, is accepted. */
typedef enum {
    TCU_GEMM_AUTO = 0,
    TCU_GEMM_GLOBAL_REG = 1, /* global -> register -> MFMA (README kernel of the reference) */
    TCU_GEMM_ALL_MEM = 2,    /* global -> LDS -> register -> MFMA, single stage */
    TCU_GEMM_PIPELINED = 3,  /* direct-to-LDS, double-buffered, 16x16x32 MFMA, 2 wavefronts per SIMD; M, N, K multiples
                                of 16; tiles of 256 x 256, 128 x 128 or 64 x 64 by a cost model of the rounds of
                                workgroups a launch takes; edge tiles (rows clamped, stores guarded, k tail zeroed in
                                LDS) where the shape is not whole tiles */
    TCU_GEMM_WAVE128 = 4,    /* same pipeline, 256 x 256 tile on 4 wavefronts (one per SIMD, 128 x 128 each),
                                accumulators in AGPRs; M, N and K multiples of 16 (edge tiles: rows clamped, stores
                                guarded, a partial last tile of K zero-filled in LDS); results identical to PIPELINED bit for bit, except where K is a
                                multiple of 16384 (rows a multiple of 32 KiB apart): there each XCD sums over K in
                                rotated order, which differs by f32 rounding */
    TCU_GEMM_TILE_PIPELINED = 5, /* the PIPELINED kernel composed from tile-library functors only (direct-to-LDS loader,
                                two-stage shared ring, ds_read_b128 operand tiles, gemm()); compile-time shapes:
                                4096^3, 1024^3, 512x768x192, 256x256x64; results identical to PIPELINED bit for bit */
    TCU_GEMM_RAGGED = 6,      /* run-time M, N, K in multiples of 16: MFMA operand tiles filled from global memory,
                                tiles beyond the edge skipped; the fallback for shapes the tiled kernels do not cover */
    TCU_GEMM_TILE_WAVE128 = 7, /* the WAVE128 kernel composed from tile-library functors only (direct-to-LDS loads dealt
                                a piece at a time, single-fragment LDS reads, gemm_scheduled() with accumulators pinned
                                in AGPRs); compile-time shapes: 4096^3, 1024^3, 512x768x192, 256x256x64; results
                                identical to WAVE128 and PIPELINED bit for bit */
    TCU_GEMM_WAVE128_KSPLIT = 8, /* 128 x 128 tile (128 x 96 where that fills the GPU better) on 4 wavefronts (one per SIMD)
                                that each own the whole tile over a quarter of every 128-wide step of K, partial tiles
                                added through LDS: for products with too few 256 x 256 tiles to fill the GPU (2048^3,
                                1552 x 1552 x 4096); K a multiple of 128 (AUTO runs it with a tail in K, any multiple of 16, too, where M and N exceed 64),
                                M and N multiples of 16 (edge tiles: rows clamped, stores guarded); the sum over K is
                                taken in four interleaved parts (differs from the other kernels by f32 rounding) */
    /* (10 is not assigned) */
    TCU_GEMM_DIRECT = 11,    /* tiles of 16 to 64 x 16 to 64 by a cost model, 8 wavefronts that split K and bring their own
                                chunks to LDS without barriers: for products with few output tiles (32 x 4096 x 4096,
                                256 x 256 x 8192); M, N, K multiples of 16; the sum over K is taken in eight interleaved
                                parts (differs from the other kernels by f32 rounding) */
    TCU_GEMM_WAVE128_NARROW = 9 /* the WAVE128 kernel with 256 x 128 workgroup tiles (a wavefront owns 128 x 64; three stages): for
                                products between the two above - too few 256 x 256 tiles to fill the GPU, too many
                                128 x 128 tiles for one round of WAVE128_KSPLIT (2048 x 2560 x 4096, 4096 x 2048 x 8192,
                                1552 x 3088 x 4096); M and N multiples of 16 (edge tiles: rows clamped, stores guarded),
                                K % 64 == 0; results identical to WAVE128 and PIPELINED bit for bit */
} tcu_gemm_algo;

/* Which back-to-back GEMM kernel to run (tcu_b2b_gemm_f16_algo). AUTO picks ROWS for many rows at N = 256; for longer N
 * STREAM where its expected time is below RESIDENT's; else RESIDENT, where it applies; TILE_RESIDENT for K = P = 64 with N in {128, 256}; else TILE_LIBRARY. */
typedef enum {
    TCU_B2B_AUTO = 0,
    TCU_B2B_TILE_LIBRARY = 1, /* composed from the 16x16 tile primitives, the reference kernel's structure */
    TCU_B2B_RESIDENT = 2,     /* A tile, 256-column blocks of B and C and the intermediate resident in LDS (K = P = 128,
                                 N % 256 == 0, M % 32 == 0); one round of loads per block */
    TCU_B2B_TILE_RESIDENT = 4, /* the RESIDENT kernel composed from tile-library functors only (direct-to-LDS loaders,
                                 16x16x32 operand tiles, the intermediate through a shared tile); compile-time sizes:
                                 K = P = 128 with N in {256, 1024, 2048} (results identical to RESIDENT bit for bit) and
                                 K = P = 64 with N in {128, 256}; M % 32 == 0 */
    /* (5 is not assigned) */
    TCU_B2B_STREAM = 6,       /* for longer N and many rows: blocks of 64 columns of B and C pass once through a ring in LDS for 128 or
                                 256 rows per workgroup, every wavefront owning 32 of them (A fragments and the intermediate in
                                 registers); K = P = 128, N % 256 == 0, N >= 512, M % 32 == 0; agrees with RESIDENT up to the
                                 order of the f32 sums inside an MFMA */
    TCU_B2B_ROWS = 3          /* for many rows (AUTO from M x batch = 32768): N = 256, K = P = 128, M % 64 == 0; a
                                 workgroup keeps B and C in LDS and walks over blocks of 256 rows, every wavefront owning
                                 64 rows (A fragments from global memory, the intermediate stays in registers); agrees
                                 with RESIDENT up to the order of the f32 sums inside an MFMA */
} tcu_b2b_algo;

/* Layout of V in tcu_flash_attn_fwd_f16. */
typedef enum {
    TCU_V_COL_MAJOR = 0, /* V stored [P, N] per batch item: the reference op's convention */
    TCU_V_ROW_MAJOR = 1  /* V stored [N, P] per batch item: the usual [seq, head_dim] */
} tcu_v_layout;

/* Which attention kernel to run (tcu_flash_attn_fwd_f16_algo). AUTO picks the kernel with the shortest expected time among KEYS
 * and, for a row-major V, WAVE64_K32 (with at least 256 whole blocks of 256 queries and N >= 320, or 192 and N >= 1024, unless
 * MFMA32_FUSED is expected to be clearly shorter), at head size 128 also WAVE64 (128 to 191 such blocks and N >= 1024), and
 * MFMA32_FUSED otherwise; for a column-major V (head size 128) WAVE64_K32 under the same conditions and WAVE64 otherwise (it
 * takes every M % 64 == 0 and N % 64 == 0). */
typedef enum {
    TCU_ATTN_AUTO = 0,
    TCU_ATTN_TILE_LIBRARY = 1, /* composed from the 16x16 tile primitives, like the reference kernel */
    TCU_ATTN_MFMA32 = 2,       /* 32x32x16 MFMA, transposing LDS reads, direct-to-LDS K/V (row-major V only) */
    TCU_ATTN_MFMA32_FUSED = 3, /* MFMA32 with the softmax of block j+1 computed speculatively under the MFMAs of
                                  block j: faster when row maxima settle early, up to ~10 % slower than MFMA32
                                  when they keep growing along the keys; same results up to rounding */
    TCU_ATTN_WAVE64 = 4,       /* 4 wavefronts x 64 queries, one per SIMD: half the LDS traffic per MFMA, all matrix
                                  instructions placed by hand, softmax of 32 keys interleaved with the MFMAs of the
                                  neighbouring 32; either V layout, head size 128, M % 64 == 0 (wavefronts of the
                                  last workgroup whose 64 queries lie beyond M idle), N % 64 == 0, N * 256 < 2^32 */
    TCU_ATTN_TILE_WAVE64 = 5,  /* the WAVE64 kernel composed from tile-library functors only (matrix instructions placed
                                  one by one with ScheduledGemm, interleaved 5-stage shared rings, fragment reads issued
                                  ahead with SharedToRegPieces / SharedToRegTrPieces); compile-time sequence lengths:
                                  (M, N) in {(2048, 2048), (512, 1024), (256, 640), (256, 320)}, head size 128, row-major
                                  V; results identical to WAVE64 bit for bit */
    TCU_ATTN_WAVE64_K32 = 6,   /* the WAVE64 design on v_mfma_f32_16x16x32_f16 (tile-library functors; twice the matrix
                                  instructions, each contracting 32 indices: the chip sustains a higher clock on them),
                                  launched as one workgroup per CU that takes its blocks of 256 queries one after the
                                  other and fetches the next one's first operands under the last steps of the current;
                                  head size 128 with either V layout or head size 64 with a row-major V, M % 64 == 0
                                  (wavefronts of a head's last block whose 64 queries lie beyond M idle), N % 64 == 0,
                                  N >= 320; results equal to WAVE64 (MFMA32_FUSED at head size 64) up to the
                                  summation order inside a matrix instruction */
    /* (7 is not assigned) */
    TCU_ATTN_KEYS = 8          /* a workgroup per 64 queries whose 4 wavefronts split the keys (and, through a workspace,
                                  several workgroups per 64 queries: tcu_flash_attn_fwd_f16_ws): for launches with few
                                  query blocks; M % 64 == 0, N % 64 == 0, head size 128 with either V layout or 64 with a
                                  row-major V; results equal to the others up to rounding and the order of the sums */
} tcu_attn_algo;

/* Which LSTM step kernel to run (tcu_lstm_f16_algo). Every B, I, H in multiples of 16 is accepted: AUTO runs a step kernel
 * of its own whose wavefronts split the columns (kernels/lstm_direct.hpp) unless W or an activation exceeds 4 GiB, then
 * STREAMING, TILE_LIBRARY or RAGGED, the first that takes the shape. */
typedef enum {
    TCU_LSTM_AUTO = 0,
    TCU_LSTM_TILE_LIBRARY = 1, /* composed from the 16x16 tile primitives, single LDS stage; (I, H) in {(1024,1024),
                                  (128,128), (64,128)}, B % 64 == 0 */
    TCU_LSTM_STREAMING = 2,    /* 32x32x16 MFMA, multi-stage direct-to-LDS ring, k split over two wavefront groups;
                                  I % 128 == 0, H % 128 == 0, B % 64 == 0 */
    TCU_LSTM_RAGGED = 3        /* run-time B, I, H in multiples of 16: MFMA operand tiles filled from global memory */
} tcu_lstm_algo;

/* Library version (major * 10000 + minor * 100 + patch). */
int tcu_version(void);

/* Message of the last error raised on the calling thread ("" if none). */
const char* tcu_last_error(void);

/* Name (as compiled) of the kernel that the calling thread's last launch through this library ran, or of the one `back` launches
 * before it; "" beyond the last four. What a call that leaves the choice to the library has run. */
const char* tcu_recent_kernel(int back);

/* Number of HIP devices visible, or a negative tcu_status. */
int tcu_device_count(void);

/*
 * C[M, N] = A[M, K] · B.  A row-major f16; B column-major f16 (stored as [N, K]); C row-major,
 * out_dtype f32 or f16; f32 accumulation.
 * Replaces the launches in the reference's examples/cpp/01_gemm/01_gemm_global_reg/main.cu:59-63
 * and examples/cpp/01_gemm/02_gemm_all_mem/main.cu:54-72 (kernels gemm.hpp:65-92 / :103-155), and
 * the ctypes entry examples/python/gemm/entry.py:56-67.
 */
int tcu_gemm_f16(const void* A, const void* B, void* C, int M, int N, int K, int out_dtype, int algo, void* stream);

/*
 * tcu_gemm_f16 (TCU_GEMM_AUTO) for products with few output tiles and a long K, where one workgroup per output
 * tile leaves most of the chip idle or short of work (e.g. 1024 x 1024 x 16384, 2048 x 2048 x 32768): K is split into
 * ranges multiplied by different workgroups (the WAVE128_KSPLIT kernel with 128 x 128 tiles, or the WAVE128 kernel where
 * those tiles fill the chip by themselves; f32 partial products into `workspace`, [splits, M, N]) and a second kernel
 * adds the partial products. tcu_gemm_workspace_bytes(M, N, K) is the workspace
 * this takes, or 0 when the product is not split (more than 128 tiles of 256 x 256, M or N not multiples of 16,
 * less than 512 of K per range, or the unsplit kernel expected to be as fast): then, and when `workspace` is NULL,
 * the call is tcu_gemm_f16 with TCU_GEMM_AUTO. The workspace (16-byte aligned device
 * memory) is the caller's and free to reuse once the work enqueued here has run. Where TCU_GEMM_DIRECT is expected to be
 * faster than the split (short M or N) the call runs that kernel and leaves the workspace alone; tcu_gemm_uses_workspace()
 * is 0 there, so that a caller that would allocate one need not. Results differ from the unsplit
 * product by the order of the f32 summation only. No counterpart in the reference, whose GEMM examples fix one
 * workgroup per output tile (examples/cpp/01_gemm/02_gemm_all_mem/main.cu:54-72).
 */
unsigned long long tcu_gemm_workspace_bytes(int M, int N, int K);
int tcu_gemm_uses_workspace(int M, int N, int K);
int tcu_gemm_f16_ws(const void* A, const void* B, void* C, int M, int N, int K, int out_dtype, void* workspace,
                    unsigned long long workspace_bytes, void* stream);

/*
 * D[b, M, P] = f16(A[b, M, K] · B[b]) · C[b].  A row-major; B column-major [K, N] (stored [N, K]);
 * C column-major [N, P] (stored [P, N]); D row-major, f32 or f16. The [M, N] intermediate
 * never leaves the chip.
 * Replaces run_fused_gemm / KeFusedGemm of the reference's
 * examples/cpp/02_fused_two_gemms/fused_gemm.cu:86-113 and fused_gemm.hpp:107-181.
 */
int tcu_b2b_gemm_f16(const void* A, const void* B, const void* C, void* D, int M, int N, int K, int P, int batch,
                     int out_dtype, void* stream);

/* tcu_b2b_gemm_f16 with an explicit kernel choice (tcu_b2b_algo); same arguments otherwise. */
int tcu_b2b_gemm_f16_algo(const void* A, const void* B, const void* C, void* D, int M, int N, int K, int P, int batch,
                          int out_dtype, int algo, void* stream);

/*
 * O[b, M, P] = softmax(scale · Q[b, M, K] · K[b]) · V[b], f16 in / f16 out, f32 softmax
 * statistics. Q row-major; keys column-major [K, N] (stored [N, K]); V per v_layout.
 * Replaces run_flash_attention / custom_flash_attention_op of the reference's
 * src/kernels/flash_attn.cu:314-456 (the body of torch.ops.tiledcuda.flash_attention_fwd).
 * The reference computes with scale = 1; pass 1.0f for that behaviour.
 * Precision of the tuned kernels (every algo but TCU_ATTN_TILE_LIBRARY): Q is multiplied by scale * log2(e) and
 * rounded to f16 before the score products, so each product term of a logit carries a relative error of 2^-11 and
 * |q * scale * 1.4427| must stay below 65504. Measured maximum output error for N(0,1) values: 1.2e-4 at logits up
 * to +-5, 1.7e-3 at +-14, 4.4e-3 at +-29 (the tile-library kernel, which scales the f32 scores like the reference:
 * 1.4e-4, 9.6e-4, 9.9e-4).
 */
int tcu_flash_attn_fwd_f16(const void* Q, const void* K, const void* V, void* O, int batch, int M, int N, int Kdim,
                           int P, float scale, int v_layout, void* stream);

/* tcu_flash_attn_fwd_f16 with an explicit kernel choice (tcu_attn_algo); same arguments otherwise. */
int tcu_flash_attn_fwd_f16_algo(const void* Q, const void* K, const void* V, void* O, int batch, int M, int N,
                                int Kdim, int P, float scale, int v_layout, int algo, void* stream);

/*
 * tcu_flash_attn_fwd_f16 for calls with few query blocks and many keys (a short block of new queries against a long
 * cache), where one workgroup per 64 queries leaves most of the chip idle: the keys are split over several workgroups,
 * their f32 partial outputs go to `workspace`, and a second kernel adds them. tcu_flash_attn_workspace_bytes(...) is the
 * workspace this takes, or 0 when the keys are not split: then, and when `workspace` is NULL, the call is
 * tcu_flash_attn_fwd_f16. The workspace (16-byte aligned device memory) is the caller's and free to reuse once the work
 * enqueued here has run; a graph that captured the call uses it at every replay. Results differ from the unsplit ones by
 * rounding and the order of the f32 sums only.
 */
unsigned long long tcu_flash_attn_workspace_bytes(int batch, int M, int N, int Kdim, int P, int v_layout);
int tcu_flash_attn_fwd_f16_ws(const void* Q, const void* K, const void* V, void* O, int batch, int M, int N, int Kdim, int P,
                              float scale, int v_layout, void* workspace, unsigned long long workspace_bytes, void* stream);

/*
 * Fused LSTM layer over T steps. x [T, B, I] f16; W [4H, I+H] f16 row-major, gate rows in the
 * order i, f, g, o, columns concat(x_t, h_{t-1}); bias [4H] f16; h0 [B, H] f16 or NULL (zeros);
 * c0 [B, H] f32 or NULL (zeros); h_all [T, B, H] f16 receives every h_t; c_out [B, H] f32
 * receives c_T (it is also the running cell state, so it must not alias c0 unless c0 == c_out).
 * One kernel per step (gate GEMM fused with the cell update). B, I and H must be multiples of 16 (whole tiles) and
 * T * B fit in 31 bits.
 * The reference snapshot has no LSTM entry (Makefile:3 names a test only).
 */
int tcu_lstm_f16(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                 void* c_out, int T, int B, int I, int H, void* stream);

/* tcu_lstm_f16 with an explicit kernel choice (tcu_lstm_algo); same arguments otherwise. */
int tcu_lstm_f16_algo(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                      void* c_out, int T, int B, int I, int H, int algo, void* stream);

/*
 * tcu_lstm_f16 with the input half of the gates hoisted out of the time loop: x · W[:, :I]^T for all T steps is one
 * large GEMM into `workspace` ([T, B, 4H] f32), and each step then streams only h_{t-1} and W[:, I:] (half the bytes
 * of a step, which is what bounds it). Same arguments and results (up to the order of the f32 summation) as
 * tcu_lstm_f16. `workspace` is device memory of at least tcu_lstm_workspace_bytes(T, B, I, H) bytes, 16-byte aligned,
 * owned by the caller and free to reuse once the work enqueued here has run. tcu_lstm_workspace_bytes returns 0 for
 * shapes this path does not take (it needs I % 128 == 0, H % 128 == 0, B % 64 == 0 and T * B a multiple of 256);
 * tcu_lstm_f16_ws then fails with TCU_ERR_UNSUPPORTED_SHAPE. No counterpart in the reference (it has no LSTM).
 */
unsigned long long tcu_lstm_workspace_bytes(int T, int B, int I, int H);
/* 1 where tcu_lstm_f16_ws is expected to be faster than tcu_lstm_f16 (long inputs: I of 2048 and more at most sizes), else 0:
 * the Python and torch entries take a workspace for it there. */
int tcu_lstm_uses_workspace(int T, int B, int I, int H);
int tcu_lstm_f16_ws(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                    void* c_out, int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes,
                    void* stream);

/*
 * The LSTM layer in two launches: the input half of the gates of all steps as one GEMM into `workspace` (f32, as in
 * tcu_lstm_f16_ws), then the whole time loop as one launch that keeps the recurrent weights in registers; a layer of which these
 * pre-activations would take more than 256 MiB runs in parts of so many steps, one after the other. T >= 2, B, I and H in
 * multiples of 16, H <= 1024, B <= 2048 (tcu_lstm_layer_workspace_bytes returns 0 for shapes this path does not take). Same
 * arguments and results (up to the order of the f32 summation) as tcu_lstm_f16; nothing is asked of the GPU: workgroups that are
 * not resident are stood in for by those that are, and every wait is for a workgroup that runs.
 * `workspace`: device memory of at least tcu_lstm_layer_workspace_bytes(T, B, I, H) bytes, 16-byte aligned, owned by the caller
 * and free to reuse once the work enqueued here has run; its first 4 KiB are synchronisation words, cleared by the call. Calls
 * that may overlap in time need a workspace each. Where x, h0 or c0 lies inside h_all the step kernels of tcu_lstm_f16 run instead.
 * No counterpart in the reference (it has no LSTM).
 */
unsigned long long tcu_lstm_layer_workspace_bytes(int T, int B, int I, int H);
/* 1 where it is expected to be faster than tcu_lstm_f16 and tcu_lstm_f16_ws (about 5 steps and more, up to 256 rows), else 0: the
 * Python and torch entries take a workspace for it there. */
int tcu_lstm_uses_layer(int T, int B, int I, int H);
int tcu_lstm_f16_layer(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all, void* c_out,
                       int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes, void* stream);
/* The same with at most `max_workgroups` workgroups, of which those that have waited `takeover_us` stand in for the others, and with
 * waits that are given up after `max_tries` polls (outputs that depend on one are NaN from that step on): for tests of a layer that
 * does not get the GPU it has room for. */
int tcu_lstm_f16_layer_limited(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                               void* c_out, int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes,
                               int max_workgroups, int takeover_us, int max_tries, void* stream);

/*
 * The LSTM layer with the whole time loop in ONE launch, for the large-hidden-size case where a step is bound by
 * streaming the recurrent weights and by the cost of a dependent launch (H in {256, 512, 768, 1024}, I % 64 == 0, B % 32 == 0, B <= 256,
 * T * B % 256 == 0; a device of 256 CUs in 8 XCDs). As in tcu_lstm_f16_ws the input half of the gates of all steps is
 * one GEMM into the workspace - here with its f32 sums rounded once to f16 (half the bytes to write and read back; the
 * gates' pre-activations then carry a relative error of 2^-11 on that half, far inside the layer's 1e-2 tolerance) -;
 * the recurrence then runs weight-stationary: every XCD keeps a copy of W[:, I:] in the registers of its 32 CUs and owns
 * 32 batch rows, and h_t is exchanged between those CUs through the XCD's L2 only.
 * Same arguments as tcu_lstm_f16_ws; results equal to its up to that rounding and the order of the f32 summation. `workspace`: device memory of
 * at least tcu_lstm_persistent_workspace_bytes(T, B, I, H) bytes (0 = shape not supported), 128-byte aligned (the step
 * counters sit in cache lines of their own), owned by the caller; its first 4 KiB are synchronisation words, cleared by
 * the call.
 * The launch needs all of its 256 workgroups resident at the same time, i.e. a GPU that is not occupied by another
 * kernel for long; its waits are bounded (2 s; TCU_LSTM_PERSISTENT_SPIN_US in the environment overrides, in
 * microseconds), and every workgroup exits normally when a wait expires. The call itself is asynchronous like all
 * others; tcu_lstm_persistent_status(workspace, stream) synchronises the stream and returns TCU_OK, or
 * TCU_ERR_INCOMPLETE when a wait expired (h_all and c_out are then invalid: run tcu_lstm_f16_ws instead).
 * No counterpart in the reference (it has no LSTM).
 */
unsigned long long tcu_lstm_persistent_workspace_bytes(int T, int B, int I, int H);
int tcu_lstm_f16_persistent(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                            void* c_out, int T, int B, int I, int H, void* workspace,
                            unsigned long long workspace_bytes, void* stream);
int tcu_lstm_persistent_status(const void* workspace, void* stream);

/*
 * tcu_lstm_f16_ws for callers that can neither allocate device memory nor bring a workspace: code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc. No counterpart in the reference. The [T, B, 4H] f32
 * gate pre-activations go to a buffer of tcu_lstm_noalloc_max_bytes() (64 MiB) that is part of the library's device
 * image (each GPU the library is used on holds its own copy until the process ends); the call allocates and frees
 * nothing. Same arguments, shape rules and results as tcu_lstm_f16_ws; shapes with T * B * 4H * 4 bytes above the
 * maximum fail with TCU_ERR_UNSUPPORTED_SHAPE (the C5 layer, T 16 x B 256 x H 1024, fits exactly). Every call on one
 * GPU uses that GPU's one buffer: calls whose work overlaps in time on one GPU (different streams, or different host
 * threads) race on it; calls on one stream are ordered and safe. Nothing in the buffer has to start at zero (the
 * projection GEMM overwrites every element a step kernel reads), and it keeps the last call's contents.
 */
unsigned long long tcu_lstm_noalloc_max_bytes(void);
int tcu_lstm_f16_noalloc(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                         void* c_out, int T, int B, int I, int H, void* stream);

/* How tcu_scatter_nd combines an update with the data it lands on. */
typedef enum {
    TCU_SCATTER_ASSIGN = 0, /* data[...] = update: what the reference's test checks (tests/python/test_scatter_nd.py:47-56) */
    TCU_SCATTER_ADD = 1     /* data[...] += update, atomically: what the reference's kernel body does (src/kernels/scatter_nd.cu:48-51) */
} tcu_scatter_mode;

/*
 * data[idx[i,0], ..., idx[i,k-1], :] (= | +=) updates[i, :] for the n index rows of `indices`.
 * data: device tensor of `rank` dimensions `data_dims` (HOST array of rank int64 values), row-major, dtype f32 or
 * f16; indices: device int64 [n, k], k <= rank <= 8; updates: device [n, prod(data_dims[k:])], same dtype as data.
 * Rows with a component outside [0, data_dims[c]) are skipped; if skipped_rows (device uint32, may be NULL) is
 * given, it is incremented once per skipped row (the caller zeroes it). With TCU_SCATTER_ASSIGN, duplicate index
 * rows leave one of their updates (unspecified which).
 * Replaces custom_scatter_op / scatter_nd<T> of the reference's src/kernels/scatter_nd.cu:57-120 (the body of
 * torch.ops.tiledcuda.scatter_nd, src/torch_bind.cc:9); unlike it, no device memory is allocated per call.
 */
int tcu_scatter_nd(void* data, const void* updates, const void* indices, const long long* data_dims, int rank,
                   long long n, int k, int dtype, int mode, void* skipped_rows, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* TCU_C_API_H_ */
