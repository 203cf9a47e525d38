// gemm_bs.hip -- FP8 GEMMs with fp32 scales behind the opus_gemm_kargs ABI.
//
//   block-scale (DeepSeek):  C[b,m,n] = sum_g P_g[m,n] * SFA[g, m] * SFB(g, n)
//       P_g = sum over the 128-wide K group g of A*B (fp32 from the MFMA)
//       SFB(g, n) = SFB[n/128, g] (GROUP_N 128) or SFB[g, n] (GROUP_N 1)
//       acc = fmaf(P_g, SFA*SFB, acc) per group, in K order
//       (opus_gemm/block_scale_gemm/README.md:7-26, scale_c_tile in
//        opus_gemm_dist/opus_gemm_mem_gemm_a2a/include/opus_gemm_utils.cuh:76-96)
//   per-tensor (fp8_gemm):  C = (sfa[0] * sfb[0]) * sum_k A*B, one fp32 chain
//
// A [batch, M, K] and B [batch, N, K] are row-major E4M3 (B is K-major, not
// preshuffled), K % 128 == 0, M and N arbitrary (rows past M/N load as zero
// through the buffer range check; a partial last N group of 128 is fine).
// C is fp32 (the reference's output type) or bf16.
//
// This file checks the arguments and picks the kernel: K split over waves for
// few rows (gemm_bs_decode.hip), the 64x256 four-wave tile below for 33-64 rows
// of many columns or batches, eight-wave tiles of 128x128, 128x256 or 256x256
// for more (gemm_bs_pp.hip), stream-K on a caller's workspace (gemm_bs_sk.hip).
#include "ga_device.hpp"
#include "ga_internal.hpp"
#include "ga_pp.hpp"

namespace ga {

enum BsMode { BS_GROUP128 = 0, BS_GROUP1 = 1, BS_TENSOR = 2 };

// ---- 64x256 tile: up to 64 rows, one tile per 256 columns --------------------------
// Four waves of 64 rows x 64 columns, K step 128, three LDS stages (two in
// flight while one is computed), A and B staged with direct-to-LDS copies of 8
// whole 128-byte rows into swizzled rows (chunk c of row r at slot
// c ^ ((r >> 1) & 7)), scales loaded into registers a step ahead, operands swapped so
// that a lane owns 4 consecutive columns of one C row. A is copied once per 256
// columns, so with a tile for every CU the weights come at memory speed
// (64x129280x7168 174 us, 5.4 TB/s).
constexpr int kRows64Cols = 256;

struct Rows64Scales {
    float sa[4];    // this lane's row of the four 16-row blocks
    float sb[4][4]; // its columns of the four 16-column blocks ([0] alone but for GROUP_N 1)
};

template <int MODE, int OUT>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void bs_rows64_kernel(ga_opus_gemm_kargs ka)
{
    constexpr int kABytes = 64 * 128, kStage = kABytes + kRows64Cols * 128;
    constexpr int kACopies = 2, kCopies = 10; // per wave and stage: of A, of both
    __shared__ __attribute__((aligned(1024))) char smem[3 * kStage];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = ka.m, N = ka.n, K = ka.k, b = blockIdx.y;
    // contiguous tiles per XCD (workgroups go to the XCDs in turn)
    int unused, tile;
    map_tile_lin(blockIdx.x, gridDim.x, 1, 1, unused, tile);
    const int n0 = tile * kRows64Cols;

    const char* pa = (const char*)ka.ptr_a + (size_t)b * ka.stride_a_batch;
    const char* pb = (const char*)ka.ptr_b + (size_t)b * ka.stride_b_batch +
                     (size_t)n0 * ka.stride_b;
    const auto ra = make_rsrc(pa, rows_bytes(M, ka.stride_a, K));
    const auto rb = make_rsrc(pb, rows_bytes(N - n0, ka.stride_b, K));
    // copy i covers rows 32i .. 32i + 31, 8 of them by this wave
    int row0, chunk;
    pp::copy_lane(wave, lane, row0, chunk);
    uint32_t voff[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; i++)
        voff[i] = (uint32_t)((i < kACopies ? i : i - kACopies) * 32 + row0) *
                      (i < kACopies ? ka.stride_a : ka.stride_b) + chunk * 16;

    const float* sfa = (const float*)ka.ptr_sfa + (size_t)b * ka.stride_sfa_batch;
    const float* sfb = (const float*)ka.ptr_sfb + (size_t)b * ka.stride_sfb_batch;
    int mrow[4], ncol[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        mrow[i] = min(i * 16 + (lane & 15), M - 1);
        ncol[i] = n0 + wave * 64 + i * 16 + (lane >> 4) * 4;
    }

    auto issue = [&](int buf, int kk) {
        char* dst = smem + buf * kStage + wave * 1024;
#pragma unroll
        for (int i = 0; i < kCopies; i++)
            lds_load16(i < kACopies ? ra : rb, (lds_void*)(dst + i * 4096), voff[i] + kk, 0);
    };
    auto load_scales = [&](int g, Rows64Scales& s) {
        if constexpr (MODE != BS_TENSOR) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                s.sa[i] = sfa[(size_t)g * ka.stride_sfa + mrow[i]];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if constexpr (MODE == BS_GROUP128) {
                    s.sb[t][0] = sfb[(size_t)(min(ncol[t], N - 1) / 128) * ka.stride_sfb + g];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        s.sb[t][j] = sfb[(size_t)g * ka.stride_sfb + min(ncol[t] + j, N - 1)];
                }
            }
        }
    };

    v4f acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int t = 0; t < 4; t++)
            acc[i][t] = (v4f){0.f, 0.f, 0.f, 0.f};

    uint32_t o0, o1;
    pp::operand_lane(lane, o0, o1);
    auto compute = [&](int buf, const Rows64Scales& s) {
        const char* la = smem + buf * kStage;
        const char* lb = la + kABytes + wave * 64 * 128;
        v8i bf[4];
#pragma unroll
        for (int t = 0; t < 4; t++)
            bf[t] = pp::lds_frag(lb + t * 2048 + o0, lb + t * 2048 + o1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const v8i af = pp::lds_frag(la + i * 2048 + o0, la + i * 2048 + o1);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if constexpr (MODE == BS_TENSOR) {
                    acc[i][t] = mfma_mx16<0, 0>(bf[t], af, acc[i][t], 127, 127);
                } else {
                    const v4f p = mfma_mx16<0, 0>(bf[t], af, (v4f){0.f, 0.f, 0.f, 0.f}, 127, 127);
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float sc = s.sa[i] * s.sb[t][MODE == BS_GROUP128 ? 0 : j];
                        acc[i][t][j] = __builtin_fmaf(p[j], sc, acc[i][t][j]);
                    }
                }
            }
        }
    };

    // Step s waits for its copies and scales (only the copies of step s + 1 are
    // younger), then, after the barrier that frees the stage of step s - 1,
    // loads the scales of step s + 1 and copies step s + 2, in that order, so
    // that the next wait leaves one step of copies in flight, then computes.
    // Two scale sets alternate; copies past the last group are not read and
    // the scales' group index is clamped to it.
    const int nsteps = K / 128;
    Rows64Scales sc0, sc1;
    issue(0, 0);
    load_scales(0, sc0);
    __builtin_amdgcn_sched_barrier(0);
    issue(1, 128);
    int buf = 0; // stage of step s
    auto step = [&](int s, const Rows64Scales& cur, Rows64Scales& nxt) {
        wait_vmcnt<kCopies>();
        barrier_lds();
        load_scales(min(s + 1, nsteps - 1), nxt);
        __builtin_amdgcn_sched_barrier(0);
        issue(buf == 0 ? 2 : buf - 1, (s + 2) * 128);
        __builtin_amdgcn_sched_barrier(0);
        compute(buf, cur);
        __builtin_amdgcn_sched_barrier(0);
        buf = buf == 2 ? 0 : buf + 1;
    };
    int s = 0;
    for (; s + 1 < nsteps; s += 2) {
        step(s, sc0, sc1);
        step(s + 1, sc1, sc0);
    }
    if (s < nsteps)
        step(s, sc0, sc1);
    wait_vmcnt<0>(); // copies past the last group land before exit

    const float tscale =
        MODE == BS_TENSOR ? ((const float*)ka.ptr_sfa)[0] * ((const float*)ka.ptr_sfb)[0] : 1.0f;
    char* pc = (char*)ka.ptr_c + (size_t)b * ka.stride_c_batch * (OUT == GA_DTYPE_F32 ? 4 : 2);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int m = i * 16 + (lane & 15);
        if (m >= M)
            continue;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int n = ncol[t];
            if (n >= N)
                continue;
            const v4f v = MODE == BS_TENSOR ? acc[i][t] * tscale : acc[i][t];
            const size_t off = (size_t)m * ka.stride_c + n;
            const bool full = n + 4 <= N && (ka.stride_c & 3) == 0;
            if constexpr (OUT == GA_DTYPE_F32) {
                float* o = (float*)pc + off;
                if (full)
                    *(v4f*)o = v;
                else
                    for (int j = 0; j < 4 && n + j < N; j++)
                        o[j] = v[j];
            } else {
                uint16_t* o = (uint16_t*)pc + off;
                if (full) {
                    uint2 pk;
                    pk.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
                    pk.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
                    *(uint2*)o = pk;
                } else {
                    for (int j = 0; j < 4 && n + j < N; j++)
                        o[j] = f32_to_bf16(v[j]);
                }
            }
        }
    }
}

template <int MODE>
static void launch_bs_rows64(const ga_opus_gemm_kargs& ka, int out_dtype, hipStream_t stream)
{
    const dim3 grid((ka.n + kRows64Cols - 1) / kRows64Cols, ka.batch);
    if (out_dtype == GA_DTYPE_F32)
        hipLaunchKernelGGL((bs_rows64_kernel<MODE, GA_DTYPE_F32>), grid, dim3(256), 0, stream, ka);
    else
        hipLaunchKernelGGL((bs_rows64_kernel<MODE, GA_DTYPE_BF16>), grid, dim3(256), 0, stream, ka);
}

static void launch_bs_rows64(const ga_opus_gemm_kargs& ka, int mode, int out_dtype,
                             hipStream_t stream)
{
    mode == BS_GROUP128 ? launch_bs_rows64<BS_GROUP128>(ka, out_dtype, stream)
    : mode == BS_GROUP1 ? launch_bs_rows64<BS_GROUP1>(ka, out_dtype, stream)
                        : launch_bs_rows64<BS_TENSOR>(ka, out_dtype, stream);
}

// Which kernel dispatch_bs runs for these kargs on a device with num_cu CUs.
// The same for every scale mode, since ga_blockscale_k_slices reports the
// K-split kernel's slices without being told the mode.
enum BsPath { BS_PATH_DECODE, BS_PATH_ROWS64, BS_PATH_QUARTER, BS_PATH_HALF, BS_PATH_PP };
static BsPath bs_path(const ga_opus_gemm_kargs& ka, int num_cu)
{
    // Up to 64 rows: the K-split kernel, unless 33-64 rows have 64x256 tiles for
    // three quarters of the CUs: from there on A, copied once per 256 columns
    // instead of 64, counts for more than the split (K-split / 64x256, 64 rows:
    // 40960x4096 29.9 / 31.2 us, 57344x4096 42.9 / 37.9, 129280x7168 229 / 174,
    // 16 batches of 4096x7168 139 / 89, 24 of 2048x2048 25.4 / 23.5).
    // More rows: the smallest tile whose tiles fit on the CUs in one round
    // (128x128, 128x256), else 256x256
    // (measured on MI355X, GROUP_N 128, bf16 C, 128x128 / 128x256 / 256x256:
    // 512x8192x8192 45.4 / 59.0 / 85.8 us, 1000x8192x8192 87.3 / 71.9 / 88.7,
    // 2048x8192x8192 177 / 147 / 118), and up to 1024 rows, as far as it was
    // measured, the K-split kernel against that tile by estimated time. A
    // tile's time is a start, and per 128-K group a little more the more CUs
    // compete for L2 and power (64 groups, 128x128: 39 us with 64 tiles, 45 with
    // 256; 128x256: 56 with 32, 72 with 256; 256x256: 85 for a round).
    // Batches: the estimate knows nothing of operands that come from memory, so
    // the K-split kernel has to win by half their time, and only against the
    // 128x128 tile (its rounds over many batches take up to 1.9 times the
    // estimate: 200 of 128x512x512 42.0 us, 256x256 28.5; 16 of 128x1024x4096 31.1,
    // 128x128 23.3; 4 of 96x4096x7168 30.8 / 34.7).
    if (ka.m <= 64) {
        const long long t64 = (long long)((ka.n + kRows64Cols - 1) / kRows64Cols) * ka.batch;
        return ka.m > 32 && 4 * t64 >= 3ll * num_cu ? BS_PATH_ROWS64 : BS_PATH_DECODE;
    }
    const long long rows = (long long)((ka.m + 127) / 128) * ka.batch;
    const long long halves = rows * ((ka.n + 255) / 256), quarters = rows * ((ka.n + 127) / 128);
    const BsPath tile = quarters <= num_cu ? BS_PATH_QUARTER
                        : halves <= num_cu ? BS_PATH_HALF
                                           : BS_PATH_PP;
    if (ka.m <= 1024 && (ka.batch == 1 || tile == BS_PATH_QUARTER)) {
        const long long t256 = (long long)((ka.m + 255) / 256) * ((ka.n + 255) / 256) * ka.batch;
        const float groups = (float)(ka.k / 128);
        const float frac = (float)(tile == BS_PATH_QUARTER ? quarters : halves) / (float)num_cu;
        const float tile_us = tile == BS_PATH_QUARTER ? 5.0f + groups * (0.53f + 0.09f * frac)
                              : tile == BS_PATH_HALF
                                  ? 6.5f + groups * (0.75f + 0.27f * frac)
                                  : (float)((t256 + num_cu - 1) / num_cu) *
                                        (10.7f + 1.2f * groups);
        const float memory_us =
            ka.batch == 1 ? 0.0f
                          : 0.53f * (float)ka.batch * ((float)ka.n * ka.k + (float)ka.m * ka.k) /
                                5.85e6f;
        if (bs_decode_estimate_us(ka, num_cu) + memory_us < tile_us)
            return BS_PATH_DECODE;
    }
    return tile;
}

static ga_status dispatch_bs(const ga_opus_gemm_kargs& ka, int mode, int out_dtype,
                             hipStream_t stream)
{
    int num_cu = 0;
    ga_status st = device_cu_count(&num_cu);
    if (st != GA_OK)
        return st;
    switch (bs_path(ka, num_cu)) {
    case BS_PATH_DECODE:
        return launch_bs_decode(ka, mode, out_dtype, stream);
    case BS_PATH_ROWS64:
        launch_bs_rows64(ka, mode, out_dtype, stream);
        break;
    case BS_PATH_QUARTER:
        launch_bs_half(ka, mode, out_dtype, 1, stream);
        break;
    case BS_PATH_HALF:
        launch_bs_half(ka, mode, out_dtype, 2, stream);
        break;
    default:
        launch_bs_pp(ka, mode, out_dtype, stream);
    }
    GA_HIP_CHECK(hipGetLastError());
    return GA_OK;
}

static ga_status check_kargs(const ga_opus_gemm_kargs* ka)
{
    if (!ka || !ka->ptr_a || !ka->ptr_b || !ka->ptr_c || !ka->ptr_sfa || !ka->ptr_sfb)
        return fail(GA_ERR_ARG, "opus kargs: null pointer");
    if (ka->m <= 0 || ka->n <= 0 || ka->k <= 0 || ka->batch <= 0)
        return fail(GA_ERR_ARG, "Invalid problem size: M, N, K and batch must be positive.");
    if (ka->k % 128 != 0)
        return fail(GA_ERR_GROUP, "K must be a multiple of GROUP_K (128), got %d", ka->k);
    if (ka->stride_a < ka->k || ka->stride_b < ka->k || ka->stride_a % 16 || ka->stride_b % 16)
        return fail(GA_ERR_SHAPE, "stride_a/stride_b must be >= K and multiples of 16");
    if (ka->stride_c < ka->n)
        return fail(GA_ERR_SHAPE, "stride_c must be >= N");
    if (ka->batch > 65535)
        return fail(GA_ERR_SHAPE, "batch > 65535");
    // operands are read through buffer descriptors based at a tile's first
    // row, which address 4 GiB: 256 rows of A and B must fit in it
    const unsigned long long lim = 0xFFFFFFF0ull;
    if (256ull * (unsigned long long)ka->stride_a > lim ||
        256ull * (unsigned long long)ka->stride_b > lim)
        return fail(GA_ERR_SHAPE, "stride_a/stride_b too large for 32-bit buffer offsets "
                                  "(256 rows must fit in 4 GiB)");
    return GA_OK;
}

// The fp32 scale matrices are read through one descriptor each.
static ga_status check_scales(const ga_opus_gemm_kargs* ka, int group_n)
{
    const unsigned long long lim = 0xFFFFFFF0ull, G = (unsigned long long)ka->k / 128;
    const unsigned long long sfa = G * (unsigned long long)ka->stride_sfa * 4;
    const unsigned long long sfb = (group_n == 128 ? ((unsigned long long)ka->n + 127) / 128 : G) *
                                   (unsigned long long)ka->stride_sfb * 4;
    if (sfa > lim || sfb > lim)
        return fail(GA_ERR_SHAPE, "scale matrices larger than 4 GiB");
    return GA_OK;
}

static ga_status check_blockscale(const ga_opus_gemm_kargs* kargs, int group_n, int out_dtype)
{
    ga_status st = check_kargs(kargs);
    if (st != GA_OK)
        return st;
    if (group_n != 128 && group_n != 1)
        return fail(GA_ERR_ARG, "group_n must be 128 or 1");
    if (out_dtype != GA_DTYPE_F32 && out_dtype != GA_DTYPE_BF16)
        return fail(GA_ERR_ARG, "out_dtype must be GA_DTYPE_F32 or GA_DTYPE_BF16");
    if (group_n == 128 && kargs->stride_sfb < kargs->k / 128)
        return fail(GA_ERR_SHAPE, "stride_sfb must be >= K/128 for GROUP_N 128");
    if (group_n == 1 && kargs->stride_sfb < kargs->n)
        return fail(GA_ERR_SHAPE, "stride_sfb must be >= N for GROUP_N 1");
    if (kargs->stride_sfa < kargs->m)
        return fail(GA_ERR_SHAPE, "stride_sfa must be >= M (SFA is [K/128, M])");
    return check_scales(kargs, group_n);
}

// Workgroups of the stream-K form for these kargs on this device (0: the
// call runs as without a workspace).
static ga_status bs_stream_k_plan(const ga_opus_gemm_kargs& ka, int* nwg)
{
    int num_cu = 0;
    ga_status st = device_cu_count(&num_cu);
    if (st != GA_OK)
        return st;
    // (never for few rows, nor where 128x128 tiles fit on the CUs in one round)
    const long long t128 = (long long)((ka.m + 127) / 128) * ((ka.n + 127) / 128) * ka.batch;
    *nwg = ka.m > 64 && t128 > num_cu ? bs_sk_workgroups(ka, num_cu) : 0;
    return GA_OK;
}

} // namespace ga

using namespace ga;

extern "C" {

ga_status ga_gemm_a8w8_blockscale(const ga_opus_gemm_kargs* kargs, int group_n, int out_dtype,
                                  void* stream)
{
    ga_status st = check_blockscale(kargs, group_n, out_dtype);
    if (st != GA_OK)
        return st;
    hipStream_t s = (hipStream_t)stream;
    return dispatch_bs(*kargs, group_n == 128 ? BS_GROUP128 : BS_GROUP1, out_dtype, s);
}

ga_status ga_blockscale_stream_k(const ga_opus_gemm_kargs* kargs, int* workgroups)
{
    if (!kargs || !workgroups)
        return fail(GA_ERR_ARG, "ga_blockscale_stream_k: null argument");
    if (kargs->m <= 0 || kargs->n <= 0 || kargs->k <= 0 || kargs->batch <= 0 ||
        kargs->k % 128 != 0)
        return fail(GA_ERR_SHAPE, "ga_blockscale_stream_k: M, N, K, batch > 0, K %% 128 == 0");
    return bs_stream_k_plan(*kargs, workgroups);
}

ga_status ga_blockscale_workspace_bytes(const ga_opus_gemm_kargs* kargs, size_t* bytes)
{
    if (!bytes)
        return fail(GA_ERR_ARG, "ga_blockscale_workspace_bytes: null argument");
    int nwg = 0;
    ga_status st = ga_blockscale_stream_k(kargs, &nwg);
    if (st != GA_OK)
        return st;
    *bytes = bs_sk_workspace_bytes(*kargs, nwg);
    return GA_OK;
}

ga_status ga_gemm_a8w8_blockscale_ws(const ga_opus_gemm_kargs* kargs, int group_n, int out_dtype,
                                     void* workspace, size_t workspace_bytes, void* stream)
{
    ga_status st = check_blockscale(kargs, group_n, out_dtype);
    if (st != GA_OK)
        return st;
    int nwg = 0;
    st = bs_stream_k_plan(*kargs, &nwg);
    if (st != GA_OK)
        return st;
    if (nwg > 0 && workspace) {
        const size_t need = bs_sk_workspace_bytes(*kargs, nwg);
        if (workspace_bytes < need)
            return fail(GA_ERR_WORKSPACE, "blockscale workspace holds %zu bytes, need %zu",
                        workspace_bytes, need);
        launch_bs_pp_sk(*kargs, group_n == 128 ? BS_GROUP128 : BS_GROUP1, out_dtype, nwg,
                        workspace, (hipStream_t)stream);
        GA_HIP_CHECK(hipGetLastError());
        return GA_OK;
    }
    return ga_gemm_a8w8_blockscale(kargs, group_n, out_dtype, stream);
}

ga_status ga_blockscale_workspace_check(const ga_opus_gemm_kargs* kargs, void* workspace,
                                       size_t workspace_bytes, void* stream)
{
    if (!kargs)
        return fail(GA_ERR_ARG, "blockscale_workspace_check: null kargs");
    int nwg = 0;
    ga_status st = bs_stream_k_plan(*kargs, &nwg);
    if (st != GA_OK || nwg == 0 || !workspace)
        return st;
    const size_t counters = bs_sk_counter_bytes(*kargs);
    if (workspace_bytes < counters)
        return fail(GA_ERR_WORKSPACE, "blockscale workspace holds %zu bytes, need %zu",
                    workspace_bytes, counters);
    hipStream_t s = (hipStream_t)stream;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    GA_HIP_CHECK(hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone)
        return fail(GA_ERR_ARG, "blockscale_workspace_check synchronises: not under capture");
    const size_t tiles = (size_t)((kargs->n + 255) / 256) * ((kargs->m + 255) / 256);
    unsigned misuse = 0;
    GA_HIP_CHECK(hipStreamSynchronize(s));
    GA_HIP_CHECK(hipMemcpy(&misuse, (const char*)workspace + tiles * 4, 4, hipMemcpyDeviceToHost));
    if (misuse == 0)
        return GA_OK;
    // cleared on the caller's stream and waited for: a hipMemset would queue
    // on the null stream, which does not order against a non-blocking stream
    GA_HIP_CHECK(hipMemsetAsync(workspace, 0, counters, s));
    GA_HIP_CHECK(hipStreamSynchronize(s));
    return fail(GA_ERR_WORKSPACE, "blockscale stream-K workspace was not zero-filled before a "
                                  "call (its tile counters did not start at zero, so some tiles "
                                  "of that call were not summed); counters cleared");
}

ga_status ga_blockscale_k_slices(const ga_opus_gemm_kargs* kargs, int* groups_per_slice)
{
    if (!kargs || !groups_per_slice)
        return fail(GA_ERR_ARG, "ga_blockscale_k_slices: null argument");
    if (kargs->m <= 0 || kargs->n <= 0 || kargs->k <= 0 || kargs->batch <= 0 ||
        kargs->k % 128 != 0)
        return fail(GA_ERR_SHAPE, "ga_blockscale_k_slices: M, N, K, batch > 0, K %% 128 == 0");
    int num_cu = 0;
    ga_status st = device_cu_count(&num_cu);
    if (st != GA_OK)
        return st;
    *groups_per_slice = bs_path(*kargs, num_cu) == BS_PATH_DECODE
                            ? bs_decode_groups_per_slice(*kargs, num_cu)
                            : kargs->k / 128;
    return GA_OK;
}

ga_status ga_fp8_gemm_per_tensor(const ga_opus_gemm_kargs* kargs, int out_dtype, void* stream)
{
    ga_status st = check_kargs(kargs);
    if (st != GA_OK)
        return st;
    if (out_dtype != GA_DTYPE_F32 && out_dtype != GA_DTYPE_BF16)
        return fail(GA_ERR_ARG, "out_dtype must be GA_DTYPE_F32 or GA_DTYPE_BF16");
    hipStream_t s = (hipStream_t)stream;
    return dispatch_bs(*kargs, BS_TENSOR, out_dtype, s);
}

} // extern "C"
