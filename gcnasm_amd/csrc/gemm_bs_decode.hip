// gemm_bs_decode.hip -- fp32-scaled FP8 GEMMs (DeepSeek block scale and
// per-tensor, opus_gemm_kargs ABI) for few rows: every CU streams its share of
// the columns, K cut over the waves of a workgroup.
//
// Same results as the tile kernels up to the K split: per 128-K group g the
// MFMA (unit E8M0 scales) gives P_g, folded as acc = fmaf(P_g, SFA*SFB, acc)
// with the scale product rounded first (scale_c_tile, opus_gemm_dist/
// opus_gemm_mem_gemm_a2a/include/opus_gemm_utils.cuh:76-96); per-tensor
// accumulates in the MFMA and scales once. K is cut into `ks` slices of whole
// groups whose chains are summed in slice order.
//
// Design:
//  * a wave owns TM x NG 16x16 tiles (TM blocks of 16 rows, NG groups of 16
//    columns) and one K slice, and has an LDS ring of its own: no wave waits
//    for another before the slices are summed;
//  * operands and scales come by direct-to-LDS copies of 8 whole 128-byte rows
//    per instruction. The MFMA's own lane layout (16 rows x 64 bytes per
//    instruction), loaded straight into registers, moves 36 KB/us into a CU;
//    whole rows move 90-100 KB/us (measured on MI355X, every CU, data in L2).
//    That rate is what bounds this kernel beyond the weights' HBM time, and
//    why row-major operands pass through LDS here;
//  * a step's fragments are read into registers, then the slot is refilled,
//    then the MFMAs run: a ring of one step (large tiles) still copies under
//    its MFMAs;
//  * the K slices of a task are waves of one workgroup; the group's 16x16 tiles
//    are shared out over them for the sum in slice order and the stores;
//  * columns past N and rows past M read as zero (range-checked buffers),
//    scale indices are clamped, stores are masked.
// Measured on MI355X (bf16 C, GROUP_N 128), operands loaded into registers or
// four-wave 128x128 / 64x256 tiles -> this kernel: 1x7168x2048 7.7 -> 5.3 us, 16x2112x7168
// 12.2 -> 5.9, 32x7168x2048 13.1 -> 5.8, 64x2112x7168 22.3 -> 8.4, 64x24576x1536
// 15.6 -> 10.8, 128x8192x8192 50.7 -> 17.5, 300x2112x7168 45.1 -> 15.7,
// 512x4096x4096 28.4 -> 17.5.
#include "ga_device.hpp"
#include "ga_internal.hpp"
#include "ga_pp.hpp"

#include <algorithm>

namespace ga {
namespace {

enum { BD_GROUP128 = 0, BD_GROUP1 = 1, BD_TENSOR = 2 };

// A wave's operands of one 128-K step in LDS: 16-row blocks of 2 KB, TM of A
// then NG of B, each 16 rows of 128 bytes with 16-byte K chunk c of row r at
// slot c ^ ((r >> 1) & 7); then the step's scales, 64 dwords of SFA (one per
// row) and 64 of SFB. D such steps make the wave's ring.
template <int TM, int NG>
struct BdCfg {
    static constexpr int kScales = (TM + NG) * 2048;
    static constexpr int kStep = kScales + 512;
    static constexpr int kMax = 20480; // 8 waves in 160 KB
    static constexpr int D = kMax / kStep;
    static constexpr int kWave = D * kStep > TM * NG * 1024 ? D * kStep : TM * NG * 1024;
    static_assert(D >= 1 && kWave <= kMax, "LDS budget");
};

__device__ __forceinline__ uint32_t bd_uni(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

template <int TM, int NG, int MODE, int OUT>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 512), amdgpu_waves_per_eu(1, 2)))
void bs_decode_kernel(ga_opus_gemm_kargs ka, int nwg, int mblocks, int ks, int gps)
{
    using Cfg = BdCfg<TM, NG>;
    constexpr int D = Cfg::D;
    constexpr int kLoadsPerStep = 2 * NG + 2 * TM + (MODE == BD_TENSOR ? 0 : 2);
    static_assert(kLoadsPerStep * (D - 1) < 64, "vmcnt range");
    __shared__ __attribute__((aligned(1024))) char smem[8 * Cfg::kWave];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slice = wave % ks, tl = wave / ks;
    int wx, mb; // column share, row block
    map_tile_lin(blockIdx.x, nwg, mblocks, mblocks, mb, wx);
    const int m0 = mb * TM * 16;
    const int M = ka.m - m0, N = ka.n, K = ka.k; // rows from m0 on
    const int b = blockIdx.y;
    const int ngroups = (N + 15) / 16;
    const int g_end = (int)(((long long)(wx + 1) * ngroups) / nwg);
    const int cg0 = (int)(((long long)wx * ngroups) / nwg) + tl * NG;
    const int ng_here = min(NG, g_end - cg0);
    const bool live = ng_here > 0;
    const int G = K / 128;
    const int gb = slice * gps;
    const int ge = min(G, gb + gps);
    const int nsteps = live ? max(0, ge - gb) : 0;
    const int r = lane & 15, g = lane >> 4;
    char* ring = smem + wave * Cfg::kWave;

    v4f acc[NG][TM];
#pragma unroll
    for (int c = 0; c < NG; c++)
#pragma unroll
        for (int i = 0; i < TM; i++)
            acc[c][i] = (v4f){0.f, 0.f, 0.f, 0.f};

    if (nsteps > 0) {
        const uint32_t lda = (uint32_t)ka.stride_a, ldb = (uint32_t)ka.stride_b;
        const char* pa = (const char*)ka.ptr_a + (size_t)b * ka.stride_a_batch + (size_t)m0 * lda;
        const auto ra = make_rsrc(pa, rows_bytes(M, lda, K));
        const char* pb = (const char*)ka.ptr_b + (size_t)b * ka.stride_b_batch +
                         (size_t)cg0 * 16 * ldb;
        const auto rb = make_rsrc(pb, rows_bytes(min(ng_here * 16, N - cg0 * 16), ldb, K));
        // copy h (0, 1) of a 16-row block: lane l fetches row 8h + l / 8 from
        // whole 128-byte lines into slot l % 8
        const uint32_t crow = (uint32_t)lane >> 3, cslot = lane & 7;
        const uint32_t c0 = (cslot ^ ((crow >> 1) & 7)) * 16, c1 = c0 ^ 64u;
        const uint32_t va0 = crow * lda + c0 + (uint32_t)gb * 128;
        const uint32_t va1 = (crow + 8) * lda + c1 + (uint32_t)gb * 128;
        const uint32_t vb0 = crow * ldb + c0 + (uint32_t)gb * 128;
        const uint32_t vb1 = (crow + 8) * ldb + c1 + (uint32_t)gb * 128;

        // scales (fp32): SFA [K/128, M], lane l row l; SFB [ceil(N/128),
        // K/128], lane l group l % NG's 128-column block, or [K/128, N], lane l
        // column l (past N: the last column's, for columns never stored)
        __amdgpu_buffer_rsrc_t rsa = ra, rsb = rb;
        uint32_t vsa = 0, vsb = 0, sa_step = 0, sb_step = 0;
        if constexpr (MODE != BD_TENSOR) {
            const float* sfa = (const float*)ka.ptr_sfa + (size_t)b * ka.stride_sfa_batch;
            const float* sfb = (const float*)ka.ptr_sfb + (size_t)b * ka.stride_sfb_batch;
            rsa = make_rsrc(sfa, rows_bytes_f32(G, ka.stride_sfa, ka.m));
            sa_step = (uint32_t)ka.stride_sfa * 4;
            vsa = ((uint32_t)gb * ka.stride_sfa + m0 + min(lane, M - 1)) * 4;
            if constexpr (MODE == BD_GROUP128) {
                const int nblk = (N + 127) / 128;
                rsb = make_rsrc(sfb, rows_bytes_f32(nblk, ka.stride_sfb, G));
                sb_step = 4;
                vsb = ((uint32_t)min(((cg0 + lane % NG) * 16) / 128, nblk - 1) * ka.stride_sfb +
                       gb) * 4;
            } else {
                rsb = make_rsrc(sfb, rows_bytes_f32(G, ka.stride_sfb, N));
                sb_step = (uint32_t)ka.stride_sfb * 4;
                vsb = ((uint32_t)gb * ka.stride_sfb + min(cg0 * 16 + lane, N - 1)) * 4;
            }
        }

        // step s into ring slot j, every operand and scale by direct-to-LDS
        // copies: nothing of a step in flight lives in a register
        auto load = [&](int s, auto J) {
            char* slot = ring + decltype(J)::value * Cfg::kStep;
            const uint32_t ok = (uint32_t)s * 128;
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const uint32_t oa = ok + (uint32_t)i * 16 * lda;
                char* dst = slot + i * 2048;
                lds_load16(ra, (lds_void*)dst, va0 + bd_uni(oa), 0);
                lds_load16(ra, (lds_void*)(dst + 1024), va1 + bd_uni(oa), 0);
            }
#pragma unroll
            for (int c = 0; c < NG; c++) {
                const uint32_t ob = ok + (uint32_t)c * 16 * ldb;
                char* dst = slot + (TM + c) * 2048;
                lds_load16(rb, (lds_void*)dst, vb0 + bd_uni(ob), 0);
                lds_load16(rb, (lds_void*)(dst + 1024), vb1 + bd_uni(ob), 0);
            }
            if constexpr (MODE != BD_TENSOR) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (lds_void*)(slot + Cfg::kScales), 4,
                                                         vsa + bd_uni((uint32_t)s * sa_step), 0, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, (lds_void*)(slot + Cfg::kScales + 256),
                                                         4, vsb + bd_uni((uint32_t)s * sb_step), 0, 0, 0);
            }
        };
        uint32_t o0, o1;
        pp::operand_lane(lane, o0, o1);
        // the step in slot j (its copies have landed): fragments and scales
        // out, then, once every one has been read, the slot's next step `next`
        // in (negative: none), then the products
        auto step = [&](int next, auto J) {
            const char* q = ring + decltype(J)::value * Cfg::kStep;
            v8i fa[TM], fb[NG];
            float sa[TM];
            v4f sb[NG];
#pragma unroll
            for (int c = 0; c < NG; c++)
                fb[c] = pp::lds_frag(q + (TM + c) * 2048 + o0, q + (TM + c) * 2048 + o1);
#pragma unroll
            for (int i = 0; i < TM; i++)
                fa[i] = pp::lds_frag(q + i * 2048 + o0, q + i * 2048 + o1);
            if constexpr (MODE != BD_TENSOR) {
                const float* qs = (const float*)(q + Cfg::kScales);
#pragma unroll
                for (int i = 0; i < TM; i++)
                    sa[i] = qs[i * 16 + r];
#pragma unroll
                for (int c = 0; c < NG; c++) {
                    if constexpr (MODE == BD_GROUP128)
                        sb[c][0] = qs[64 + c];
                    else
                        sb[c] = *(const v4f*)(qs + 64 + c * 16 + g * 4);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            wait_lgkmcnt0();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            if (next >= 0)
                load(next, J);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < NG; c++)
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    if constexpr (MODE == BD_TENSOR) {
                        acc[c][i] = mfma_mx16<0, 0>(fb[c], fa[i], acc[c][i], 127, 127);
                    } else {
                        const v4f p =
                            mfma_mx16<0, 0>(fb[c], fa[i], (v4f){0.f, 0.f, 0.f, 0.f}, 127, 127);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float sc = MODE == BD_GROUP128 ? sa[i] * sb[c][0] : sa[i] * sb[c][e];
                            acc[c][i][e] = __builtin_fmaf(p[e], sc, acc[c][i][e]);
                        }
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
        };

        // In the loop every step issues the copies of the step D ahead, so the
        // wait before a step leaves exactly the D - 1 younger steps in flight.
        // In the last whole block some steps have none to issue: the wait
        // counts only the block's own younger steps. What is left waits for
        // everything.
        static_for<D>([&](auto J) {
            if ((int)J < nsteps)
                load((int)J, J);
            __builtin_amdgcn_sched_barrier(0);
        });
        int s = 0;
        for (; s + 2 * D <= nsteps; s += D)
            static_for<D>([&](auto J) {
                wait_vmcnt<kLoadsPerStep * (D - 1)>();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                step(s + D + (int)J, J);
            });
        if (s + D <= nsteps) {
            static_for<D>([&](auto J) {
                wait_vmcnt<kLoadsPerStep * (D - 1 - decltype(J)::value)>();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                const int next = s + D + (int)J;
                step(next < nsteps ? next : -1, J);
            });
            s += D;
        }
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        static_for<D>([&](auto J) {
            if ((int)J < nsteps - s)
                step(-1, J);
        });
    }

    // K slices of a column group summed in slice order, the group's 16x16
    // tiles shared out over its waves: wave z of the ks sums and stores tiles
    // z, z + ks, ...
    constexpr int NT = NG * TM;
    float* mine = (float*)ring;
#pragma unroll
    for (int c = 0; c < NG; c++)
#pragma unroll
        for (int i = 0; i < TM; i++)
            *(v4f*)(mine + (i * NG + c) * 256 + lane * 4) = acc[c][i];
    __syncthreads();
    if (!live)
        return;

    // lane holds C[m][n .. n+3], m = 16i + lane%16, n = 16cg + 4(lane/16)
    float tscale = 1.0f;
    if constexpr (MODE == BD_TENSOR)
        tscale = ((const float*)ka.ptr_sfa)[0] * ((const float*)ka.ptr_sfb)[0];
    char* pc = (char*)ka.ptr_c + ((size_t)b * ka.stride_c_batch + (size_t)m0 * ka.stride_c) *
                                     (OUT == GA_DTYPE_F32 ? 4 : 2);
    auto store = [&](int c, int i, const v4f& a) {
        const int n = (cg0 + c) * 16 + g * 4;
        const int m = i * 16 + r;
        if (c >= ng_here || n >= N || m >= M)
            return;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] = MODE == BD_TENSOR ? a[e] * tscale : a[e];
        const size_t off = (size_t)m * ka.stride_c + n;
        const bool full = n + 4 <= N && (ka.stride_c & 3) == 0;
        if constexpr (OUT == GA_DTYPE_F32) {
            float* o = (float*)pc + off;
            if (full)
                *(v4f*)o = (v4f){v[0], v[1], v[2], v[3]};
            else
                for (int e = 0; e < 4 && n + e < N; e++)
                    o[e] = v[e];
        } else {
            uint16_t* o = (uint16_t*)pc + off;
            if (full) {
                uint2 pk;
                pk.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
                pk.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
                *(uint2*)o = pk;
            } else {
                for (int e = 0; e < 4 && n + e < N; e++)
                    o[e] = f32_to_bf16(v[e]);
            }
        }
    };
    const char* part = smem + tl * ks * Cfg::kWave + lane * 16;
    for (int f = slice; f < NT; f += ks) {
        v4f t = *(const v4f*)(part + f * 1024);
        for (int z = 1; z < ks; z++) {
            const v4f u = *(const v4f*)(part + z * Cfg::kWave + f * 1024);
            t = (v4f){t[0] + u[0], t[1] + u[1], t[2] + u[2], t[3] + u[3]};
        }
        store(f % NG, f / NG, t);
    }
}

// How a problem is cut: row blocks of 16 * tm rows, ng 16-column groups per
// wave, ks K slices (waves) per column task, nwg column shares; est: the
// estimated time in us.
struct BsdPlan {
    int tm, ng, ks, nwg;
    float est;
};

// The cut with the smallest estimated time. A workgroup (one per CU: its rings
// take most of the LDS) starts, runs `steps` steps of its waves, sums its
// slices and stores; a step's time is its copies (A once per slice, a further
// task's copy of it from L1 a little cheaper), a share of the memory latency
// that a ring of D steps leaves, and the MFMAs of the waves of a SIMD. The
// coefficients are a fit to 640 times measured on MI355X (bf16 C, GROUP_N 128,
// seven (N, K) from 1000x1024 to 24576x1536 and 8192x8192, 1-768 rows): the cut
// it picks is on average 2 % slower than the fastest of those measured.
BsdPlan bsd_plan(const ga_opus_gemm_kargs& ka, int num_cu)
{
    static const struct {
        int tm, ng, depth;
    } kShapes[] = {{1, 1, BdCfg<1, 1>::D}, {1, 2, BdCfg<1, 2>::D}, {2, 1, BdCfg<2, 1>::D},
                   {2, 2, BdCfg<2, 2>::D}, {4, 2, BdCfg<4, 2>::D}, {4, 4, BdCfg<4, 4>::D}};
    const int groups = (ka.n + 15) / 16;
    const int G = ka.k / 128;
    const float bytes_us =
        ((float)ka.n * ka.k + (float)ka.m * ka.k) * (float)ka.batch / 5.85e6f;
    BsdPlan best = {0, 0, 0, 0, 0.0f};
    for (const auto& sh : kShapes) {
        // rows: one block of 16 or 32, or blocks of 32 (up to 128 rows) or 64
        if (ka.m <= 16 ? sh.tm != 1 : ka.m <= 32 ? sh.tm != 2
                                    : (sh.tm == 1 || sh.ng == 1 || (sh.tm == 2 && ka.m > 128)))
            continue;
        const long long blocks = (long long)((ka.m + 16 * sh.tm - 1) / (16 * sh.tm)) * ka.batch;
        for (int ks = 2; ks <= 8; ks *= 2) {
            if (ks > 2 && ks > G)
                continue;
            // equal shares of the column groups for every CU, at most 8 waves
            const int tt = (groups + sh.ng - 1) / sh.ng, most = sh.ng * (8 / ks);
            int nwg = (int)std::min<long long>(std::max<long long>(1, num_cu / blocks), tt);
            nwg = std::max(nwg, (groups + most - 1) / most);
            const int share = (groups + nwg - 1) / nwg, tasks = (share + sh.ng - 1) / sh.ng;
            const long long rounds = (nwg * blocks + num_cu - 1) / num_cu;
            if (ks == 8 && rounds > 1 && ka.m <= 16)
                continue; // eight short waves per group: the starts dominate
            const int steps = (G + ks - 1) / ks, waves = tasks * ks;
            const float step = 0.0133f * ks * (sh.tm + tasks * sh.ng) +
                               0.0101f * (tasks - 1) * ks * sh.tm + 0.25f / sh.depth +
                               0.0144f * sh.tm * sh.ng * ((waves + 3) / 4);
            const float est =
                1.5f + std::max(bytes_us, (float)rounds * (1.1f + 0.12f * waves +
                                                           0.08f * sh.tm * sh.ng + steps * step));
            if (best.tm == 0 || est < best.est)
                best = {sh.tm, sh.ng, ks, nwg, est};
        }
    }
    return best;
}

template <int TM, int NG, int MODE, int OUT>
ga_status launch_bsd(const ga_opus_gemm_kargs& ka, const BsdPlan& p, hipStream_t stream)
{
    const int groups = (ka.n + 15) / 16;
    const int gps = (ka.k / 128 + p.ks - 1) / p.ks;
    const int share = (groups + p.nwg - 1) / p.nwg;
    const int tasks = (share + NG - 1) / NG;
    const int mblocks = (ka.m + 16 * TM - 1) / (16 * TM);
    // the kernel's row blocks and LDS rings assume this
    if (p.tm != TM || p.ng != NG || tasks * p.ks > 8)
        return fail(GA_ERR_ARG, "block-scale decode: plan %dx%d, %d slices, %d shares", p.tm, p.ng,
                    p.ks, p.nwg);
    hipLaunchKernelGGL((bs_decode_kernel<TM, NG, MODE, OUT>), dim3(p.nwg * mblocks, ka.batch),
                       dim3(64 * tasks * p.ks), 0, stream, ka, p.nwg, mblocks, p.ks, gps);
    GA_HIP_CHECK(hipGetLastError());
    return GA_OK;
}

template <int MODE, int OUT>
ga_status launch_bsd_rows(const ga_opus_gemm_kargs& ka, int num_cu, hipStream_t stream)
{
    const BsdPlan p = bsd_plan(ka, num_cu);
    switch (p.tm * 8 + p.ng) {
    case 1 * 8 + 1: return launch_bsd<1, 1, MODE, OUT>(ka, p, stream);
    case 1 * 8 + 2: return launch_bsd<1, 2, MODE, OUT>(ka, p, stream);
    case 2 * 8 + 1: return launch_bsd<2, 1, MODE, OUT>(ka, p, stream);
    case 2 * 8 + 2: return launch_bsd<2, 2, MODE, OUT>(ka, p, stream);
    case 4 * 8 + 2: return launch_bsd<4, 2, MODE, OUT>(ka, p, stream);
    default: return launch_bsd<4, 4, MODE, OUT>(ka, p, stream);
    }
}

} // namespace

int bs_decode_groups_per_slice(const ga_opus_gemm_kargs& ka, int num_cu)
{
    const int G = ka.k / 128;
    const int ks = bsd_plan(ka, num_cu).ks;
    return (G + ks - 1) / ks;
}

float bs_decode_estimate_us(const ga_opus_gemm_kargs& ka, int num_cu)
{
    return bsd_plan(ka, num_cu).est;
}

ga_status launch_bs_decode(const ga_opus_gemm_kargs& ka, int mode, int out_dtype,
                           hipStream_t stream)
{
    int num_cu = 0;
    ga_status st = device_cu_count(&num_cu);
    if (st != GA_OK)
        return st;
    const bool f32 = out_dtype == GA_DTYPE_F32;
    if (mode == BD_GROUP128)
        return f32 ? launch_bsd_rows<BD_GROUP128, GA_DTYPE_F32>(ka, num_cu, stream)
                   : launch_bsd_rows<BD_GROUP128, GA_DTYPE_BF16>(ka, num_cu, stream);
    if (mode == BD_GROUP1)
        return f32 ? launch_bsd_rows<BD_GROUP1, GA_DTYPE_F32>(ka, num_cu, stream)
                   : launch_bsd_rows<BD_GROUP1, GA_DTYPE_BF16>(ka, num_cu, stream);
    return f32 ? launch_bsd_rows<BD_TENSOR, GA_DTYPE_F32>(ka, num_cu, stream)
               : launch_bsd_rows<BD_TENSOR, GA_DTYPE_BF16>(ka, num_cu, stream);
}

} // namespace ga
