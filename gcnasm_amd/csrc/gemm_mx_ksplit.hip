// gemm_mx_ksplit.hip -- MX GEMM (f4gemm ABI) for some tens to hundreds of rows:
// small tiles, K cut over the waves of a workgroup.
//
// The tiles of 128 and 256 rows leave most CUs idle here, and a 4-wave tile
// waits out its whole chain of copies, LDS reads and MFMAs at every K step
// (300x2112x7168 in the fp32-scaled twin, gemm_bs_decode.hip: 45 us on 51
// CUs). As there:
//  * a wave owns TM x NG 16x16 tiles and one K slice, and has an LDS ring of its
//    own: no wave waits for another before the slices are summed;
//  * operands and scales come by direct-to-LDS copies: row-major operands as 8
//    whole 128-byte rows per instruction (a fragment-shaped load of 16 rows x
//    64 bytes moves 36 KB/us into a CU, whole rows 90-100, the contiguous bytes
//    of preshuffled B 130; measured on MI355X, every CU, data in L2), a step's
//    scales as the whole 256-byte shuffled blocks of its rows and columns;
//  * a step's fragments are read into registers, then the slot is refilled,
//    then the MFMAs run;
//  * the K slices of a column task are waves of one workgroup, one fp32 chain
//    each, summed in slice order (the order of the split-K reduce, so a
//    caller's split needs no workspace here), its 16x16 tiles shared out over
//    its waves for the sum and the stores.
// MXFP4: a step is 256 K, the same 128 bytes per row, two MFMAs per tile.
// Measured on MI355X against the tiles and the few-row kernels that ran before
// (MXFP8, preshuffled B): 64x4096x4096 12.4 -> 6.9 us, 64x8192x8192 23.2 -> 14.8,
// 128x8192x8192 29.7 -> 18.4, 256x2048x2048 11.8 -> 6.1, 512x1040x4096 17.8 ->
// 11.7, 128x8192x28672 148 -> 72; MXFP4 128x8192x8192 19.2 -> 12.2.
#include "ga_device.hpp"
#include "ga_internal.hpp"
#include "ga_pp.hpp"

#include <algorithm>

namespace ga {
namespace {

// One step of a wave in LDS: 16-row blocks of 2 KB, TM of A then NG of B, then
// the 256-byte scale blocks (32 rows x 256 K) of A and of B. Row-major blocks
// are 16 rows of 128 bytes with 16-byte K chunk c of row r at slot
// c ^ ((r >> 1) & 7); preshuffled B keeps its byte order [K/16][row][16 B].
template <int TM, int NG>
struct KsCfg {
    static_assert(TM % 2 == 0 && NG % 2 == 0, "whole 32-row scale blocks");
    static constexpr int SA = TM / 2, SB = NG / 2;
    static constexpr int kScales = (TM + NG) * 2048;
    static constexpr int kStep = kScales + (SA + SB) * 256;
    static constexpr int kMax = 20480; // 8 waves in 160 KB
    static constexpr int D = kMax / kStep;
    static constexpr int kWave = D * kStep > TM * NG * 1024 ? D * kStep : TM * NG * 1024;
    static_assert(D >= 1 && kWave <= kMax, "LDS budget");
};

__device__ __forceinline__ uint32_t ks_uni(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

// Column share wx of nwg, row block mb of mblocks; ks (2, 4 or 8) slices of kpt elements
// (a multiple of 256) each.
template <int TM, int NG, bool BPS, bool FP4, int F>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 512), amdgpu_waves_per_eu(1, 2)))
void mx_ksplit_kernel(ga_f4gemm_kargs args, int nwg, int mblocks, int ks, int kpt,
                      const ga_splitk_ws_handle* __restrict__ wsh)
{
    using Cfg = KsCfg<TM, NG>;
    constexpr int D = Cfg::D, kEPB = FP4 ? 2 : 1;
    constexpr int kLoadsPerStep = 2 * (TM + NG) + Cfg::SA + Cfg::SB;
    static_assert(kLoadsPerStep * (D - 1) < 64, "vmcnt range");
    __shared__ __attribute__((aligned(1024))) char smem[8 * Cfg::kWave];
    // a caller's slot that is shorter than its split-K layout keeps the call
    // from writing anything, though the partials do not pass through it
    if (wsh && !resolve_ws(wsh, ks, args.M, args.N))
        return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slice = wave % ks, tl = wave / ks;
    int wx, mb;
    map_tile_lin(blockIdx.x, nwg, mblocks, mblocks, mb, wx);
    const int m0 = mb * TM * 16;
    const int M = (int)args.M - m0, N = (int)args.N, K = (int)args.K; // rows from m0 on
    // shares of whole pairs of 16-column groups, so that a wave's groups share
    // scale blocks two by two
    const int npairs = (N / 16 + 1) / 2;
    const int p_end = (int)(((long long)(wx + 1) * npairs) / nwg);
    const int cp0 = (int)(((long long)wx * npairs) / nwg) + tl * (NG / 2);
    const int cg0 = cp0 * 2;
    const int ng_here = min(min(NG, (p_end - cp0) * 2), N / 16 - cg0);
    const bool live = ng_here > 0;
    const int kb = slice * kpt;
    const int ke = min(K, kb + kpt);
    const int nsteps = live ? max(0, (ke - kb) / (128 * kEPB)) : 0;
    const int kbb = kb / kEPB, Kb = K / kEPB; // bytes
    const int r = lane & 15, g = lane >> 4;
    char* ring = smem + wave * Cfg::kWave;

    v4f acc[NG][TM];
#pragma unroll
    for (int c = 0; c < NG; c++)
#pragma unroll
        for (int i = 0; i < TM; i++)
            acc[c][i] = (v4f){0.f, 0.f, 0.f, 0.f};

    if (nsteps > 0) {
        const uint32_t lda = args.stride_A0 / kEPB, ldb = args.stride_B0 / kEPB; // bytes
        const char* pa = (const char*)args.ptr_A + (size_t)m0 * lda;
        const auto ra = make_rsrc(pa, rows_bytes(M, lda, Kb));
        // copy h (0, 1) of a row-major block: lane l fetches row 8h + l / 8
        // from whole 128-byte lines into slot l % 8
        const uint32_t crow = (uint32_t)lane >> 3, cslot = lane & 7;
        const uint32_t c0 = (cslot ^ ((crow >> 1) & 7)) * 16, c1 = c0 ^ 64u;
        const uint32_t va0 = crow * lda + c0 + (uint32_t)kbb;
        const uint32_t va1 = (crow + 8) * lda + c1 + (uint32_t)kbb;
        // B: columns past the wave's groups read as zero
        __amdgpu_buffer_rsrc_t rb;
        uint32_t vb0, vb1, b_step, b_grp;
        if (BPS) {
            rb = make_rsrc((const char*)args.ptr_B + (size_t)cg0 * Kb * 16,
                           (uint32_t)ng_here * (uint32_t)Kb * 16);
            vb0 = (uint32_t)lane * 16 + (uint32_t)kbb * 16;
            vb1 = vb0 + 1024;
            b_step = 2048;
            b_grp = (uint32_t)Kb * 16;
        } else {
            rb = make_rsrc((const char*)args.ptr_B + (size_t)cg0 * 16 * ldb,
                           rows_bytes(ng_here * 16, ldb, Kb));
            vb0 = crow * ldb + c0 + (uint32_t)kbb;
            vb1 = (crow + 8) * ldb + c1 + (uint32_t)kbb;
            b_step = 128;
            b_grp = 16 * ldb;
        }
        // scales: 256-byte blocks (row / 32, K / 256), lane l's dword row l % 16
        // (and 16 more), K block l / 16; byte 2 * (128-K half) + row half
        const uint32_t sna = args.stride_ScaleA0, snb = args.stride_ScaleB0;
        const auto rsa = make_rsrc(args.ptr_ScaleA, (uint32_t)(((int)args.M + 31) / 32 * 32) * sna);
        const auto rsb = make_rsrc(args.ptr_ScaleB, (uint32_t)((N + 31) / 32 * 32) * snb);
        const uint32_t sa_blk = (sna / 8) * 256, sb_blk = (snb / 8) * 256;
        const uint32_t vsa = (uint32_t)(m0 / 32) * sa_blk + (uint32_t)(kb / 256) * 256 + lane * 4;
        const uint32_t vsb = (uint32_t)cp0 * sb_blk + (uint32_t)(kb / 256) * 256 + lane * 4;

        auto load = [&](int s, auto J) {
            char* slot = ring + decltype(J)::value * Cfg::kStep;
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const uint32_t oa = (uint32_t)s * 128 + (uint32_t)i * 16 * lda;
                lds_load16(ra, (lds_void*)(slot + i * 2048), va0 + ks_uni(oa), 0);
                lds_load16(ra, (lds_void*)(slot + i * 2048 + 1024), va1 + ks_uni(oa), 0);
            }
#pragma unroll
            for (int c = 0; c < NG; c++) {
                const uint32_t ob = (uint32_t)s * b_step + (uint32_t)c * b_grp;
                char* dst = slot + (TM + c) * 2048;
                lds_load16(rb, (lds_void*)dst, vb0 + ks_uni(ob), 0);
                lds_load16(rb, (lds_void*)(dst + 1024), vb1 + ks_uni(ob), 0);
            }
            const uint32_t q = (uint32_t)(FP4 ? s : s >> 1) * 256;
            char* sc = slot + Cfg::kScales;
#pragma unroll
            for (int i = 0; i < Cfg::SA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (lds_void*)(sc + i * 256), 4,
                                                         vsa + ks_uni(q + i * sa_blk), 0, 0, 0);
#pragma unroll
            for (int c = 0; c < Cfg::SB; c++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb,
                                                         (lds_void*)(sc + (Cfg::SA + c) * 256), 4,
                                                         vsb + ks_uni(q + c * sb_blk), 0, 0, 0);
        };
        uint32_t o0, o1;
        pp::operand_lane(lane, o0, o1);
        const uint32_t b0 = BPS ? (uint32_t)lane * 16 : o0, b1 = BPS ? b0 + 1024 : o1;
        // step s in slot j (its copies have landed): fragments and scales out,
        // then, once every one has been read, step `next` in (negative:
        // none), then the products
        auto step = [&](int s, int next, auto J) {
            const char* q = ring + decltype(J)::value * Cfg::kStep;
            const char* qs = q + Cfg::kScales + lane * 4;
            // MXFP8: the step's 128-K half of each scale dword in bytes 0-1
            const uint32_t sh = FP4 ? 0u : (uint32_t)(s & 1) * 16;
            v8i fa[TM], fb[NG];
            uint32_t sa[Cfg::SA], sb[Cfg::SB];
#pragma unroll
            for (int i = 0; i < Cfg::SA; i++)
                sa[i] = *(const uint32_t*)(qs + i * 256) >> sh;
#pragma unroll
            for (int c = 0; c < Cfg::SB; c++)
                sb[c] = *(const uint32_t*)(qs + (Cfg::SA + c) * 256) >> sh;
#pragma unroll
            for (int c = 0; c < NG; c++)
                fb[c] = pp::lds_frag(q + (TM + c) * 2048 + b0, q + (TM + c) * 2048 + b1);
#pragma unroll
            for (int i = 0; i < TM; i++)
                fa[i] = pp::lds_frag(q + i * 2048 + o0, q + i * 2048 + o1);
            __builtin_amdgcn_sched_barrier(0);
            wait_lgkmcnt0();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            if (next >= 0)
                load(next, J);
            __builtin_amdgcn_sched_barrier(0);
            static_for<NG>([&](auto CC) {
                constexpr int c = decltype(CC)::value;
                static_for<TM>([&](auto II) {
                    constexpr int i = decltype(II)::value;
                    if constexpr (FP4) {
                        acc[c][i] = mfma_mx16_fp4<(c & 1), (i & 1)>(
                            fb[c], fa[i], acc[c][i], (int)sb[c >> 1], (int)sa[i >> 1]);
                        acc[c][i] = mfma_mx16_fp4<2 + (c & 1), 2 + (i & 1)>(
                            hi16(fb[c]), hi16(fa[i]), acc[c][i], (int)sb[c >> 1], (int)sa[i >> 1]);
                    } else {
                        acc[c][i] = mfma_mx16<(c & 1), (i & 1), fmt_of_b(F), fmt_of_a(F)>(
                            fb[c], fa[i], acc[c][i], (int)sb[c >> 1], (int)sa[i >> 1]);
                    }
                });
            });
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
                step(s + (int)J, s + D + (int)J, J);
            });
        if (s + D <= nsteps) {
            static_for<D>([&](auto J) {
                wait_vmcnt<kLoadsPerStep * (D - 1 - decltype(J)::value)>();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                const int next = s + D + (int)J;
                step(s + (int)J, next < nsteps ? next : -1, J);
            });
            s += D;
        }
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        static_for<D>([&](auto J) {
            if ((int)J < nsteps - s)
                step(s + (int)J, -1, J);
        });
    }

    // K slices summed in slice order: wave z of a task's ks sums and stores
    // its 16x16 tiles z, z + ks, ...
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
    // lane holds C[m][n .. n+3], m = 16i + lane%16, n = 16cg + 4(lane/16); the
    // library is built with -ffp-contract=off: alpha*v and + beta*c round
    // separately
    const int ldd = (int)args.stride_C0;
    const float alpha = args.alpha, beta = args.beta;
    const bool use_c = beta != 0.0f && args.ptr_C != nullptr;
    auto store = [&](int c, int i, const v4f& v) {
        const int m = i * 16 + r, n = (cg0 + c) * 16 + g * 4;
        if (c >= ng_here || m >= M)
            return;
        const size_t off = (size_t)(m0 + m) * ldd + n;
        uint16_t o[4];
        const uint16_t* cin = use_c ? (const uint16_t*)args.ptr_C + off : nullptr;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float x = alpha * v[j];
            if (use_c)
                x = x + beta * bf16_to_f32(cin[j]);
            o[j] = f32_to_bf16(x);
        }
        uint2 pk;
        pk.x = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
        pk.y = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
        *(uint2*)((uint16_t*)args.ptr_D + off) = pk;
    };
    const char* part = smem + tl * ks * Cfg::kWave + lane * 16;
    for (int f = slice; f < NT; f += ks) {
        v4f t = *(const v4f*)(part + f * 1024);
        for (int z = 1; z < ks; z++)
            t = t + *(const v4f*)(part + z * Cfg::kWave + f * 1024);
        store(f % NG, f / NG, t);
    }
}

// How a problem is cut: row blocks of 16 * tm rows, ng 16-column groups per
// wave, ks K slices of kpt elements (waves) per column task, nwg column shares;
// est: the estimated time in us.
struct KsPlan {
    int tm, ng, ks, kpt, nwg;
    float est;
};

// The cut with the smallest estimated time. A workgroup (one per CU: its rings
// take most of the LDS) starts, runs `steps` steps of its waves, sums its
// slices and stores; a step's time is its copies (A once per slice, a further
// task's copy of it from L1 a little cheaper), a share of the memory latency
// that a ring of D steps leaves, and the MFMAs of the waves of a SIMD. The
// coefficients are a fit to 900 times measured on MI355X (MXFP8 and MXFP4,
// eight (N, K) from 3072x1024 to 28672x8192, 65-1000 rows): the cut it picks
// is on average 2 % slower than the fastest of those measured. More slices have
// to promise 5 %.
KsPlan ks_plan(const ga_f4gemm_kargs& args, bool fp4, int gdz, int num_cu)
{
    static const struct {
        int tm, ng, depth;
    } kShapes[] = {{2, 2, KsCfg<2, 2>::D}, {4, 2, KsCfg<4, 2>::D}, {4, 4, KsCfg<4, 4>::D}};
    const int M = (int)args.M, N = (int)args.N, K = (int)args.K;
    const int pairs = (N / 16 + 1) / 2, units = (K + 255) / 256;
    const float bytes_us = ((float)N * K + (float)M * K) / (fp4 ? 2.0f : 1.0f) / 5.85e6f;
    KsPlan best = {0, 0, 0, 0, 0, 0.0f};
    for (const auto& sh : kShapes) {
        KsPlan mine = {0, 0, 0, 0, 0, 0.0f};
        const long long blocks = (M + 16 * sh.tm - 1) / (16 * sh.tm);
        for (int ks = gdz > 1 ? gdz : 2; ks <= 8; ks *= 2) {
            if (gdz > 1 ? ks != gdz : (ks > 2 && ks > units))
                continue;
            // a caller's split keeps its slices, else equal ones of whole 256-K
            // scale blocks
            const int kpt = gdz > 1 ? ((K >> args.log2_k_split) + 255) / 256 * 256
                                    : (units + ks - 1) / ks * 256;
            const int tt = (pairs + sh.ng / 2 - 1) / (sh.ng / 2), most = sh.ng / 2 * (8 / ks);
            int nwg = (int)std::min<long long>(std::max<long long>(1, num_cu / blocks), tt);
            nwg = std::max(nwg, (pairs + most - 1) / most);
            const int share = (pairs + nwg - 1) / nwg;
            const int tasks = (share + sh.ng / 2 - 1) / (sh.ng / 2);
            const long long rounds = (nwg * blocks + num_cu - 1) / num_cu;
            const int steps = kpt / (fp4 ? 256 : 128), waves = tasks * ks;
            const float step = 0.0165f * ks * (sh.tm + tasks * sh.ng) +
                               0.014f * (tasks - 1) * ks * sh.tm + 0.181f / sh.depth +
                               0.0186f * sh.tm * sh.ng * ((waves + 3) / 4);
            const float est =
                1.5f + std::max(bytes_us, (float)rounds * (1.34f + 0.01f * waves +
                                                           0.088f * sh.tm * sh.ng + steps * step));
            if (mine.tm == 0 || est < 0.95f * mine.est)
                mine = {sh.tm, sh.ng, ks, kpt, nwg, est};
        }
        if (mine.tm != 0 && (best.tm == 0 || mine.est < best.est))
            best = mine;
    }
    return best;
}

template <int TM, int NG, bool BPS, bool FP4, int F>
void launch_ks(const ga_f4gemm_kargs& args, const KsPlan& p, const ga_splitk_ws_handle* wsh,
               hipStream_t stream)
{
    const int pairs = ((int)args.N / 16 + 1) / 2;
    const int share = (pairs + p.nwg - 1) / p.nwg;
    const int tasks = (share + NG / 2 - 1) / (NG / 2);
    const int mblocks = ((int)args.M + 16 * TM - 1) / (16 * TM);
    hipLaunchKernelGGL((mx_ksplit_kernel<TM, NG, BPS, FP4, F>), dim3(p.nwg * mblocks),
                       dim3(64 * tasks * p.ks), 0, stream, args, p.nwg, mblocks, p.ks, p.kpt, wsh);
}

template <bool BPS, bool FP4, int F>
void launch_ks_shape(const ga_f4gemm_kargs& args, const KsPlan& p, const ga_splitk_ws_handle* wsh,
                     hipStream_t stream)
{
    if (p.tm == 2)
        launch_ks<2, 2, BPS, FP4, F>(args, p, wsh, stream);
    else if (p.ng == 2)
        launch_ks<4, 2, BPS, FP4, F>(args, p, wsh, stream);
    else
        launch_ks<4, 4, BPS, FP4, F>(args, p, wsh, stream);
}

template <bool FP4, int F>
void launch_ks_b(const ga_f4gemm_kargs& args, const KsPlan& p, bool bps,
                 const ga_splitk_ws_handle* wsh, hipStream_t stream)
{
    bps ? launch_ks_shape<true, FP4, F>(args, p, wsh, stream)
        : launch_ks_shape<false, FP4, F>(args, p, wsh, stream);
}

} // namespace

float mx_ksplit_estimate_us(const ga_f4gemm_kargs& args, bool fp4, int num_cu)
{
    return ks_plan(args, fp4, 1, num_cu).est;
}

void mx_ksplit_cut(const ga_f4gemm_kargs& args, bool fp4, int gdz, int num_cu, int* rows,
                   int* cols, int* slices)
{
    const KsPlan p = ks_plan(args, fp4, gdz, num_cu);
    *rows = 16 * p.tm;
    *cols = 16 * p.ng;
    *slices = p.ks;
}

void launch_mx_ksplit(const ga_f4gemm_kargs& args, int gdz, bool bps, bool fp4, int fmt,
                      const ga_splitk_ws_handle* wsh, int num_cu, hipStream_t stream)
{
    const KsPlan p = ks_plan(args, fp4, gdz, num_cu);
    if (fp4) {
        launch_ks_b<true, 0>(args, p, bps, wsh, stream);
        return;
    }
    switch (fmt) {
    case 1: launch_ks_b<false, 1>(args, p, bps, wsh, stream); break;
    case 2: launch_ks_b<false, 2>(args, p, bps, wsh, stream); break;
    case 3: launch_ks_b<false, 3>(args, p, bps, wsh, stream); break;
    default: launch_ks_b<false, 0>(args, p, bps, wsh, stream); break;
    }
}

} // namespace ga
