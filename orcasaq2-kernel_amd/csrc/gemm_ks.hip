// EXL3 decode-GEMM for 17 .. KS_MAX_ROWS rows, split over the inputs:
//   C = fp16( H( fp16(H(A * suh)) . W_q ) * svh )
// Replaces the fused exl3_gemm of orcasaq2/ops.py:46-49 (17..144 rows) and the reconstruct branch
// of orcasaq2/ops.py:50-59 above it.
//
// What bounds it: at few rows the decode (four vector instructions per weight: state,
// multiply-add, mask, half sum; 17408 x 5120 takes ~10 us of issue on the whole chip), at 128
// rows the matrix pipe beside it (32x32x16 MFMAs at ~20 ns each under the card's power limit).
// So each weight is decoded once per 128-row tile, straight into the B operands of the lane that
// needs them, and what is left is kept off the critical path:
//   * set-up: fp16(H(A * suh)) in the order of the MFMA A fragments, so that a step's fragments
//     are contiguous kilobytes that go to LDS by direct loads;
//   * decode: a workgroup of eight waves takes 128 outputs and a run of steps (32 inputs each);
//     four pairs of waves split the steps, the two waves of a pair 64 outputs each.  A and the
//     trellis words run up to five steps ahead through an LDS ring (no registers held, one
//     barrier per step); the fragments of a step are multiplied while those of the next are
//     decoded into the registers just read;
//   * the pairs' sums meet in LDS; a segment (128 outputs of a row tile) that one workgroup does
//     alone is finished there, the segments left over after whole rounds are split over all the
//     workgroups' pairs evenly and leave fp32 sums in slots;
//   * finishing launch: slots added in workgroup order (deterministic), output Hadamard, svh.  One
//     more launch (~5 us) instead of the last workgroup of each tile adding all of its slots while
//     the others have left (20-40 us of the stream-K launches this replaced).
// Measured on MI355X, us per call in a HIP graph, this / the stream-K launch it replaced, at 17, 64,
// 128, 256 rows: 17408 -> 5120 K = 4 31 / 47, 38 / 66, 47 / 92, 75 / 114; 5120 -> 17408 K = 3
// 30 / 43, 36 / 55, 47 / 74, 81 / 105; 5120 -> 6144 K = 4 20 / 27, 25 / 39, 30 / 57, 39 / 65.
#include "exl3_common.h"
#include "gemm_ks_plan.h"

#include <atomic>

namespace exl3 {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 ks_mfma(const f16x8& a, const f16x8& b, const f32x16& c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Set-up: fp16(H128(A * suh)) of every shard in A-fragment order, one workgroup per (shard,
// 128-input block, 32-row tile); rows past the call's are zero.
__global__ __launch_bounds__(512) void ks_prep_kernel(const KsPrepArgs p)
{
    const int b = blockIdx.x, m = blockIdx.y, s = blockIdx.z;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15;
    const int row = 4 * wv + (lane >> 4), grow = 32 * m + row;
    uint4 o = {0u, 0u, 0u, 0u};
    if (grow < p.rows) {
        uint4 x, sg;
        __builtin_memcpy(&x, p.A + (long)grow * p.ic + b * 128 + 8 * l16, 16);
        __builtin_memcpy(&sg, p.suh[s] + b * 128 + 8 * l16, 16);
        float v[8], f[8];
        if (p.bf) x = uint4{act_pair(x.x, 1), act_pair(x.y, 1), act_pair(x.z, 1), act_pair(x.w, 1)};
        had_unpack(x, v);
        had_unpack(sg, f);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] *= f[i];
        had16_stages(v, l16);
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint16_t h0 = __builtin_bit_cast(uint16_t, (_Float16)(v[2 * i] * 0.08838834764831845f));
            const uint16_t h1 = __builtin_bit_cast(uint16_t, (_Float16)(v[2 * i + 1] * 0.08838834764831845f));
            w[i] = (uint32_t)h0 | ((uint32_t)h1 << 16);
        }
        o = uint4{w[0], w[1], w[2], w[3]};
    }
    reinterpret_cast<uint4*>(p.Ah[s])[ks_prep_chunk(p, b, m, row, l16)] = o;
}

// Workgroup barrier that orders LDS accesses only (__syncthreads() would also wait for this
// wave's global stores).
__device__ __forceinline__ void ks_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Decode of a fragment (F = 0, 1: rows 0..7 of columns c, c + 8; 2, 3: rows 8..15) in four stages
// of eight independent instructions each: with two waves per SIMD, one weight's chain of dependent
// instructions (state, multiply-add, mask, half sum) issued alone leaves most issue slots empty.
// Position of word e (0..7) of the fragment.
template <int F, int E>
constexpr int ks_pos() { return 4 * (F & 1) + 2 * (F >> 1) + 8 * (E >> 1) + (E & 1); }

template <int K, int CB, int Q>
__device__ __forceinline__ uint32_t ks_dec_state(const uint32_t (&w)[K + 1], const Dot2Consts& kc)
{
    using P = StatePlan<K, Q>;
    if constexpr (P::kind <= 1) {
        const uint32_t src = w[P::wi];
        if constexpr (CB == CB_MCG) return P::kind == 1 ? (src >> 16) : (src & 0xffffu);
        else return P::kind == 1 ? sdwa_add_hi(src, kc.off) : sdwa_add_lo(src, kc.off);
    } else
        return state_field<K, Q>(w);
}

template <int K, int CB, int Q>
__device__ __forceinline__ uint32_t ks_dec_mul(uint32_t s, const Dot2Consts& kc)
{
    if constexpr (CB == CB_MCG) return s * CBMCG_MUL;
    else if constexpr (StatePlan<K, Q>::kind <= 1) return s * CB3_MUL;
    else return mad_lo(s, kc.mul, CB3_ADD);
}

// f(integral_constant<int, I>) for I = B .. E - 1, in order.
template <int B, int E, class F>
__device__ __forceinline__ void ks_static_for(F&& f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        ks_static_for<B + 1, E>(f);
    }
}

template <int MT>
struct KsAcc {
    f32x16 c[MT][2];   // [32-row block][column half]
};

// Direct-to-LDS load: 4 * N bytes a lane from base + voff (bytes) to LDS byte address dst + 4 * N * lane.
// Inline assembly, so the compiler's wait insertion does not see it (it would wait for every such
// load before any later LDS read); the step waits order it.
template <int N>
__device__ __forceinline__ void ks_dma(const void* base, uint32_t voff, uint32_t dst)
{
    if constexpr (N == 4)
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(dst) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "s"(dst) : "memory", "m0");
}

// Until at most N vector-memory operations of this wave are outstanding.
template <int N>
__device__ __forceinline__ void ks_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }

// Steps p0 .. p1 - 1 of a wave, nmax >= p1 - p0 barriers in all (the workgroup's waves meet at
// every step).  Stage i % NB of the LDS ring holds A of step i and the words of step i + 1,
// both read into registers during step i - 1; loads run NB - 1 steps ahead of that.  Per fragment: the MFMAs of step i, then the decode of the same
// fragment of step i + 1 into the registers they have read.
template <int K, int CB, int MT>
__device__ __forceinline__ void ks_steps(KsAcc<MT>& acc, const KsShard& S, const char* lds, uint32_t lds_base, int cg, int m0,
                                         int mtt, int p0, int p1, int nmax, int wave, int lane, const Dot2Consts& kc)
{
    constexpr int NB = ks_nb(MT);
    constexpr int L = MT + ks_w_runs(K);   // loads per stage
    const int n = p1 - p0;
    const int pair = wave >> 1, half = wave & 1;
    if (n <= 0) {
        for (int i = 0; i < nmax; i++) ks_barrier();
        return;
    }
    const char* wb = reinterpret_cast<const char*>(S.trellis + ks_b_word(p0, 0, S.tc, cg, half, K));
    uint32_t wl[2];
#pragma unroll
    for (int r = 0; r < 2; r++) wl[r] = 4u * (uint32_t)(ks_b_word(0, lane, S.tc, 0, 0, K) + ks_w_run(K, r, lane));
    const long wstep = (long)2 * S.tc * 32 * K;
    // this wave loads fragments half * MT .. + MT - 1 of the pair's 2 MT
    const char* ab = reinterpret_cast<const char*>(S.Ah) + 16 * ks_a_chunk(p0, mtt, m0, 0, 0) + half * MT * 1024;
    const long astep = (long)mtt * 2048;
    const uint32_t al = 16u * lane;
    auto dma_w = [&](int i, int st) {
        const char* b = wb + i * wstep;
        const uint32_t dst = lds_base + ks_stage_w(MT, st, wave);
        ks_dma<K == 1 ? 1 : 4>(b, wl[0], dst);
        if constexpr (ks_w_runs(K) == 2) ks_dma<4>(b, wl[1], dst + 1024);
    };
    auto dma = [&](int i, int st) {
        const uint32_t dst = lds_base + ks_stage_a(MT, st, pair) + half * MT * 1024;
#pragma unroll
        for (int t = 0; t < MT; t++) ks_dma<4>(ab + i * astep + t * 1024, al, dst + t * 1024);
        dma_w(min(i + 1, n - 1), st);
    };
    // word offsets of this lane's chunk and of the word before it (tail-biting)
    const int w0_off = ks_w_off(K, K - 1, (lane & 7) ? lane - 1 : lane + 7);
    auto read_w = [&](uint32_t (&w)[K + 1], int st) {
        const char* p = lds + ks_stage_w(MT, st, wave);
        w[0] = *reinterpret_cast<const uint32_t*>(p + w0_off);
        if constexpr (K >= 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(p + 16 * lane);
            w[1] = v.x; w[2] = v.y; w[3] = v.z; w[4] = v.w;
        }
        if constexpr (K == 8) {
            const uint4 v = *reinterpret_cast<const uint4*>(p + 1024 + 16 * lane);
            w[5] = v.x; w[6] = v.y; w[7] = v.z; w[8] = v.w;
        } else {
#pragma unroll
            for (int j = K < 4 ? 0 : 4; j < K; j++) w[j + 1] = *reinterpret_cast<const uint32_t*>(p + ks_w_off(K, j, lane));
        }
    };
    // Stage s has landed when at most the loads of the younger stages are outstanding: at step
    // s - 1 those are issued up to stage min(n - 1, s + NB - 2).
    auto wait_stage = [&](int s) {
        const int r = n - 1 - s;
        if (r >= NB - 2) ks_wait_vm<(NB - 2) * L>();
        else if (NB > 5 && r == 3) ks_wait_vm<3 * L>();
        else if (NB > 4 && r == 2) ks_wait_vm<2 * L>();
        else if (NB > 3 && r == 1) ks_wait_vm<L>();
        else ks_wait_vm<0>();
    };
    const std::integral_constant<int, 0> c0;
    const std::integral_constant<int, 1> c1;
    const std::integral_constant<int, 2> c2;
    const std::integral_constant<int, 3> c3;
    const std::integral_constant<int, -1> none;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    f16x8 a[MT][2];
    u32x4 bf[4];
    auto read_a = [&](auto fi, int st) {
        constexpr int f = decltype(fi)::value;
        const char* as = lds + ks_stage_a(MT, st, pair) + 16 * lane;
#pragma unroll
        for (int m = 0; m < MT; m++) a[m][f] = *reinterpret_cast<const f16x8*>(as + (m * 2 + f) * 1024);
    };
    // Stage t of the decode of fragment d from wd.
    uint32_t x[8];
    auto stage = [&](auto ti, auto di, const uint32_t (&wd)[K + 1]) {
        constexpr int t = decltype(ti)::value, d = decltype(di)::value;
        if constexpr (t < 3)
            ks_static_for<0, 8>([&](auto ei) {
                constexpr int e = decltype(ei)::value, Q = ks_pos<d, e>();
                if constexpr (t == 0) x[e] = ks_dec_state<K, CB, Q>(wd, kc);
                else if constexpr (t == 1) x[e] = ks_dec_mul<K, CB, Q>(x[e], kc);
                else x[e] = (x[e] & kc.mask) ^ kc.flip;
            });
        else
#pragma unroll
            for (int j = 0; j < 4; j++) bf[d][j] = pack_sum(x[2 * j], x[2 * j + 1]);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Quarter q of a step: its MT MFMAs on fragment q, between them the stages of the decode of
    // fragment d (if any) from wd.  An MFMA waiting for the matrix pipe holds up the other wave's
    // vector instructions too, so MFMAs are not issued back to back where there is decode work.
    auto quarter = [&](auto qi, auto di, const uint32_t (&wd)[K + 1]) {
        constexpr int q = decltype(qi)::value, d = decltype(di)::value;
        ks_static_for<0, MT>([&](auto mi) {
            constexpr int m = decltype(mi)::value;
            acc.c[m][q & 1] = ks_mfma(a[m][q >> 1], __builtin_bit_cast(f16x8, bf[q]), acc.c[m][q & 1]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (d >= 0) ks_static_for<4 * m / MT, 4 * (m + 1) / MT>([&](auto ti) { stage(ti, di, wd); });
        });
    };
    auto decode = [&](auto di, const uint32_t (&wd)[K + 1]) {
        ks_static_for<0, 4>([&](auto ti) { stage(ti, di, wd); });
    };
    // the words of step 0 go through the last stage's area, which its own loads reach only after
    // the first barrier
    dma_w(0, NB - 1);
#pragma unroll
    for (int i = 0; i < NB - 1; i++)
        if (i < n) dma(i, i);
    if (n >= NB - 1) ks_wait_vm<(NB - 1) * L>();
    else ks_wait_vm<0>();
    uint32_t w[K + 1], wo[K + 1];   // words of the next step, of the current one
    read_w(w, NB - 1);
    decode(c0, w);
    decode(c1, w);
    decode(c2, w);
#pragma unroll
    for (int j = 0; j <= K; j++) wo[j] = w[j];
    if (n >= NB - 1) ks_wait_vm<(NB - 2) * L>();
    else ks_wait_vm<0>();
    ks_barrier();
    if (NB - 1 < n) dma(NB - 1, NB - 1);
    read_a(c0, 0);
    read_a(c1, 0);
    read_w(w, 0);
    int st = 0;   // stage of step i; its A is in registers by the barrier of step i
    for (int i = 0; i + 1 < n; i++) {
        const int nx = st + 1 == NB ? 0 : st + 1;
        wait_stage(i + 1);
        ks_barrier();
        if (i + NB < n) dma(i + NB, st);
        __builtin_amdgcn_sched_barrier(0);
        quarter(c0, c3, wo);
        quarter(c1, c0, w);
        read_a(c0, nx);
        __builtin_amdgcn_sched_barrier(0);
        quarter(c2, c1, w);
        quarter(c3, c2, w);
        read_a(c1, nx);
#pragma unroll
        for (int j = 0; j <= K; j++) wo[j] = w[j];
        read_w(w, nx);
        __builtin_amdgcn_sched_barrier(0);
        st = nx;
    }
    quarter(c0, c3, wo);
    quarter(c1, none, wo);
    quarter(c2, none, wo);
    quarter(c3, none, wo);
    for (int i = n; i < nmax; i++) ks_barrier();
}

// Output rows: the fp32 row staged at `st` (128 outputs, lane l the pair 2 l, 2 l + 1) through
// the output Hadamard and svh.
template <int N>
__device__ __forceinline__ void ks_rows_out(const float* st, int row0, int rows, const KsShard& S, int cg, int bf, int lane)
{
    const uint32_t sv = reinterpret_cast<const uint32_t*>(S.svh + cg * 128)[lane];
    const float s0 = (float)__builtin_bit_cast(_Float16, (uint16_t)(sv & 0xffffu));
    const float s1 = (float)__builtin_bit_cast(_Float16, (uint16_t)(sv >> 16));
    float v0[N], v1[N];
#pragma unroll
    for (int r = 0; r < N; r++) {
        const float2 x = *reinterpret_cast<const float2*>(st + r * KS_LDC + 2 * lane);
        v0[r] = x.x;
        v1[r] = x.y;
    }
    wave_fwht128_n<N>(v0, v1, fwht_signs(lane));
#pragma unroll
    for (int r = 0; r < N; r++)
        if (row0 + r < rows)
            reinterpret_cast<uint32_t*>(S.C + (long)(row0 + r) * S.ldc + cg * 128)[lane] =
                out_pair(v0[r] * s0, v1[r] * s1, bf);
}

// The waves' accumulators of 32-row block m to LDS, by column position.
template <int MT>
__device__ __forceinline__ void ks_stage(const KsAcc<MT>& acc, int m, int pair, int half, int lane, float* red)
{
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            *reinterpret_cast<float4*>(red + ks_red(pair, 64 * half + 32 * h + (lane & 31), 2 * j + (lane >> 5))) =
                float4{acc.c[m][h][4 * j], acc.c[m][h][4 * j + 1], acc.c[m][h][4 * j + 2], acc.c[m][h][4 * j + 3]};
}

// The staged sums of pairs k0 .. k1 - 1 at (column position, quad), in pair order.
__device__ __forceinline__ float4 ks_sum(const float* red, int k0, int k1, int cpos, int quad)
{
    float4 v = *reinterpret_cast<const float4*>(red + ks_red(k0, cpos, quad));
    for (int k = k0 + 1; k < k1; k++) {
        const float4 x = *reinterpret_cast<const float4*>(red + ks_red(k, cpos, quad));
        v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
    }
    return v;
}

template <int CB, int MT>
__global__ __launch_bounds__(128 * KS_NP) __attribute__((amdgpu_waves_per_eu(KS_NP / 2, KS_NP / 2)))
void gemm_ks_kernel(const KsArgs a)
{
    constexpr int NP = KS_NP, T = 128 * NP, NV = 1024 / T;
    extern __shared__ __attribute__((aligned(16))) float red[];
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(void __attribute__((address_space(3)))*)red);
    const int g = ks_logical(blockIdx.x, gridDim.x);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pair = wave >> 1, half = wave & 1;
    const int lane = tid & 63;
    const Dot2Consts kc = dot2_consts();
    // the launch arguments' lines of the shard table into the scalar cache, all at once: the
    // shard's own fields are read at an index known only later
#pragma unroll
    for (int i = 0; i < KS_MAXSH; i++) asm volatile("" ::"s"(a.sh[i].cbeg));
    const int rounds = a.full + (a.nrem ? 1 : 0);
    for (int round = 0; round < rounds; round++) {
        // this pair's segment and its run among the segment's pairs: a whole segment over the
        // workgroup's pairs, or a split one over some of the launch's
        const bool split = round == a.full;
        int seg = round * a.G + g, k = pair, nmax = ks_run_max(a.whole);
        KsCut cut = a.whole;
        int s0 = 0, last0 = NP;   // split: pairs 0 .. last0 - 1 hold split segment s0, the others s0 + 1
        if (split) {
            const int j0 = NP * g;
            s0 = ks_seg_of(a, j0);
            const int next = ks_pair0(a, s0 + 1);
            last0 = min(NP, next - j0);
            const int s = s0 + (pair >= last0);
            k = j0 + pair - (pair >= last0 ? next : ks_pair0(a, s0));
            cut = ks_cut(a, s);
            // barriers of the round: the most steps of any pair (a later segment has fewer pairs)
            nmax = ks_run_max(ks_cut(a, last0 < NP ? s0 + 1 : s0));
            seg = a.full * a.G + s;
        }
        const KsSeg sg = ks_seg(a, seg);
        const KsShard& S = a.sh[sg.si];
        const int p0 = ks_run(cut, k), p1 = ks_run(cut, k + 1);
        KsAcc<MT> acc;
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc.c[m][h][e] = 0.f;
#define KS_CASE(KK) case KK: ks_steps<KK, CB, MT>(acc, S, reinterpret_cast<const char*>(red), lds_base, sg.cg, sg.rt * MT, a.mtt, p0, p1, nmax, wave, lane, kc); break;
        switch (S.K) {
            KS_CASE(1) KS_CASE(2) KS_CASE(3) KS_CASE(4) KS_CASE(5) KS_CASE(6) KS_CASE(7) KS_CASE(8)
        }
#undef KS_CASE
        ks_barrier();   // every wave is done with the ring
        // the pairs' partial sums added in pair order, 32 rows at a time
        if (split) {
            float4* const slot0 = reinterpret_cast<float4*>(a.slots) + ks_slot(s0, g, MT);
#pragma unroll
            for (int m = 0; m < MT; m++) {
                if (m) ks_barrier();
                ks_stage<MT>(acc, m, pair, half, lane, red);
                ks_barrier();
#pragma unroll
                for (int kk = 0; kk < NV; kk++) {
                    const int idx = tid + T * kk, quad = idx >> 7, cpos = idx & 127;
                    slot0[ks_slot_in(8 * m + quad, cpos)] = ks_sum(red, 0, last0, cpos, quad);
                    if (last0 < NP) slot0[MT * 1024 + ks_slot_in(8 * m + quad, cpos)] = ks_sum(red, last0, NP, cpos, quad);
                }
            }
        } else {
#pragma unroll
            for (int m = 0; m < MT; m++) {
                ks_stage<MT>(acc, m, pair, half, lane, red);
                ks_barrier();
                float4 v[NV];
#pragma unroll
                for (int kk = 0; kk < NV; kk++) {
                    const int idx = tid + T * kk;
                    v[kk] = ks_sum(red, 0, NP, idx & 127, idx >> 7);
                }
                ks_barrier();
#pragma unroll
                for (int kk = 0; kk < NV; kk++) {
                    const int idx = tid + T * kk, quad = idx >> 7, col = ks_out_col(idx & 127);
                    float* st = red + 4 * quad * KS_LDC + col;
                    st[0] = v[kk].x;
                    st[KS_LDC] = v[kk].y;
                    st[2 * KS_LDC] = v[kk].z;
                    st[3 * KS_LDC] = v[kk].w;
                }
                ks_barrier();
                constexpr int NR = 32 / (2 * NP);
                ks_rows_out<NR>(red + wave * NR * KS_LDC, 32 * (sg.rt * MT + m) + wave * NR, a.rows, S, sg.cg, a.bf, lane);
                ks_barrier();
            }
        }
    }
}

// Eight rows (two quads) of one split segment: its slots added in workgroup order, then the
// output Hadamard and svh.
__global__ __launch_bounds__(256) void ks_finish_kernel(const KsArgs a, int mt)
{
    __shared__ float st[8 * KS_LDC];
    const int s = blockIdx.y, o = blockIdx.x;
    const KsSeg sg = ks_seg(a, a.full * a.G + s);
    const int row0 = 32 * mt * sg.rt + 8 * o;
    if (row0 >= a.rows) return;
    const int g_lo = ks_pair0(a, s) / KS_NP, g_hi = (ks_pair0(a, s + 1) - 1) / KS_NP;
    const int tid = threadIdx.x, quad = 2 * o + (tid >> 7), cpos = tid & 127;
    const KsShard& S = a.sh[sg.si];
    float4 v = {0.f, 0.f, 0.f, 0.f};
    constexpr int B = 8;
    for (int g0 = g_lo; g0 <= g_hi; g0 += B) {
        float4 x[B];
#pragma unroll
        for (int i = 0; i < B; i++)
            x[i] = reinterpret_cast<const float4*>(a.slots)[ks_slot(s, min(g0 + i, g_hi), mt) + ks_slot_in(quad, cpos)];
#pragma unroll
        for (int i = 0; i < B; i++)
            if (g0 + i <= g_hi) {
                v.x += x[i].x; v.y += x[i].y; v.z += x[i].z; v.w += x[i].w;
            }
    }
    float* p = st + 4 * (tid >> 7) * KS_LDC + ks_out_col(cpos);
    p[0] = v.x;
    p[KS_LDC] = v.y;
    p[2 * KS_LDC] = v.z;
    p[3 * KS_LDC] = v.w;
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    ks_rows_out<2>(st + 2 * wave * KS_LDC, row0 + 2 * wave, a.rows, S, sg.cg, a.bf, tid & 63);
}

// ---------------------------------------------------------------- host side

template <int CB>
static const void* ks_fn(int mt)
{
    switch (mt) {
    case 1: return reinterpret_cast<const void*>(&gemm_ks_kernel<CB, 1>);
    case 2: return reinterpret_cast<const void*>(&gemm_ks_kernel<CB, 2>);
    case 3: return reinterpret_cast<const void*>(&gemm_ks_kernel<CB, 3>);
    default: return reinterpret_cast<const void*>(&gemm_ks_kernel<CB, 4>);
    }
}

// The kernel's opt-in to its LDS (above 64 KiB), once per device and kernel: ~1 us of host time.
static void ks_lds_optin(const void* fn, int mt, int cb)
{
    static std::atomic<uint32_t> done[64];
    int dev = 0;
    (void)hipGetDevice(&dev);
    const uint32_t bit = 1u << (4 * cb + mt - 1);
    if (dev < 64 && (done[dev].load(std::memory_order_relaxed) & bit)) return;
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, ks_lds(mt));
    (void)hipGetLastError();
    if (e == hipSuccess && dev < 64) done[dev].fetch_or(bit, std::memory_order_relaxed);
}

size_t gemm_ks_shard_bytes(int rows, int ic, int oc) { return ks_shard_bytes(rows, ic, oc, device_cus()); }

int gemm_ks_dispatch(const uint16_t* A, const GemvShard* shards, int nshards, int rows, char* ws, size_t ws_bytes,
                     hipStream_t stream, const char* what)
{
    return ks_plan(A, shards, nshards, rows, ws, ws_bytes, what, device_cus(), [&](const KsLaunch& L) {
        hipLaunchKernelGGL(ks_prep_kernel, dim3(L.prep->nblk, L.prep->mtt, L.prep->nsh), dim3(512), 0,
                           stream, *L.prep);
        int rc = check_launch(what);
        if (rc != EXL3_OK) return rc;
        const void* fn = L.cb == CB_MCG ? ks_fn<CB_MCG>(L.mt) : ks_fn<CB_3INST>(L.mt);
        ks_lds_optin(fn, L.mt, L.cb);
        KsArgs a = *L.args;
        void* kargs[] = {&a};
        (void)hipLaunchKernel(fn, dim3((unsigned)L.G), dim3(128 * KS_NP), kargs, ks_lds(L.mt), stream);
        rc = check_launch(what);
        if (rc != EXL3_OK || a.nrem == 0) return rc;
        hipLaunchKernelGGL(ks_finish_kernel, dim3(4 * L.mt, a.nrem), dim3(256), 0, stream, a, L.mt);
        return check_launch(what);
    });
}

}  // namespace exl3
