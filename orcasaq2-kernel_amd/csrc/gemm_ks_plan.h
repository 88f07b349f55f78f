// Work plan of the K-split decode-GEMM (gemm_ks.hip): row tiles, the split of a launch's work
// into workgroup ranges and wave runs, the launch argument blocks, every global and LDS index
// the kernels form, the workspace layout, and the host-side grouping of shards into launches.
//
// Plain integer arithmetic marked __host__ __device__ (or host-only planning): the kernels call
// these functions, and the CPU address replay (replay/addr_replay.hip) calls the very same ones
// to walk every workgroup, wave and lane of a launch.
#pragma once

#include <algorithm>

#include "exl3_launch.h"

namespace exl3 {

#define KS_HD __host__ __device__ __forceinline__

constexpr int KS_MAXSH = 8;        // shards per launch
constexpr int KS_PIN = 32;         // inputs per step (two tile rows)
constexpr int KS_LDQ = 36;         // floats per staged column of 32 rows (padded)
constexpr int KS_LDC = 132;        // floats per row of the output staging
// Least steps per pair a launch is spread for: below, splitting further costs more in slots than
// it saves in steps (2048 -> 2048 at 24 rows, 1 / 2 / 4 steps: 13.5 / 12.6 / 13.7 us per call;
// 2048 -> 2048 + 2 x 512 at 128 rows, 2 / 4 / 8: 24.4 / 21.7 / 23.6).
KS_HD constexpr int ks_min_steps(int mt) { return mt == 1 ? 2 : 4; }
constexpr int KS_NP = 4;           // wave pairs of a workgroup: a pair shares its steps, 64 outputs each wave
constexpr int KS_WBYTES = 2048;    // LDS of a wave's trellis words of one step (64 lanes x 8 words)

// LDS ring of a workgroup with row tiles of 32 * mt rows: a stage holds each pair's A fragments
// of one step (2 mt of 1 KiB) and each wave's words of the next; as many stages as fit 160 KiB.
KS_HD constexpr int ks_stage_bytes(int mt) { return KS_NP * mt * 2048 + 2 * KS_NP * KS_WBYTES; }
KS_HD constexpr int ks_nb(int mt) { return mt == 1 ? 6 : 163840 / ks_stage_bytes(mt); }
KS_HD constexpr int ks_lds(int mt) { return ks_nb(mt) * ks_stage_bytes(mt); }
KS_HD constexpr int ks_stage_a(int mt, int st, int pair) { return st * ks_stage_bytes(mt) + pair * mt * 2048; }
KS_HD constexpr int ks_stage_w(int mt, int st, int wave)
{
    return st * ks_stage_bytes(mt) + KS_NP * mt * 2048 + wave * KS_WBYTES;
}
// A lane's K words of a step reach LDS as one run of 16 bytes a lane (K = 1: 4 bytes), for
// K >= 5 a second one 1 KiB further: direct-to-LDS loads exist for 4 and 16 bytes, so K = 2 loads
// its chunk's pair, K = 3 the word before its chunk too (the first chunk of a tile: the word
// after), and the second run overlaps the first for K < 8.  First word of run r, from the
// chunk's first word.
KS_HD constexpr int ks_w_run(int K, int r, int lane)
{
    if (r == 1) return K - 4;
    if (K == 2) return -2 * (lane & 1);
    if (K == 3) return (lane & 7) ? -1 : 0;
    return 0;
}
KS_HD constexpr int ks_w_runs(int K) { return K > 4 ? 2 : 1; }
// Byte offset of word i of lane l's chunk inside the wave's area.
KS_HD constexpr int ks_w_off(int K, int i, int lane)
{
    if (K == 1) return 4 * lane;
    const int r = i >= 4;
    return 1024 * r + 16 * lane + 4 * (i - ks_w_run(K, r, lane));
}

// Division of a non-negative int by a launch constant (a division routine in every wave's
// prologue costs more than the loads behind it).
struct KsDiv {
    uint32_t m;
    int sh;
};
KS_HD int ks_div(int x, KsDiv d) { return (int)(((uint64_t)(uint32_t)x * d.m) >> d.sh); }
// P = c q + r cut into c runs.
struct KsCut {
    int q, r;
};

struct KsShard {
    const uint16_t* Ah;        // fp16(H(A * suh)) of this shard in A-fragment order (ks_a_chunk)
    const uint32_t* trellis;   // (ic/16, oc/16, 8K) u32
    const uint16_t* svh;       // (oc)
    uint16_t* C;               // (rows, ldc), columns [0, oc)
    long ldc;
    int tc, cbeg, K;           // tile columns, first 128-output column group of the shard, bits
};

// A segment is one row tile of one column group (128 outputs of one shard): P = ic / 32 steps.
// Segments are numbered column group first (over the launch's shards), then row tile, so that
// the row tiles of the same weights are neighbours.  Each of the G workgroups takes `full`
// whole segments; the nrem segments left over are split over all the workgroups' pairs, each
// segment over a run of whole pairs (a workgroup's worth at least, as nrem < G), so a
// workgroup's pairs meet at most two of them.
struct KsArgs {
    float* slots;              // (nrem + G) x MT x 32 x 128 fp32 partial sums
    int rows, P, mtt;          // mtt: 32-row tiles in all (row tiles x MT)
    int bf;                    // outputs are bfloat16
    int nrt, nshards, G, full, nrem;
    // the split segments' pairs and steps: the first pextra of them have pbase + 1 pairs, the
    // others pbase; among c pairs the first P % c have P / c + 1 steps, the others P / c
    int pbase, pextra;
    KsDiv dbase, dbase1, dnrt;  // division by pbase, pbase + 1, nrt
    KsCut whole, cbase, cbase1; // P cut into KS_NP, pbase, pbase + 1 runs
    KsShard sh[KS_MAXSH];
};

struct KsPrepArgs {
    const uint16_t* A;
    int rows, ic, nsh, nblk, mtt;
    int bf;                    // A is bfloat16
    const uint16_t* suh[KS_MAXSH];
    uint16_t* Ah[KS_MAXSH];
};

// First pair of split segment s (the pairs of all workgroups in order), its pair count, and the
// split segment of pair j.
KS_HD int ks_pair0(const KsArgs& a, int s) { return s * a.pbase + (s < a.pextra ? s : a.pextra); }
KS_HD int ks_npairs(const KsArgs& a, int s) { return a.pbase + (s < a.pextra); }
KS_HD int ks_seg_of(const KsArgs& a, int j)
{
    const int big = a.pextra * (a.pbase + 1);
    return j < big ? ks_div(j, a.dbase1) : a.pextra + ks_div(j - big, a.dbase);
}
// The cut of a split segment's steps among its pairs.
KS_HD const KsCut& ks_cut(const KsArgs& a, int s) { return s < a.pextra ? a.cbase1 : a.cbase; }
// First step of run k of a cut, and the most steps of any run.
KS_HD int ks_run(const KsCut& c, int k) { return k * c.q + (k < c.r ? k : c.r); }
KS_HD int ks_run_max(const KsCut& c) { return c.q + (c.r > 0); }

// Workgroup of launch slot b of G: slots go to the 8 XCDs in turn, so each XCD gets a
// contiguous block of ranges (neighbouring row tiles and column groups share its L2).
KS_HD int ks_logical(int b, int G) { return (G & 7) ? b : (b & 7) * (G >> 3) + (b >> 3); }

KS_HD int ks_shard_of(const KsArgs& a, int c)
{
    int si = 0;
#pragma unroll
    for (int i = 1; i < KS_MAXSH; i++)
        if (i < a.nshards && c >= a.sh[i].cbeg) si = i;
    return si;
}

// Segment seg of the launch: row tile, shard and its column group.
struct KsSeg {
    int rt, si, cg;
};
KS_HD KsSeg ks_seg(const KsArgs& a, int seg)
{
    KsSeg s;
    const int c = ks_div(seg, a.dnrt);
    s.rt = seg - c * a.nrt;
    s.si = ks_shard_of(a, c);
    s.cg = c - a.sh[s.si].cbeg;
    return s;
}

// 16-byte chunk of Ah that lane l loads for step p, 32-row tile m (of mtt), half f: row
// l % 32 of the tile, inputs 32 p + 16 (l / 32) + 8 f .. + 7.
KS_HD long ks_a_chunk(int p, int mtt, int m, int f, int lane) { return (((long)p * mtt + m) * 2 + f) * 64 + lane; }

// First u32 of the chunk lane l decodes of half u (64 outputs) of a column group at step p:
// chunk l % 8 of tile (2 p + l / 32, 8 cg + 4 u + (l % 32) / 8).
KS_HD long ks_b_word(int p, int lane, int tc, int cg, int u, int K)
{
    return ((long)(2 * p + (lane >> 5)) * tc + 8 * cg + 4 * u + ((lane & 31) >> 3)) * (8 * K) + (lane & 7) * K;
}

// Partial sums.  A lane's accumulator of the column half h holds rows 8 j + 4 (l / 32) + e
// (register 4 j + e) of column position 32 (2 u + h) + l % 32, u the wave's half of the group; a
// quad is four consecutive rows.  Staged: float offset of (pair, column position, quad).
KS_HD int ks_red(int pair, int cpos, int quad) { return (pair * 128 + cpos) * KS_LDQ + 4 * quad; }
// Output of the column group at a column position (the chunk of lane n gives columns n % 8 and
// n % 8 + 8 of tile n / 8).
KS_HD int ks_out_col(int cpos)
{
    const int n = cpos & 31;
    return 64 * (cpos >> 6) + 16 * (n >> 3) + 8 * ((cpos >> 5) & 1) + (n & 7);
}
// Slot of (split segment, workgroup), in 16-byte units, and (quad of the row tile, column
// position) inside it.  A workgroup's pairs hold consecutive split segments and a segment
// consecutive pairs, so s + g names each (segment, workgroup) once.
KS_HD long ks_slot(int s, int g, int mt) { return (long)(s + g) * mt * 1024; }
KS_HD int ks_slot_in(int quad, int cpos) { return quad * 128 + cpos; }

// Set-up: lane l of wave v holds inputs 8 (l % 16) .. + 7 of 128-input block b for row 4 v + l / 16
// of 32-row tile m.
KS_HD long ks_prep_chunk(const KsPrepArgs& a, int b, int m, int row, int l16)
{
    return ks_a_chunk(4 * b + (l16 >> 2), a.mtt, m, l16 & 1, 32 * ((l16 >> 1) & 1) + row);
}

// ---------------------------------------------------------------- host: tiles, workspace, plan

inline size_t ks_align(size_t x) { return (x + 255) & ~(size_t)255; }

// Rows as nrt row tiles of 32 * mt rows: at most 128 rows per tile (a taller tile's
// accumulators do not fit), the tiles as even as whole 32-row blocks allow.
struct KsRows {
    int nrt, mt;
};
inline KsRows ks_rows(int rows)
{
    const int nrt = (rows + 127) / 128;
    return KsRows{nrt, ((rows + nrt - 1) / nrt + 31) / 32};
}

inline size_t ks_ah_bytes(int rows, int ic)
{
    const KsRows t = ks_rows(rows);
    return ks_align((size_t)t.nrt * t.mt * 32 * ic * 2);
}

// Workgroups of a launch: one per CU, fewer where a pair would get under ks_min_steps steps.
inline int ks_wgs(long steps, int mt, int cus)
{
    return (int)std::min<long>(cus, std::max<long>(1, steps / (KS_NP * ks_min_steps(mt))));
}

// A shard's share of a call's workspace: its activations, and slots for its segments and the
// workgroups of a launch.
inline size_t ks_shard_bytes(int rows, int ic, int oc, int cus)
{
    const KsRows t = ks_rows(rows);
    return ks_ah_bytes(rows, ic) + (size_t)2 * cus * t.mt * 16384;
}

// Division by d of anything below 2^31 (Granlund and Montgomery): multiply by m, shift by sh.
inline KsDiv ks_magic(uint32_t d)
{
    int l = 0;
    while ((1ull << l) < d) l++;
    return KsDiv{(uint32_t)(((1ull << (31 + l)) / d) + 1), 31 + l};
}

struct KsLaunch {
    int mt, cb, G;
    const KsArgs* args;       // decode launch of G workgroups; finishing launch of 4 mt x nrem
    const KsPrepArgs* prep;   // set-up launch of nblk x mtt x nsh workgroups
};

// Shards that read the same A (rows x ic): per codebook, groups of up to KS_MAXSH shards, each
// one set-up, one decode and (where segments are split) one finishing launch.
template <class Emit>
int ks_plan(const uint16_t* A, const GemvShard* shards, int nshards, int rows, char* ws, size_t ws_bytes,
            const char* what, int cus, Emit&& emit)
{
    const int ic = shards[0].ic;
    const KsRows t = ks_rows(rows);
    const size_t ah = ks_ah_bytes(rows, ic);
    bool done[EXL3_MAX_SHARDS] = {false};
    size_t off = 0;
    for (int i = 0; i < nshards; i++) {
        if (done[i]) continue;
        KsArgs a = {};
        KsPrepArgs p = {};
        a.rows = p.rows = rows;
        a.bf = p.bf = shards[i].bf;
        a.P = ic / KS_PIN;
        a.mtt = p.mtt = t.nrt * t.mt;
        p.A = A;
        p.ic = ic;
        p.nblk = ic / 128;
        int ncg = 0;
        for (int s = i; s < nshards && a.nshards < KS_MAXSH; s++) {
            const GemvShard& d = shards[s];
            if (done[s] || d.cb != shards[i].cb) continue;
            if (d.K < 1 || d.K > 8) return set_error(EXL3_ERR_ARG, "%s: K=%d is not in 1..8", what, d.K);
            p.suh[a.nshards] = d.suh;
            p.Ah[a.nshards] = reinterpret_cast<uint16_t*>(ws + off);
            off += ah;
            a.sh[a.nshards++] = KsShard{p.Ah[p.nsh], d.trellis, d.svh, d.C, d.ldc, d.oc / 16, ncg, d.K};
            p.nsh++;
            ncg += d.oc / 128;
            done[s] = true;
        }
        a.nrt = t.nrt;
        const int nsegs = t.nrt * ncg;
        a.G = ks_wgs((long)nsegs * a.P, t.mt, cus);
        a.full = nsegs / a.G;
        a.nrem = nsegs % a.G;
        const int np = KS_NP * a.G;
        a.pbase = a.nrem ? np / a.nrem : 1;
        a.pextra = a.nrem ? np % a.nrem : 0;
        a.dbase = ks_magic(a.pbase);
        a.dbase1 = ks_magic(a.pbase + 1);
        a.dnrt = ks_magic(a.nrt);
        a.whole = KsCut{a.P / KS_NP, a.P % KS_NP};
        a.cbase = KsCut{a.P / a.pbase, a.P % a.pbase};
        a.cbase1 = KsCut{a.P / (a.pbase + 1), a.P % (a.pbase + 1)};
        a.slots = reinterpret_cast<float*>(ws + off);
        if (a.nrem) off += (size_t)(a.nrem + a.G) * t.mt * 16384;
        if (off > ws_bytes)
            return set_error(EXL3_ERR_WORKSPACE, "%s: workspace of %zu bytes, %zu needed", what, ws_bytes, off);
        const KsLaunch L = {t.mt, shards[i].cb, a.G, &a, &p};
        const int rc = emit(L);
        if (rc != EXL3_OK) return rc;
    }
    return EXL3_OK;
}

}  // namespace exl3
