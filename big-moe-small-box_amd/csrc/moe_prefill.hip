// Prefill-size expert products: grouped GEMMs on the MFMA units over EXL3 trellis weights, each weight decoded once per
// workgroup, straight into the MFMA operand registers of the wave that multiplies it (below, "grouped GEMM"). fp32
// accumulation; each output element is one fixed sum (k ascending in MFMA blocks), independent of scheduling.
//
//   k_pf_prep_tok : rotated gate / up inputs of every dispatch row, xt = RN16(H128(x * suh) * R), token-major
//   k_pf_gemm<false> : gate or up products of one 256-column block -> fp16 [row][128-block][gate | up][128]
//   (k_gu_epi)    : fp16 gate / up -> epilogue -> fp16 down-input rows (shared with the decode path)
//   k_pf_gemm<true>  : down products of one 256-column block -> fp32 [row][128-block][128]
//   (k_dn_combine): rotation * svh, slots summed in slot order (shared with the decode path)
#include "moe_kernels.hpp"

#include <algorithm>

namespace bmx {

constexpr int PF_M = 128;                    // rows per group

// Workgroups are handed to the 8 XCDs round-robin (block b runs on XCD b % 8). Renumber so that chunks of 16
// consecutive logical blocks (the column blocks of one row group) share an XCD, and the chunks go round-robin over the
// XCDs: a group's units read its A rows through one L2, and the groups that exist (the grid is sized for the most a batch
// can have) spread over all XCDs. Blocks past the last whole 128-block round keep their number.
__device__ __forceinline__ int xcd_block(int bid, int nblk)
{
    constexpr int C = 16;
    if (bid >= nblk / (8 * C) * (8 * C)) return bid;
    const int xcd = bid % 8, i = bid / 8;
    return ((i / C) * 8 + xcd) * C + i % C;
}

// ---- rotated inputs: 16 lanes per (row, matrix, run of PREP_BPU 128-blocks), 8 consecutive inputs per lane -------------
__global__ __launch_bounds__(256) void k_pf_prep(GvArgs a)
{
    prep_unit(a, (long)blockIdx.x * 16 + (threadIdx.x >> 4));
}

static dim3 prep_grid(int R_max, int H)
{
    return dim3((unsigned)(((long)2 * R_max * ((H / 128 + PREP_BPU - 1) / PREP_BPU) + 15) / 16));
}

// ---- rotated inputs, token-major (the prefill path) --------------------------------------------------------------------
// Unit u = (token, run of PREP_BPU 128-blocks) by a 16-lane group: the token's inputs are loaded once and rotated into
// the rows of all its picks and its shared-expert row, gate and up (the same values as prep_unit, which reads the
// token's inputs once per row and matrix, 12 times at top-6: 441 MB of HBM reads for C3's 805 MB of rows, 205 MB
// here). Lane j first fetches slot k0 + j's row and its expert's suh addresses, so the dependent index loads run once
// per 16 slots, side by side; the slot loop takes them by shuffles within the group.
__device__ __forceinline__ void prep_tok_unit(const GvArgs& a, long u)
{
    const int nblk = a.H / 128, nrun = (nblk + PREP_BPU - 1) / PREP_BPU;
    const int j = threadIdx.x & 15, run = (int)(u % nrun);
    const long t = u / nrun;
    if (t >= a.T) return;                 // the whole 16-lane group: the shuffles below stay inside it
    float xv[PREP_BPU][8];
    const uint16_t* xr = a.x + (size_t)t * a.H + 8 * j;
#pragma unroll
    for (int i = 0; i < PREP_BPU; ++i)
        if (run * PREP_BPU + i < nblk) unpack8(ldg4(xr + 128 * (run * PREP_BPU + i)), xv[i]);
    const int ns = a.topk + (a.has_shared ? 1 : 0);
    for (int k0 = 0; k0 < ns; k0 += 16)
    {
        const int kj = k0 + j;
        int rj = -1;
        if (kj < a.topk) rj = a.inv[t * a.topk + kj];
        else if (kj < ns) rj = a.offsets[a.E] + (int)t;
        uint64_t su0 = 0, su1 = 0;
        if (rj >= 0)
        {
            const int e = a.row_expert[rj];
            const bmx_expert& ex = e == a.E ? *a.shared : a.experts[e];
            su0 = reinterpret_cast<uint64_t>(ex.suh[0]);
            su1 = reinterpret_cast<uint64_t>(ex.suh[1]);
        }
        const int kn = ns - k0 < 16 ? ns - k0 : 16;
        for (int k = 0; k < kn; ++k)
        {
            const int r = __shfl(rj, k, 16);
            if (r < 0) continue;              // a dropped pick: no row
#pragma unroll
            for (int mat = 0; mat < 2; ++mat)
            {
                const uint64_t sa = mat ? su1 : su0;
                const uint32_t lo = __shfl((uint32_t)sa, k, 16), hi = __shfl((uint32_t)(sa >> 32), k, 16);
                const uint16_t* su = reinterpret_cast<const uint16_t*>(((uint64_t)hi << 32) | lo) + 8 * j;
                uint16_t* dst = a.xt + ((size_t)mat * a.R_max + r) * a.H + 8 * j;
#pragma unroll
                for (int i = 0; i < PREP_BPU; ++i)
                {
                    const int b = run * PREP_BPU + i;
                    if (b >= nblk) break;
                    float v[8], s[8];
                    unpack8(ldg4(su + 128 * b), s);
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[q] = xv[i][q] * s[q];
                    had128_x8(v);
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[q] = v[q] * (R_SCALE * had128_x8_sign());
                    __builtin_nontemporal_store(pack8_r(v), reinterpret_cast<u32x4*>(dst + 128 * b));
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_pf_prep_tok(GvArgs a)
{
    prep_tok_unit(a, (long)blockIdx.x * 16 + (threadIdx.x >> 4));
}

static dim3 prep_tok_grid(int T, int H)
{
    const long units = (long)T * ((H / 128 + PREP_BPU - 1) / PREP_BPU);
    return dim3((unsigned)std::max(1L, (units + 15) / 16));
}

// Step barrier: the wave's LDS operations are done (its global loads, register prefetches for later steps, may still be in
// flight; the compiler waits for those where their registers are used).
__device__ __forceinline__ void step_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0); vmcnt (63) and expcnt (7) at their maxima: no wait
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// ---- grouped GEMM ----------------------------------------------------------------------------------------------------
// Work unit: (group of <= 128 rows, matrix, 256-column block); 4 waves, all alike, two workgroups per CU. Wave w owns the
// columns of parity w & 1 (strip half) of 128-column block w >> 1, all rows of the group, and decodes its weights straight
// into the B operand registers of v_mfma_f32_32x32x16_f16: lane L holds the strip of tile-row L / 32 of a pair of tile-rows
// (32 k), so an operand's k index 8 (L / 32) + j is input row 8 q + j of that tile-row (q: the strip's upper or lower
// eight rows), and its column is the lane's strip column. No B fragment passes through the LDS, and no weight is decoded
// twice in a workgroup. The A rows (64 k at a time) are staged in LDS in operand order and shared by the 4 waves.
// What bounds it: the decode (115 VALU per 32 k and wave) and the MFMAs (16 at 128 rows) of two waves overlap on a SIMD, and
// the chip then runs into its power limit (the shader clock falls to 1.7-1.9 GHz, VALU 0.7 busy, MFMA 0.45). Layer times, four
// MFMA and eight decode waves handing B over through LDS -> eight equal waves of 512 columns -> decode and products
// interleaved -> this: 8,192 tokens (384 experts, top-6, H 4096, I 2048, K 2 / 3) 5,008 -> 4,427 -> 4,192 -> 4,135 us; 517
// tokens 1,878 -> 1,433 -> 1,401 -> 1,336; 2,048 tokens (H 5120, I 2304, K 2.5 / 2) 3,612 -> 2,959 -> 2,903 -> 2,755. Units of
// at most 32 rows without stages and barriers, as the mid-size kernel runs them: the same time (the clock is the limit).
// The scheduling fences keep a pair's operand reads, decode and products apart: the compiler otherwise moves two pairs'
// decodes together and spills.
constexpr int PF_WAVES = 4;
constexpr int PF_KSTEP = 64;                               // k per LDS stage
constexpr int PF_SUBS = PF_KSTEP / 32;                     // pairs of tile-rows per stage
constexpr int PF_ST_U4 = PF_M * PF_KSTEP / 8;              // a stage, 16-byte chunks: [sub][q][row block][64 lanes]
constexpr int PF_COLS = 256;                               // output columns of a unit
// the products on their way out: rows of 256 columns, padded by 16 bytes (fp16: 128 rows; fp32: 64 rows at a time)
constexpr int PF_OUT_H = PF_COLS * 2 + 16, PF_OUT_F = PF_COLS * 4 + 16;
constexpr int PF_LDS = PF_M * PF_OUT_H > 2 * PF_ST_U4 * 16 ? PF_M * PF_OUT_H : 2 * PF_ST_U4 * 16;
static_assert(PF_OUT_F * PF_M / 2 <= PF_LDS, "half the rows in fp32 fit");
__shared__ u32x4 pf_lds[PF_LDS / 16];

struct PfJob {
    int g, mat, cb, e, r0, nr, K, N, nb128;
    const bmx_expert* ex;
};

// Words of a half strip: stream positions 32 HALF .. 32 HALF + 31 of the lane's strip and the 16 bits before them. W0:
// the first of the strip's words that the half reads (-1: the last word of the strip before it, the ring's wrap included).
// rows: the tile-rows' address (the same on every lane); strip, prev: the lane's offsets of the strip and of the word
// before it.
template <int F, int HALF> struct HalfWords {
    static constexpr int Q0 = ring_end<F>(32 * HALF) - 16, Q1 = ring_end<F>(32 * HALF + 31);   // first, last + 1 bit
    static constexpr int W0 = Q0 < 0 ? -1 : Q0 / 32, W1 = (Q1 + 31) / 32, NW = W1 - W0;
    typedef uint32_t Buf[NW];
};

template <int F, int HALF>
__device__ __forceinline__ void load_half(typename HalfWords<F, HALF>::Buf& w, const uint8_t* rows, uint32_t strip, uint32_t prev)
{
    using S = HalfWords<F, HALF>;
#pragma unroll
    for (int i = 0; i < S::NW; ++i) w[i] = S::W0 + i < 0 ? ldg(rows + prev, 0) : ldg(rows + strip, S::W0 + i);
}

// B operand (CI, Q) of a half strip: the eight input rows 8 Q .. + 7 of strip column HALF + 2 CI, four pairs of weights.
template <int F, int HALF, int CI, int Q>
__device__ __forceinline__ u32x4 decode_b(const typename HalfWords<F, HALF>::Buf& w)
{
    using S = HalfWords<F, HALF>;
    constexpr RingTab<F> tab;
    uint32_t own[S::NW];
#pragma unroll
    for (int k = 0; k + 1 < S::NW; ++k) own[k] = w[k + 1];
    own[S::NW - 1] = 0u;
    u32x4 b;
#pragma unroll
    for (int g = 0; g < 4; ++g)
    {
        const int j = 32 * HALF + 8 * g + 4 * CI + 2 * Q;      // strip_cidx(j) = HALF + 2 CI, strip_dw(j) = g + 4 Q
        // window bit 0 is the first bit of w[0]: strip word W0 (tab.q counts from the word before the strip)
        b[g] = cb_pair(win_state(w[0], own, tab.q[j] - 32 - 32 * S::W0),
                       win_state(w[0], own, tab.q[j + 1] - 32 - 32 * S::W0));
    }
    return b;
}

// A rows of a stage: thread t copies 16-byte chunk t & 7 of row t >> 3 of every row block (128 bytes of a row per 8
// lanes). In LDS chunk c = 4 sub + 2 h + q of row r is lane 32 h + r % 32 of operand (sub, q, r / 32); lanes are exchanged
// by a XOR with 2 c, which spreads the eight chunks of two rows over the 16 bank groups.
template <int NMB>
__device__ __forceinline__ void pf_stage_load(u32x4 (&st)[NMB], const uint16_t* rows, int K, uint32_t off, uint32_t last,
                                              int k0)
{
#pragma unroll
    for (int m = 0; m < NMB; ++m)
        st[m] = ldg4(reinterpret_cast<const char*>(rows + (size_t)(32 * m) * K + k0) + (m + 1 < NMB ? off : last));
}

template <int NMB>
__device__ __forceinline__ void pf_stage_store(const u32x4 (&st)[NMB], u32x4* __restrict__ lds)
{
    const int r = threadIdx.x >> 3, c = threadIdx.x & 7;
#pragma unroll
    for (int m = 0; m < NMB; ++m)
        lds[(((c >> 2) * 2 + (c & 1)) * 4 + m) * 64 + 32 * ((c >> 1) & 1) + (r ^ (2 * c))] = st[m];
}

// One operand slot of a wave: operand (CI, Q) of the words w is decoded into b while the products of the operand before
// it (bp, columns 1 - CI, rows ap) run, one MFMA per 28 / NMB VALU instructions: the two waves of a SIMD march in step
// from barrier to barrier, so an MFMA burst and a decode burst would each leave the other unit idle.
template <int F, int HALF, int CI, int Q, int NMB>
__device__ __forceinline__ void pf_slot(const typename HalfWords<F, HALF>::Buf& w, u32x4& b, const u32x4& bp,
                                        const f16x8 (&ap)[NMB], f32x16 (&acc)[2][NMB])
{
    b = decode_b<F, HALF, CI, Q>(w);
#pragma unroll
        for (int m = 0; m < NMB; ++m)
            acc[1 - CI][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ap[m], __builtin_bit_cast(f16x8, bp), acc[1 - CI][m],
                                                                    0, 0, 0);
#pragma unroll
        for (int m = 0; m < NMB; ++m)
        {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);            // MFMA
            __builtin_amdgcn_sched_group_barrier(0x2, 28 / NMB, 0);     // VALU
        }
    __builtin_amdgcn_sched_barrier(0);
}

// The A operands (q) of pair j of a stage
template <int NMB>
__device__ __forceinline__ void pf_a_read(f16x8 (&a)[NMB], const u32x4* __restrict__ lds, int j, int q)
{
    const int lane = threadIdx.x & 63, h = lane >> 5;
#pragma unroll
    for (int m = 0; m < NMB; ++m)
        a[m] = __builtin_bit_cast(f16x8, lds[((2 * j + q) * 4 + m) * 64 + 32 * h +
                                             ((lane & 31) ^ (2 * (4 * j + 2 * h + q)))]);
    __builtin_amdgcn_sched_barrier(0);        // read a slot ahead of their use
}

// The unit's k-loop of one wave, NMB 32-row blocks: stages of 64 k, two pairs of tile-rows each, two stages per trip. The
// words of a pair are requested four pairs ahead (each register set again right after its use), the A rows one stage
// ahead; one barrier per stage. WORK false: a wave without columns (past the matrix's last block), which only copies A
// rows.
template <int F, int HALF, int NMB, bool WORK>
__device__ __forceinline__ void pf_loop(const PfJob& jb, const uint8_t* mat_base, const uint16_t* asrc, int cbo,
                                        f32x16 (&acc)[2][NMB])
{
    constexpr int TB = Fmt<F>::TB;
    using S = HalfWords<F, HALF>;
    const int lane = threadIdx.x & 63, h = lane >> 5, t = (lane >> 2) & 7, s = lane & 3;
    const uint32_t row_bytes = (uint32_t)(jb.N / 16) * TB;
    // offsets from wave-uniform addresses; the word before a strip is the tile's last one for its first strip
    const uint32_t strip = (uint32_t)h * row_bytes + (uint32_t)(cbo * 8 + t) * TB + (uint32_t)s * (TB / 4);
    const uint32_t prev = s ? strip - 4 : strip + TB - 4;
    const int KT = jb.K / (2 * PF_KSTEP);
    const uint16_t* rows = asrc + (size_t)jb.r0 * jb.K;
    // the thread's row in a row block; in the last block rows past the group's end read its last row
    const int r = threadIdx.x >> 3;
    const uint32_t off = 2u * ((uint32_t)r * (uint32_t)jb.K + 8u * (threadIdx.x & 7));
    const uint32_t last = 2u * ((uint32_t)min(r, jb.nr - 1 - 32 * (NMB - 1)) * (uint32_t)jb.K + 8u * (threadIdx.x & 7));
    u32x4 st[NMB];
    typename S::Buf w[2 * PF_SUBS];
    u32x4 b0, b1;
    f16x8 a0[NMB], a1[NMB];
    pf_stage_load<NMB>(st, rows, jb.K, off, last, 0);
    if (WORK)
    {
#pragma unroll
        for (int j = 0; j < 2 * PF_SUBS; ++j)
            load_half<F, HALF>(w[j], mat_base + (size_t)(2 * j) * row_bytes, strip, prev);
        // the pipeline starts with an operand of zeros (its products add nothing)
        b1 = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int m = 0; m < NMB; ++m) a1[m] = f16x8{};
    }
    pf_stage_store<NMB>(st, pf_lds);
    step_barrier();
    for (int i = 0; i < KT; ++i)
    {
        const int in = min(i + 1, KT - 1);          // past the last trip: its own loads again, never used
        const uint8_t* pn = mat_base + (size_t)(4 * PF_SUBS) * in * row_bytes;
#pragma unroll
        for (int g = 0; g < 2; ++g)
        {
            const u32x4* lds = pf_lds + g * PF_ST_U4;
            pf_stage_load<NMB>(st, rows, jb.K, off, last, g == 0 ? (2 * i + 1) * PF_KSTEP : 2 * in * PF_KSTEP);
            if (WORK)
            {
#pragma unroll
                for (int j = 0; j < PF_SUBS; ++j)
                {
                    typename S::Buf& wj = w[PF_SUBS * g + j];
                    // the words stay allocated until here (a load in flight into a register that is free again would
                    // force a wait)
#pragma unroll
                    for (int k = 0; k < S::NW; ++k) asm volatile("" :: "v"(wj[k]));
                    pf_a_read<NMB>(a0, lds, j, 0);
                    pf_slot<F, HALF, 0, 0, NMB>(wj, b0, b1, a1, acc);
                    pf_slot<F, HALF, 1, 0, NMB>(wj, b1, b0, a0, acc);
                    pf_a_read<NMB>(a1, lds, j, 1);
                    pf_slot<F, HALF, 0, 1, NMB>(wj, b0, b1, a0, acc);
                    pf_slot<F, HALF, 1, 1, NMB>(wj, b1, b0, a1, acc);
                    load_half<F, HALF>(wj, pn + (size_t)(2 * (PF_SUBS * g + j)) * row_bytes, strip, prev);
                }
            }
            pf_stage_store<NMB>(st, pf_lds + (1 - g) * PF_ST_U4);
            step_barrier();
        }
    }
    if (WORK)
#pragma unroll
        for (int m = 0; m < NMB; ++m)
            acc[1][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1[m], __builtin_bit_cast(f16x8, b1), acc[1][m], 0, 0, 0);
}

// The unit's products out of the accumulators, through LDS (the A stages are done with) so that whole rows of the unit's
// columns are stored 16 bytes per lane: accumulator element v of lane L is row 8 (v / 4) + 4 (L / 32) + v % 4 of its row
// block, column lane_col(L, HALF + 2 ci) of the wave's 128-column block. Gate / up products are stored as fp16 (the value
// the epilogue would round them to), down products as fp32, 64 rows at a time.
template <bool DOWN, int NMB>
__device__ __forceinline__ void pf_out(const GvArgs& a, const PfJob& jb, const f32x16 (&acc)[2][NMB])
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    char* lds = reinterpret_cast<char*>(pf_lds);
    constexpr int RB = DOWN ? 2 : NMB;                                // row blocks per round
    constexpr int ES = DOWN ? 4 : 2, RS = DOWN ? PF_OUT_F : PF_OUT_H;
#pragma unroll
    for (int m0 = 0; m0 < NMB; m0 += RB)
    {
        if (m0) step_barrier();                                       // the round before is read out
#pragma unroll
        for (int m = m0; m < NMB && m < m0 + RB; ++m)
#pragma unroll
            for (int ci = 0; ci < 2; ++ci)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                {
                    const int row = 32 * (m - m0) + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                    const int col = 128 * (wave >> 1) + lane_col(lane, (wave & 1) + 2 * ci);
                    char* p = lds + row * RS + col * ES;
                    if (DOWN) *reinterpret_cast<float*>(p) = acc[ci][m][v];
                    else *reinterpret_cast<uint16_t*>(p) = f2h_r(0.0f + acc[ci][m][v]);
                }
        step_barrier();
        // 16-byte pieces: PPR per row; piece q of a row is in 128-column block q / PPB
        constexpr int PPR = PF_COLS * ES / 16, PPB = PPR / 2;
        const int rows = min(jb.nr - 32 * m0, 32 * RB);
        for (int i = threadIdx.x; i < rows * PPR; i += PF_WAVES * 64)
        {
            const int row = i / PPR, q = i % PPR, cbo = 2 * jb.cb + q / PPB;
            if (cbo >= jb.nb128) continue;
            const u32x4 v = *reinterpret_cast<const u32x4*>(lds + row * RS + q * 16);
            const size_t r = (size_t)(jb.r0 + 32 * m0 + row);
            char* out = DOWN ? reinterpret_cast<char*>(a.part_dn + (r * a.NBH + cbo) * 128)
                             : reinterpret_cast<char*>(reinterpret_cast<uint16_t*>(a.part_gu) + (r * a.NB + cbo) * 256 +
                                                       jb.mat * 128);
            *reinterpret_cast<u32x4*>(out + (q % PPB) * 16) = v;
        }
    }
}

template <bool DOWN, int F, int HALF, int NMB>
__device__ __forceinline__ void pf_unit(const GvArgs& a, const PfJob& jb, const uint8_t* base, const uint16_t* asrc, int cbo)
{
    f32x16 acc[2][NMB];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NMB; ++j) acc[i][j] = f32x16{};
    if (cbo < jb.nb128) pf_loop<F, HALF, NMB, true>(jb, base, asrc, cbo, acc);
    else pf_loop<F, HALF, NMB, false>(jb, base, asrc, cbo, acc);
    pf_out<DOWN, NMB>(a, jb, acc);
}

template <bool DOWN, int F, int HALF>
__device__ __forceinline__ void pf_unit_rows(const GvArgs& a, const PfJob& jb, const uint8_t* base, const uint16_t* asrc,
                                             int cbo)
{
    switch ((jb.nr + 31) / 32)
    {
        case 1: pf_unit<DOWN, F, HALF, 1>(a, jb, base, asrc, cbo); break;
        case 2: pf_unit<DOWN, F, HALF, 2>(a, jb, base, asrc, cbo); break;
        case 3: pf_unit<DOWN, F, HALF, 3>(a, jb, base, asrc, cbo); break;
        default: pf_unit<DOWN, F, HALF, 4>(a, jb, base, asrc, cbo); break;
    }
}

template <bool DOWN, int F>
__device__ __forceinline__ void pf_unit_half(const GvArgs& a, const PfJob& jb, const uint8_t* base, const uint16_t* asrc,
                                             int wave)
{
    const int cbo = 2 * jb.cb + (wave >> 1);
    if (wave & 1) pf_unit_rows<DOWN, F, 1>(a, jb, base, asrc, cbo);
    else pf_unit_rows<DOWN, F, 0>(a, jb, base, asrc, cbo);
}

template <bool DOWN>
__global__ __launch_bounds__(PF_WAVES * 64, 2) void k_pf_gemm(GvArgs a)
{
    const int nb128 = DOWN ? a.NBH : a.NB;     // 128-column blocks of the output
    const int NB2 = (nb128 + 1) / 2;
    const int lid = xcd_block(blockIdx.x, gridDim.x);
    PfJob jb;
    jb.nb128 = nb128;
    if (DOWN) { jb.g = lid / NB2; jb.mat = 2; jb.cb = lid % NB2; }
    else { jb.g = lid / (2 * NB2); jb.mat = (lid / NB2) & 1; jb.cb = lid % NB2; }
    if (jb.g >= *a.ngroups) return;
    jb.e = a.groups[3 * jb.g];
    if (group_skipped(a, jb.e)) return;
    jb.r0 = a.groups[3 * jb.g + 1];
    jb.nr = a.groups[3 * jb.g + 2];
    jb.ex = jb.e == a.E ? a.shared : a.experts + jb.e;
    jb.K = DOWN ? a.I : a.H;
    jb.N = DOWN ? a.H : a.I;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint16_t* asrc = DOWN ? a.act_rows : a.xt + (size_t)jb.mat * a.R_max * a.H;
    const uint8_t* base = reinterpret_cast<const uint8_t*>(jb.ex->tr[jb.mat]);
    switch (jb.ex->fmt[jb.mat])
    {
        case BMX_TF_K2: pf_unit_half<DOWN, BMX_TF_K2>(a, jb, base, asrc, wave); break;
        case BMX_TF_K25: pf_unit_half<DOWN, BMX_TF_K25>(a, jb, base, asrc, wave); break;
        case BMX_TF_K3: pf_unit_half<DOWN, BMX_TF_K3>(a, jb, base, asrc, wave); break;
        default: pf_unit_half<DOWN, BMX_TF_K4>(a, jb, base, asrc, wave); break;
    }
}

// ---- mid-size grouped GEMM: groups of <= 32 rows, every wave on its own ------------------------------------------------
// For decode batches of several tokens (a few rows per expert): a wave's unit is (group of <= 32 rows, matrix, 128-column
// block, k-split). Per pair of tile-rows (32 k) a lane holds one whole strip, four columns of 16 rows, and decodes it
// straight into the B operands of eight v_mfma_f32_32x32x16_f16 (lane L: tile-row L / 32, as in the prefill GEMM); the A
// operands, 32 bytes of a row per lane, come from memory (the L1 and L2 hold the few rows). Nothing goes through LDS and
// no wave waits for another, so three waves per SIMD keep the VALU busy, which bounds it: 230 VALU per strip of 64 weights
// and lane. The fp32 products of each k-split go to the partial layout the epilogues sum in split order. The workgroup's
// four waves take consecutive column blocks of the same rows. Against eight waves that decoded
// into LDS between barriers (and spilled): 77 tokens 679 -> 591 us, 8 tokens 195 -> 165, 16 tokens on ~12 experts 102 -> 86.
// No exit test between the two strips of a trip: 8 tokens 165 -> 155.5, 16 tokens 81 -> 77, 77 tokens 540 -> 529.
constexpr int MID_M = 32;
constexpr int MID_WAVES = 4;
constexpr int MID_D = 2;                      // strips of trellis words in flight per wave

// B operand (C, Q) of a whole strip: the eight input rows 8 Q .. + 7 of strip column C
template <int F, int C, int Q>
__device__ __forceinline__ u32x4 strip_b(uint32_t prev, const uint32_t (&own)[Fmt<F>::TB / 16])
{
    constexpr RingTab<F> tab;
    u32x4 b;
#pragma unroll
    for (int g = 0; g < 4; ++g)
    {
        const int j = 32 * (C & 1) + 8 * g + 4 * (C >> 1) + 2 * Q;      // strip_cidx(j) = C, strip_dw(j) = g + 4 Q
        b[g] = cb_pair(win_state(prev, own, tab.q[j]), win_state(prev, own, tab.q[j + 1]));
    }
    return b;
}

template <int F, int C, int Q>
__device__ __forceinline__ void mid_mul(uint32_t prev, const uint32_t (&own)[Fmt<F>::TB / 16], const u32x4& a, f32x16 (&acc)[4])
{
    acc[C] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, strip_b<F, C, Q>(prev, own)),
                                                    acc[C], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);        // one operand's decode at a time: the registers of two would cost a wave per SIMD
}

// pairs of tile-rows s0 .. s0 + n - 1 of the wave's unit (n > 0). ap: the lane's A row at k 16 (L / 32)
template <int F>
__device__ __forceinline__ void mid_run(const PfJob& jb, const uint8_t* mat_base, const uint16_t* ap, int s0, int n,
                                        f32x16 (&acc)[4])
{
    constexpr int TB = Fmt<F>::TB, NW = TB / 16;
    const int lane = threadIdx.x & 63, h = lane >> 5, t = (lane >> 2) & 7, s = lane & 3;
    const size_t pair_bytes = (size_t)(jb.N / 16) * TB * 2;
    const uint8_t* p = mat_base + (size_t)s0 * pair_bytes + h * (pair_bytes / 2) + (size_t)(jb.cb * 8 + t) * TB + s * (TB / 4);
    ap += 32 * s0;
    uint32_t w[MID_D][NW];
    u32x4 a[MID_D][2];
    // past the last pair: the last one again
    auto fetch = [&](int d, int i) {
        const int j = min(i, n - 1);
        load_words(w[d], p + (size_t)j * pair_bytes);
        a[d][0] = ldg4(ap + 32 * j);
        a[d][1] = ldg4(ap + 32 * j + 8);
    };
#pragma unroll
    for (int d = 0; d < MID_D; ++d) fetch(d, d);
    static_assert(MID_D == 2, "n is even: a split is whole k-steps of 64");
    for (int i = 0; i < n; i += MID_D)
#pragma unroll
        for (int d = 0; d < MID_D; ++d)
        {
            const uint32_t prev = __builtin_amdgcn_mov_dpp(w[d][NW - 1], 0x93, 0xf, 0xf, false);
            mid_mul<F, 0, 0>(prev, w[d], a[d][0], acc);
            mid_mul<F, 1, 0>(prev, w[d], a[d][0], acc);
            mid_mul<F, 2, 0>(prev, w[d], a[d][0], acc);
            mid_mul<F, 3, 0>(prev, w[d], a[d][0], acc);
            mid_mul<F, 0, 1>(prev, w[d], a[d][1], acc);
            mid_mul<F, 1, 1>(prev, w[d], a[d][1], acc);
            mid_mul<F, 2, 1>(prev, w[d], a[d][1], acc);
            mid_mul<F, 3, 1>(prev, w[d], a[d][1], acc);
            fetch(d, i + d + MID_D);
        }
}

// One unit of the mid-size GEMM: (group or heavy-expert chunk, matrix, four 128-column blocks, k-split) from its index lid.
template <bool DOWN>
__device__ __forceinline__ void mid_unit(const GvArgs& a, int lid)
{
    const int nb128 = DOWN ? a.NBH : a.NB;
    const int NB4 = (nb128 + MID_WAVES - 1) / MID_WAVES, KS = DOWN ? a.KS_dn : a.KS_gu;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int ksp = lid % KS;
    lid /= KS;
    PfJob jb;
    jb.nb128 = nb128;
    jb.cb = lid % NB4 * MID_WAVES + wave;
    lid /= NB4;
    jb.mat = DOWN ? 2 : lid & 1;
    jb.g = DOWN ? lid : lid >> 1;
    if (jb.cb >= nb128) return;
    if (a.split_min)
    {
        // split path: units over (unique expert, chunk of 32 rows); only the heavy experts' rows are computed here
        const int u = jb.g / a.split_chunks, q = jb.g % a.split_chunks;
        if (u >= *a.nuniq) return;
        jb.e = a.uexp[u];
        const int c = a.counts[jb.e];
        if (MID_M * q >= c || !split_heavy(a, jb.e)) return;
        if (group_skipped(a, jb.e)) return;
        jb.r0 = a.offsets[jb.e] + MID_M * q;
        jb.nr = min(MID_M, c - MID_M * q);
    }
    else
    {
        if (jb.g >= *a.ngroups) return;
        jb.e = a.groups[3 * jb.g];
        if (group_skipped(a, jb.e)) return;
        jb.r0 = a.groups[3 * jb.g + 1];
        jb.nr = a.groups[3 * jb.g + 2];
    }
    jb.ex = jb.e == a.E ? a.shared : a.experts + jb.e;
    jb.K = DOWN ? a.I : a.H;
    jb.N = DOWN ? a.H : a.I;
    const int lane = threadIdx.x & 63, n = jb.K / 32 / KS, s0 = ksp * n;
    const uint16_t* asrc = DOWN ? a.act_rows : a.xt + (size_t)jb.mat * a.R_max * a.H;
    const uint16_t* ap = asrc + (size_t)(jb.r0 + min(lane & 31, jb.nr - 1)) * jb.K + 16 * (lane >> 5);
    const uint8_t* base = reinterpret_cast<const uint8_t*>(jb.ex->tr[jb.mat]);
    f32x16 acc[4] = {};
    switch (jb.ex->fmt[jb.mat])
    {
        case BMX_TF_K2: mid_run<BMX_TF_K2>(jb, base, ap, s0, n, acc); break;
        case BMX_TF_K25: mid_run<BMX_TF_K25>(jb, base, ap, s0, n, acc); break;
        case BMX_TF_K3: mid_run<BMX_TF_K3>(jb, base, ap, s0, n, acc); break;
        default: mid_run<BMX_TF_K4>(jb, base, ap, s0, n, acc); break;
    }
    // accumulator element v of lane L: row 8 (v / 4) + 4 (L / 32) + v % 4, column lane_col(L, c); row stride of the partial
    // layout in floats
    const int rs = DOWN ? a.NBH * 128 : a.NB * 256;
    const size_t r0 = (size_t)ksp * a.R_max + jb.r0 + 4 * (lane >> 5);
    float* out = (DOWN ? a.part_dn + jb.cb * 128 : a.part_gu + jb.cb * 256 + jb.mat * 128) + r0 * rs + lane_col(lane, 0);
#pragma unroll
    for (int v = 0; v < 16; ++v)
    {
        const int dr = 8 * (v >> 2) + (v & 3);
        if (dr + 4 * (lane >> 5) >= jb.nr) continue;
        *reinterpret_cast<float2*>(out + (size_t)dr * rs) = make_float2(acc[0][v], acc[1][v]);
        *reinterpret_cast<float2*>(out + (size_t)dr * rs + 8) = make_float2(acc[2][v], acc[3][v]);
    }
}

template <bool DOWN>
__global__ __launch_bounds__(MID_WAVES * 64, 3) void k_mid_gemm(GvArgs a)
{
    if (!a.split_min)
    {
        mid_unit<DOWN>(a, blockIdx.x);
        return;
    }
    // split path: a grid of at most MID_SPLIT_WGS workgroups loops over the units of the call's unique experts, so a call
    // that keeps every expert on the GEMV pays for few idle workgroups (none past the first check when no expert can
    // reach split_min rows)
    if (a.split_min > a.T + 1 && 2 * a.offsets[a.NE] < a.split_ratio2 * *a.nuniq) return;
    const int nb128 = DOWN ? a.NBH : a.NB;
    const int per = (DOWN ? 1 : 2) * ((nb128 + MID_WAVES - 1) / MID_WAVES) * (DOWN ? a.KS_dn : a.KS_gu);
    const int units = *a.nuniq * a.split_chunks * per;
    for (int lid = blockIdx.x; lid < units; lid += gridDim.x) mid_unit<DOWN>(a, lid);
}

// ---- plan and launch -------------------------------------------------------------------------------------------------
struct PrefillPlan {
    int NB, NBH, G_max, R_max;
    size_t xt_bytes, part_gu_bytes, act_bytes, part_dn_bytes;
};

static PrefillPlan prefill_plan(const MoeShape& m)
{
    PrefillPlan p;
    p.NB = m.I / 128;
    p.NBH = m.H / 128;
    p.G_max = groups_max(m.T, m.topk, m.E, m.shared, PF_M);
    p.R_max = m.T * m.topk + (m.shared ? m.T : 0);
    p.xt_bytes = (size_t)2 * p.R_max * m.H * 2;
    p.part_gu_bytes = (size_t)p.R_max * p.NB * 256 * 4;
    p.act_bytes = (size_t)p.R_max * m.I * 2;
    p.part_dn_bytes = (size_t)p.R_max * p.NBH * 128 * 4;
    return p;
}

int prefill_rows_per_group() { return PF_M; }

// BMX_PF_FAST_ACT=0: the prefill path's epilogue keeps the fixed-sequence activation of the decode path
static bool prefill_fast_act()
{
    const char* v = getenv("BMX_PF_FAST_ACT");
    return !(v && *v == '0');
}

// ---- mid-size path ------------------------------------------------------------------------------------------------------
struct MidPlan {
    int NB, NBH, G_max, R_max, KS_gu, KS_dn;
    size_t xt_bytes, part_gu_bytes, act_bytes, part_dn_bytes;
};

// k-split: the most splits that keep at least 16 k-steps of 64 each, gate / up and down (BMX_MID_MIN_STEPS,
// BMX_MID_MIN_STEPS_DN: that many instead, and none of the rules below). More splits even out the SIMDs' shares and fill a
// chip that the call's units leave idle, at the price of partial sums that the epilogues add. Two rules take them, down to
// 8 and 4 steps:
// - While a matrix's partials stay within MID_FEW_BYTES: the routing, unknown here, may put all rows on a few experts, and
//   partials of that size cost little where it does not. Measured (layer us, gate / up steps x down steps): 8 tokens (72
//   rows, ~60 experts of H 4096, I 1536) 8 x 4: 165, 16 x 4: 169, 8 x 16: 178, 32 x 16: 194; 16 tokens on ~12 experts (96
//   rows, I 2048) 8 x 4: 86, 4 x 4: 92, 16 x 4: 95, 16 x 16: 103. 64 experts of H 2048, I 768, 192 and 512 rows: picks
//   spread 88 -> 83 and 94 -> 92, tokens of one context 74 -> 54 and 82 -> 69. Past 12 MiB the spread calls pay: 18
//   tokens of the first layer 354 us within it, 362 at 16 MiB; 1,024 rows of the last 105, at 24 MiB 108.
// - Splits one after another while a matrix has fewer waves than the chip SIMDs (MID_FILL), counting one group per expert
//   the picks can reach or per 32 rows: layers of few experts. With 16 x 16 steps and now: 32 experts of H 1024, I 1024,
//   192 rows (256 waves a matrix) 79 -> 52 us; 8 of H 2048, I 1024, 192 rows (256 and 128 waves) 110 -> 85; 17 of H 1024,
//   I 512, 1,000 rows 77 -> 63; 8 of H 4096, I 2048, 256 rows (1,024 and 512) 151 -> 147. Past the line they cost more
//   than they give: 8 of H 4096, I 2048, 800 rows (3,200 and 1,600 waves) 196 at 16 x 16, 218 at 8 x 8; 64 of H 2048, I
//   768, 768 rows (1,536 and 1,024) 101 and 108.
// No split past the 16 steps' that would take the call past EXTRA_SPLITS_WS (gate / up first).
constexpr long MID_FEW_BYTES = 12 << 20;
constexpr long MID_FILL = 1024;
static int mid_split(int ksteps, bool down, long split_bytes, long waves, long budget)
{
    const char* v = getenv(down ? "BMX_MID_MIN_STEPS_DN" : "BMX_MID_MIN_STEPS");
    const bool forced = v && *v;
    const int min_steps = forced ? atoi(v) : 16, few_steps = down ? 4 : 8;
    int best = 1;
    for (int d = 2; d <= ksteps; ++d)
    {
        if (ksteps % d) continue;
        const long bytes = d * split_bytes;
        const bool few = !forced && ksteps / d >= few_steps && bytes <= budget &&
                         (bytes <= MID_FEW_BYTES || best * waves < MID_FILL);
        if (ksteps / d >= min_steps || few) best = d;
    }
    return best;
}

static MidPlan mid_plan(const MoeShape& m, bool extra = true)
{
    MidPlan p;
    p.NB = m.I / 128;
    p.NBH = m.H / 128;
    p.G_max = groups_max(m.T, m.topk, m.E, m.shared, MID_M);
    p.R_max = m.T * m.topk + (m.shared ? m.T : 0);
    p.xt_bytes = (size_t)2 * p.R_max * m.H * 2;
    p.act_bytes = (size_t)p.R_max * m.I * 2;
    const long gu = (long)p.R_max * p.NB * 256 * 4, dn = (long)p.R_max * p.NBH * 128 * 4;     // one split's partials
    const long groups = std::max<long>(std::min(m.E, m.T * m.topk) + (m.shared ? 1 : 0), p.R_max / MID_M);
    auto splits = [&](bool down, long budget) {
        return down ? mid_split(m.I / 64, true, dn, groups * p.NBH, budget)
                    : mid_split(m.H / 64, false, gu, 2 * groups * p.NB, budget);
    };
    const long room = extra ? (long)EXTRA_SPLITS_WS - (long)(p.xt_bytes + p.act_bytes) : 0;
    p.KS_gu = splits(false, room - splits(true, 0) * dn);
    p.KS_dn = splits(true, room - p.KS_gu * gu);
    p.part_gu_bytes = p.KS_gu * gu;
    p.part_dn_bytes = p.KS_dn * dn;
    return p;
}

int mid_rows_per_group() { return MID_M; }

// workgroups across a matrix's 128-column blocks
static int mid_blocks(int nb128) { return (nb128 + MID_WAVES - 1) / MID_WAVES; }

size_t mid_ws_bytes(const MoeShape& m)
{
    const MidPlan p = mid_plan(m);
    return align_up(p.xt_bytes, 256) + align_up(p.part_gu_bytes, 256) + align_up(p.act_bytes, 256) +
           align_up(p.part_dn_bytes, 256);
}

int launch_mid_experts(const MoeShape& m, const void* x, const bmx_routes* r, float* y_rows, void* act_rows, void* ws,
                       size_t ws_bytes, float* combine_out, const void* combine_w, hipStream_t s, int stages)
{
    if (m.H % 128 || m.I % 128 || m.H <= 0 || m.I <= 0)
        return set_error(BMX_ERR_ARG, "moe experts: H (%d) and I (%d) must be multiples of 128", m.H, m.I);
    if (ws_bytes < mid_ws_bytes(m))
        return set_error(BMX_ERR_WORKSPACE, "moe experts: workspace %zu < %zu", ws_bytes, mid_ws_bytes(m));
    if (!r->row_expert) return set_error(BMX_ERR_ARG, "moe experts: routes without row_expert");
    const MidPlan p = mid_plan(m);
    char* w = static_cast<char*>(ws);
    GvArgs a;
    a.experts = m.experts; a.shared = m.shared_ex; a.E = m.E; a.H = m.H; a.I = m.I; a.act = m.act; a.gated = m.gated;
    a.limit = m.limit;
    a.x = static_cast<const uint16_t*>(x);
    a.row_token = r->row_token; a.groups = r->groups; a.ngroups = r->ngroups; a.row_expert = r->row_expert;
    a.xt = reinterpret_cast<uint16_t*>(w);
    w += align_up(p.xt_bytes, 256);
    a.part_gu = reinterpret_cast<float*>(w);
    w += align_up(p.part_gu_bytes, 256);
    a.act_rows = act_rows ? static_cast<uint16_t*>(act_rows) : reinterpret_cast<uint16_t*>(w);
    w += align_up(p.act_bytes, 256);
    a.part_dn = reinterpret_cast<float*>(w);
    a.y_rows = y_rows;
    a.KS_gu = p.KS_gu; a.KS_dn = p.KS_dn; a.NB = p.NB; a.NBH = p.NBH; a.R_max = p.R_max;
    a.NE = m.E + (m.shared ? 1 : 0);
    a.out = combine_out; a.w = static_cast<const uint16_t*>(combine_w); a.inv = r->inv; a.offsets = r->offsets;
    a.T = m.T; a.topk = m.topk; a.has_shared = m.shared;
    a.fresh = m.fresh;
    a.sh_gate = m.shared_gate;
    a.filter = 0;
    a.act_in_down = 0;
    a.gu_half = 0;
    int rc = BMX_OK;
    if (stages & (1 << BMX_STAGE_PREP))
        hipLaunchKernelGGL(k_pf_prep, prep_grid(p.R_max, m.H), dim3(256), 0, s, a);
    for (int f = 0; f < 3; ++f)
    {
        const int st = f == 0 ? BMX_STAGE_GATE_UP : f == 1 ? BMX_STAGE_GATE_UP_RESIDENT : BMX_STAGE_GATE_UP_STAGED;
        if (!(stages & (1 << st))) continue;
        GvArgs b = a;
        b.filter = f;
        hipLaunchKernelGGL(k_mid_gemm<false>, dim3((unsigned)(p.G_max * 2 * mid_blocks(p.NB) * p.KS_gu)),
                           dim3(MID_WAVES * 64), 0, s, b);
    }
    if (stages & (1 << BMX_STAGE_ACT)) rc = launch_epilogue(a, BMX_STAGE_ACT, s);
    for (int f = 0; f < 3 && !rc; ++f)
    {
        const int st = f == 0 ? BMX_STAGE_DOWN : f == 1 ? BMX_STAGE_DOWN_RESIDENT : BMX_STAGE_DOWN_STAGED;
        if (!(stages & (1 << st))) continue;
        GvArgs b = a;
        b.filter = f;
        hipLaunchKernelGGL(k_mid_gemm<true>, dim3((unsigned)(p.G_max * mid_blocks(p.NBH) * p.KS_dn)),
                           dim3(MID_WAVES * 64), 0, s, b);
    }
    if (!rc && (stages & (1 << BMX_STAGE_COMBINE))) rc = launch_epilogue(a, BMX_STAGE_COMBINE, s);
    if (!rc && (stages & (1 << BMX_STAGE_DOWN_OUT))) rc = launch_epilogue(a, BMX_STAGE_DOWN_OUT, s);
    if (rc) return rc;
    return check_launch("moe experts (mid-size path)");
}

// ---- split path: the heavy experts' share ---------------------------------------------------------------------------
void split_mid_splits(const MoeShape& m, int* ks_gu, int* ks_dn, bool extra)
{
    const MidPlan p = mid_plan(m, extra);
    *ks_gu = p.KS_gu;
    *ks_dn = p.KS_dn;
}

// The prep of the heavy experts' rows and their mid-size GEMMs. a: the split path's arguments with KS_gu / KS_dn set to
// the mid-size splits (KS_gu_mid / KS_dn_mid); nu_max: the most unique experts a call can have.
constexpr long MID_SPLIT_WGS = 1024;

void launch_split_mid(const GvArgs& a, int stage, int nu_max, hipStream_t s)
{
    const long units = (long)nu_max * a.split_chunks;
    if (stage == BMX_STAGE_PREP)
        hipLaunchKernelGGL(k_pf_prep, prep_grid(a.R_max, a.H), dim3(256), 0, s, a);
    else if (stage == BMX_STAGE_DOWN || stage == BMX_STAGE_DOWN_RESIDENT || stage == BMX_STAGE_DOWN_STAGED)
        hipLaunchKernelGGL(k_mid_gemm<true>, dim3((unsigned)std::min(MID_SPLIT_WGS, units * mid_blocks(a.NBH) * a.KS_dn)),
                           dim3(MID_WAVES * 64), 0, s, a);
    else
        hipLaunchKernelGGL(k_mid_gemm<false>,
                           dim3((unsigned)std::min(MID_SPLIT_WGS, units * 2 * mid_blocks(a.NB) * a.KS_gu)),
                           dim3(MID_WAVES * 64), 0, s, a);
}

size_t prefill_ws_bytes(const MoeShape& m)
{
    const PrefillPlan p = prefill_plan(m);
    return align_up(p.xt_bytes, 256) + align_up(p.part_gu_bytes, 256) + align_up(p.act_bytes, 256) +
           align_up(p.part_dn_bytes, 256);
}

int launch_prefill_experts(const MoeShape& m, const void* x, const bmx_routes* r, float* y_rows, void* act_rows,
                           void* ws, size_t ws_bytes, float* combine_out, const void* combine_w, hipStream_t s,
                           int stages)
{
    if (m.H % 128 || m.I % 128 || m.H <= 0 || m.I <= 0)
        return set_error(BMX_ERR_ARG, "moe experts: H (%d) and I (%d) must be multiples of 128", m.H, m.I);
    if (ws_bytes < prefill_ws_bytes(m))
        return set_error(BMX_ERR_WORKSPACE, "moe experts: workspace %zu < %zu", ws_bytes, prefill_ws_bytes(m));
    if (!r->row_expert) return set_error(BMX_ERR_ARG, "moe experts: routes without row_expert");
    const PrefillPlan p = prefill_plan(m);
    char* w = static_cast<char*>(ws);
    GvArgs a;
    a.experts = m.experts; a.shared = m.shared_ex; a.E = m.E; a.H = m.H; a.I = m.I; a.act = m.act; a.gated = m.gated;
    a.limit = m.limit;
    a.x = static_cast<const uint16_t*>(x);
    a.row_token = r->row_token; a.groups = r->groups; a.ngroups = r->ngroups; a.row_expert = r->row_expert;
    a.xt = reinterpret_cast<uint16_t*>(w);
    w += align_up(p.xt_bytes, 256);
    a.part_gu = reinterpret_cast<float*>(w);
    w += align_up(p.part_gu_bytes, 256);
    a.act_rows = act_rows ? static_cast<uint16_t*>(act_rows) : reinterpret_cast<uint16_t*>(w);
    w += align_up(p.act_bytes, 256);
    a.part_dn = reinterpret_cast<float*>(w);
    a.y_rows = y_rows;
    a.KS_gu = 1; a.KS_dn = 1; a.NB = p.NB; a.NBH = p.NBH; a.R_max = p.R_max;
    a.NE = m.E + (m.shared ? 1 : 0);
    a.out = combine_out; a.w = static_cast<const uint16_t*>(combine_w); a.inv = r->inv; a.offsets = r->offsets;
    a.T = m.T; a.topk = m.topk; a.has_shared = m.shared;
    a.fresh = m.fresh;
    a.sh_gate = m.shared_gate;
    a.filter = 0;
    a.act_in_down = 0;
    a.gu_half = 1;
    a.fast_act = prefill_fast_act() ? 1 : 0;
    int rc = BMX_OK;
    if (stages & (1 << BMX_STAGE_PREP))
        hipLaunchKernelGGL(k_pf_prep_tok, prep_tok_grid(m.T, m.H), dim3(256), 0, s, a);
    for (int f = 0; f < 3; ++f)
    {
        const int st = f == 0 ? BMX_STAGE_GATE_UP : f == 1 ? BMX_STAGE_GATE_UP_RESIDENT : BMX_STAGE_GATE_UP_STAGED;
        if (!(stages & (1 << st))) continue;
        GvArgs b = a;
        b.filter = f;
        hipLaunchKernelGGL(k_pf_gemm<false>, dim3((unsigned)(p.G_max * 2 * ((p.NB + 1) / 2))), dim3(PF_WAVES * 64), 0, s, b);
    }
    if (stages & (1 << BMX_STAGE_ACT)) rc = launch_epilogue(a, BMX_STAGE_ACT, s);
    for (int f = 0; f < 3 && !rc; ++f)
    {
        const int st = f == 0 ? BMX_STAGE_DOWN : f == 1 ? BMX_STAGE_DOWN_RESIDENT : BMX_STAGE_DOWN_STAGED;
        if (!(stages & (1 << st))) continue;
        GvArgs b = a;
        b.filter = f;
        hipLaunchKernelGGL(k_pf_gemm<true>, dim3((unsigned)(p.G_max * ((p.NBH + 1) / 2))), dim3(PF_WAVES * 64), 0, s, b);
    }
    if (!rc && (stages & (1 << BMX_STAGE_COMBINE))) rc = launch_epilogue(a, BMX_STAGE_COMBINE, s);
    if (!rc && (stages & (1 << BMX_STAGE_DOWN_OUT))) rc = launch_epilogue(a, BMX_STAGE_DOWN_OUT, s);
    if (rc) return rc;
    return check_launch("moe experts (prefill path)");
}

}  // namespace bmx
