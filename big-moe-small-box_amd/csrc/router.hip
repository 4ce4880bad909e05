// Router and decode-size route + dispatch.
//
// One wavefront per token. Lane l holds experts l, l + 64, ...; the strict total order is larger choice, then lower
// index (a 64-bit key: order-preserving value bits over the complement of the index). The group limit takes each
// group's top-2 by wave-wide DPP maxima of the keys, then the groups by their top-2 sums; the top-k itself is a
// bitwise search for the k-th largest value by wave ballots followed by a rank of the k picks. The order is the one
// the oracle's sequential selection produces, independent of scheduling.
#include "bmx_common.hpp"
#include "bmx_internal.hpp"
#include "router_wave.hpp"

#include <algorithm>

namespace bmx {

// four tokens per workgroup, so that a chunk's waves spread over every CU (2,048 tokens: 16 per workgroup leave half of them
// without one; 10.0 -> 8.9 us)
constexpr int RK_WAVES = 4;
template <int J>
__global__ __launch_bounds__(RK_WAVES * 64) void k_router(RouterArgs a)
{
    __shared__ TopkLds tl[RK_WAVES];
    const int t = blockIdx.x * RK_WAVES + (threadIdx.x >> 6);
    if (t < a.T) route_token_wave<J>(a, t, tl[threadIdx.x >> 6]);
}

// ---- fused decode kernel: route every token, then the counting sort of its picks, in one workgroup ------------------
template <int J>
__global__ __launch_bounds__(RT_THREADS) void k_route_dispatch_small(RouterArgs a, SmallDispatch d)
{
    __shared__ int pe[SM_MAXN];          // local expert of each pick (-1: dropped)
    __shared__ int cnt[RT_MAXE + 1];
    __shared__ TopkLds tl[RT_WAVES];
    const int E = a.E, n = a.T * a.topk, tid = threadIdx.x, lane = tid & 63;
    for (int t = tid >> 6; t < a.T; t += RT_WAVES)
    {
        const int pk = route_token_wave<J>(a, t, tl[tid >> 6]);
        if (lane < a.topk) pe[t * a.topk + lane] = pk;
    }
    if (a.T <= 64)
    {
        __shared__ int soff[RT_MAXE + 1];
        __shared__ uint64_t smask[RT_MAXE + 1];
        if (a.T > 1) lds_barrier();          // one token: wave 0 routed it and reads its own LDS writes in order
        if (tid < 64) dispatch_wave<J + 1>(pe, n, E, a.T, a.topk, d, cnt, soff, smask);
        return;
    }
    lds_barrier();
    const int NE = E + (d.shared ? 1 : 0);
    __shared__ int4 pe4[SM_MAXN / 4];        // the picks again, padded with -1 to a multiple of 4
    __shared__ int4 gc4[SM_MAXN / 4];        // per pick: groups of its expert if it is the expert's first pick, else 0
    const int n4 = (n + 3) >> 2;
    int* pev = reinterpret_cast<int*>(pe4);
    int* gcv = reinterpret_cast<int*>(gc4);
    for (int p = tid; p < 4 * n4; p += blockDim.x) pev[p] = p < n ? pe[p] : -1;
    lds_barrier();
    // counts and offsets per expert (the shared segment last)
    int nvalid = 0;
    for (int q = 0; q < n4; ++q)
    {
        const int4 v = pe4[q];
        nvalid += (v.x >= 0) + (v.y >= 0) + (v.z >= 0) + (v.w >= 0);
    }
    for (int e = tid; e < NE; e += blockDim.x)
    {
        int c = 0, below = 0;
        if (e < E)
            for (int q = 0; q < n4; ++q)
            {
                const int4 v = pe4[q];
                c += (v.x == e) + (v.y == e) + (v.z == e) + (v.w == e);
                below += (v.x >= 0 && v.x < e) + (v.y >= 0 && v.y < e) + (v.z >= 0 && v.z < e) + (v.w >= 0 && v.w < e);
            }
        else { c = a.T; below = nvalid; }
        cnt[e] = c;
        d.r.counts[e] = c;
        d.r.offsets[e] = below;
        if (e == NE - 1) d.r.offsets[NE] = below + c;
    }
    lds_barrier();
    for (int p = tid; p < 4 * n4; p += blockDim.x)
    {
        const int e = pev[p];
        int first = e >= 0;
        for (int q = 0; q < p && first; ++q) first = pev[q] != e;
        gcv[p] = first ? (cnt[e] + d.rpg - 1) / d.rpg : 0;
    }
    lds_barrier();
    int nu_r = 0, ng_r = 0;
    for (int q = 0; q < n4; ++q)
    {
        const int4 g = gc4[q];
        nu_r += (g.x > 0) + (g.y > 0) + (g.z > 0) + (g.w > 0);
        ng_r += g.x + g.y + g.z + g.w;
    }
    // rows: stable by (expert, pick); the expert's first pick also places its groups and its uexp entry
    for (int p = tid; p < n; p += blockDim.x)
    {
        const int e = pev[p];
        if (e < 0) { d.r.inv[p] = -1; continue; }
        int row = 0, ui = 0, g0 = 0;
        for (int q4 = 0; q4 < n4; ++q4)
        {
            const int4 v = pe4[q4], g = gc4[q4];
            const int q = 4 * q4;
            row += (v.x >= 0 && (v.x < e || (v.x == e && q < p))) + (v.y >= 0 && (v.y < e || (v.y == e && q + 1 < p))) +
                   (v.z >= 0 && (v.z < e || (v.z == e && q + 2 < p))) + (v.w >= 0 && (v.w < e || (v.w == e && q + 3 < p)));
            ui += (g.x > 0 && v.x < e) + (g.y > 0 && v.y < e) + (g.z > 0 && v.z < e) + (g.w > 0 && v.w < e);
            g0 += (v.x < e ? g.x : 0) + (v.y < e ? g.y : 0) + (v.z < e ? g.z : 0) + (v.w < e ? g.w : 0);
        }
        d.r.inv[p] = row;
        d.r.row_token[row] = p / a.topk;
        d.r.row_slot[row] = p % a.topk;
        d.r.row_expert[row] = e;
        const int ng = gcv[p];
        if (ng > 0)
        {
            const int c = cnt[e];
            d.r.uexp[ui] = e;
            for (int q = 0; q < ng; ++q)
            {
                d.r.groups[3 * (g0 + q) + 0] = e;
                d.r.groups[3 * (g0 + q) + 1] = row + q * d.rpg;
                d.r.groups[3 * (g0 + q) + 2] = min(d.rpg, c - q * d.rpg);
            }
        }
    }
    if (d.shared)
    {
        for (int t = tid; t < a.T; t += blockDim.x)
        {
            d.r.row_token[nvalid + t] = t;
            d.r.row_slot[nvalid + t] = -1;
            d.r.row_expert[nvalid + t] = E;
        }
        for (int q = tid; q * d.rpg < a.T; q += blockDim.x)
        {
            d.r.groups[3 * (ng_r + q) + 0] = E;
            d.r.groups[3 * (ng_r + q) + 1] = nvalid + q * d.rpg;
            d.r.groups[3 * (ng_r + q) + 2] = min(d.rpg, a.T - q * d.rpg);
        }
        if (tid == 0) d.r.uexp[nu_r] = E;
    }
    if (tid == 0)
    {
        *d.r.nuniq = nu_r + (d.shared ? 1 : 0);
        *d.r.ngroups = ng_r + (d.shared ? (a.T + d.rpg - 1) / d.rpg : 0);
    }
}

int check_router(int T, int E, int topk, int n_group, int topk_group, int score_fn, const void* logits,
                        const void* sel, const void* w)
{
    if (T < 0 || E <= 0 || E > RT_MAXE || topk <= 0 || topk > RT_MAXK || topk > E)
        return set_error(BMX_ERR_ARG, "bmx_router_topk: unsupported sizes T=%d E=%d topk=%d", T, E, topk);
    if (n_group < 1 || n_group > RT_MAXG || E % n_group || topk_group < 1 || topk_group > n_group)
        return set_error(BMX_ERR_ARG, "bmx_router_topk: bad groups n_group=%d topk_group=%d (E=%d)", n_group, topk_group, E);
    if (n_group > 1 && topk > topk_group * (E / n_group))
        return set_error(BMX_ERR_ARG, "bmx_router_topk: topk %d exceeds the experts of %d groups", topk, topk_group);
    if (score_fn != BMX_SCORE_SOFTMAX && score_fn != BMX_SCORE_SIGMOID && score_fn != BMX_SCORE_SQRTSP)
        return set_error(BMX_ERR_ARG, "bmx_router_topk: unknown score function %d", score_fn);
    if (T > 0 && (!logits || !sel || !w)) return set_error(BMX_ERR_ARG, "bmx_router_topk: null pointer");
    return BMX_OK;
}

static RouterArgs router_args(const void* logits, const float* bias, int T, int E, int topk, int n_group,
                              int topk_group, int score_fn, int renorm, float scale, int64_t first, int64_t* sel, void* w)
{
    RouterArgs a;
    a.logits = static_cast<const uint16_t*>(logits); a.bias = bias; a.T = T; a.E = E; a.topk = topk; a.G = n_group;
    a.TG = topk_group; a.score_fn = score_fn; a.renorm = renorm; a.scale = scale; a.first = first; a.sel = sel;
    a.w = static_cast<uint16_t*>(w);
    return a;
}


int launch_router(const void* logits, const float* bias, int T, int E, int topk, int n_group, int topk_group,
                  int score_fn, int renorm, float scale, int64_t first, int64_t* sel, void* w, hipStream_t s)
{
    int rc = check_router(T, E, topk, n_group, topk_group, score_fn, logits, sel, w);
    if (rc || T == 0) return rc;
    const RouterArgs a = router_args(logits, bias, T, E, topk, n_group, topk_group, score_fn, renorm, scale, first, sel, w);
    const dim3 grid((unsigned)((T + RK_WAVES - 1) / RK_WAVES)), block(RK_WAVES * 64);
    const int J = (E + 63) / 64;
    switch (J)
    {
        case 1: hipLaunchKernelGGL(k_router<1>, grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL(k_router<2>, grid, block, 0, s, a); break;
        case 3: hipLaunchKernelGGL(k_router<3>, grid, block, 0, s, a); break;
        case 4: hipLaunchKernelGGL(k_router<4>, grid, block, 0, s, a); break;
        case 5: hipLaunchKernelGGL(k_router<5>, grid, block, 0, s, a); break;
        case 6: hipLaunchKernelGGL(k_router<6>, grid, block, 0, s, a); break;
        case 7: case 8: hipLaunchKernelGGL(k_router<8>, grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL(k_router<16>, grid, block, 0, s, a); break;
    }
    return check_launch("bmx_router_topk");
}

bool route_dispatch_small_fits(int T, int E, int topk) { return (long)T * topk <= SM_MAXN && E <= RT_MAXE; }

int launch_route_dispatch_small(const void* logits, const float* bias, int T, int E, int topk, int n_group,
                                int topk_group, int score_fn, int renorm, float scale, int64_t first, int64_t* sel,
                                void* w, int shared, int rpg, const bmx_routes* routes, hipStream_t s)
{
    int rc = check_router(T, E, topk, n_group, topk_group, score_fn, logits, sel, w);
    if (rc || T == 0) return rc;
    if (!route_dispatch_small_fits(T, E, topk)) return set_error(BMX_ERR_ARG, "route+dispatch: too many picks (%d)", T * topk);
    const RouterArgs a = router_args(logits, bias, T, E, topk, n_group, topk_group, score_fn, renorm, scale, first, sel, w);
    SmallDispatch d;
    d.shared = shared ? 1 : 0;
    d.rpg = rpg;
    d.r = *routes;
    const int J = (E + 63) / 64;
    const dim3 grid(1), block(RT_THREADS);
    switch (J)
    {
        case 1: hipLaunchKernelGGL(k_route_dispatch_small<1>, grid, block, 0, s, a, d); break;
        case 2: hipLaunchKernelGGL(k_route_dispatch_small<2>, grid, block, 0, s, a, d); break;
        case 3: hipLaunchKernelGGL(k_route_dispatch_small<3>, grid, block, 0, s, a, d); break;
        case 4: hipLaunchKernelGGL(k_route_dispatch_small<4>, grid, block, 0, s, a, d); break;
        case 5: hipLaunchKernelGGL(k_route_dispatch_small<5>, grid, block, 0, s, a, d); break;
        case 6: hipLaunchKernelGGL(k_route_dispatch_small<6>, grid, block, 0, s, a, d); break;
        case 7: case 8: hipLaunchKernelGGL(k_route_dispatch_small<8>, grid, block, 0, s, a, d); break;
        default: hipLaunchKernelGGL(k_route_dispatch_small<16>, grid, block, 0, s, a, d); break;
    }
    return check_launch("route + dispatch");
}

// The arguments of launch_route_dispatch_small for a one-token gate / up GEMV that routes and dispatches the token itself
int route_fuse_args(const void* logits, const float* bias, int T, int E, int topk, int n_group, int topk_group,
                    int score_fn, int renorm, float scale, int64_t first, int64_t* sel, void* w, int shared, int rpg,
                    const bmx_routes* routes, RouteFuse* out)
{
    int rc = check_router(T, E, topk, n_group, topk_group, score_fn, logits, sel, w);
    if (rc) return rc;
    if (T != 1 || !route_dispatch_small_fits(T, E, topk))
        return set_error(BMX_ERR_ARG, "route in GEMV: one token and at most %d experts", RT_MAXE);
    out->ra = router_args(logits, bias, T, E, topk, n_group, topk_group, score_fn, renorm, scale, first, sel, w);
    out->sd.shared = shared ? 1 : 0;
    out->sd.rpg = rpg;
    out->sd.r = *routes;
    out->J = (E + 63) / 64;
    return BMX_OK;
}

// ---- router projection: logits = z W^T on the MFMA units ----------------------------------------------------------------
// logits[t][e] = RN16(sum_h z[t][h] W[e][h]): z fp16 [T][H] (the MoE input rows), W fp16 [E][H] (the router's gate weight
// as checkpoints store it), fp32 accumulation. A logit is eight sums: each quarter of H in k-steps of 16, the even and the
// odd steps of a quarter apart; then even + odd per quarter, and the quarters in order. Both kernels below add in exactly
// this order (a step is one MFMA with lane L's operand the k values 8 (L / 32) .. + 7 of row L % 32), so a token's logits
// do not depend on how many tokens share its call. Their eight waves are the eight sums.
constexpr int RL_WAVES = 8;

// A wave's accumulators in LDS, element v of block b at red[wave][b][v][lane] (row 8 (v / 4) + 4 (lane / 32) + v % 4 of
// the block's 32 tokens, column lane % 32 of its 32 experts); the eight sums added in the order above and stored by all
// threads. NE: the tile's 32-expert blocks, EB: the experts of a block in use.
template <int NB, int NE, int EB>
__device__ __forceinline__ void rl_finish(const f32x16 (&acc)[NB], float* red, int t0, int e0, int T, int E,
                                          uint16_t* __restrict__ out)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) red[((wave * NB + b) * 16 + v) * 64 + lane] = acc[b][v];
    lds_barrier();
    for (int i = threadIdx.x; i < NB * 1024; i += RL_WAVES * 64)
    {
        const int L = i & 63, v = (i >> 6) & 15, b = i >> 10;
        float q[RL_WAVES / 2];
#pragma unroll
        for (int w = 0; w < RL_WAVES; w += 2) q[w / 2] = red[w * NB * 1024 + i] + red[(w + 1) * NB * 1024 + i];
        const float r = ((q[0] + q[1]) + q[2]) + q[3];
        const int tt = t0 + 32 * (b / NE) + 8 * (v >> 2) + 4 * (L >> 5) + (v & 3), e = e0 + 32 * (b % NE) + (L & 31);
        if (tt < T && e < E && (L & 31) < EB) out[(size_t)tt * E + e] = f2h_r(r);
    }
}

// Decode steps, a few tokens: eight experts a workgroup (the MFMA's other columns are copies that nobody stores: the matrix
// unit is idle anyway, and small tiles spread the weight's read over the CUs). Wave w copies expert row w to LDS, all of it
// requested at once up to H = 5120, the tokens' rows follow, and the chains run out of LDS: one trip to memory, in whole
// cache lines, and little code (cold instructions cost as much as cold data here: the same with operands in registers and
// the 40 steps unrolled took 13.5 us). Rows are padded by 16 bytes against bank conflicts. The rows have to fit
// RL_FEW_LDS. 1 token, 384 experts, H 5120: 16.5 -> 6.2 us.
constexpr int RL_FEW_EB = RL_WAVES, RL_FEW_U = 10;
constexpr size_t RL_FEW_LDS = 128 * 1024;
static size_t rl_few_lds(int T, int H) { return (size_t)(RL_FEW_EB + T) * (H * 2 + 16); }
__global__ __launch_bounds__(RL_WAVES * 64, 2) void k_router_logits_few(const uint16_t* __restrict__ z,
                                                                        const uint16_t* __restrict__ W, int T, int H, int E,
                                                                        uint16_t* __restrict__ out)
{
    extern __shared__ u32x4 rows[];                    // [experts, then tokens][H / 8 + 1]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int e0 = blockIdx.x * RL_FEW_EB, P = H / 8;
    for (int r = wave; r < RL_FEW_EB + T; r += RL_WAVES)
    {
        const uint16_t* src = r < RL_FEW_EB ? W + (size_t)min(e0 + r, E - 1) * H : z + (size_t)(r - RL_FEW_EB) * H;
        for (int i0 = lane; i0 < P; i0 += 64 * RL_FEW_U)
        {
            u32x4 f[RL_FEW_U];
#pragma unroll
            for (int u = 0; u < RL_FEW_U; ++u) f[u] = ldg4(src + 8 * min(i0 + 64 * u, P - 1));
#pragma unroll
            for (int u = 0; u < RL_FEW_U; ++u)
                if (i0 + 64 * u < P) rows[r * (P + 1) + i0 + 64 * u] = f[u];
        }
    }
    lds_barrier();
    const int kq = H / 4, n = (kq / 16 + 1 - (wave & 1)) / 2;            // the wave's steps
    const u32x4* p = rows + ((wave >> 1) * kq + 16 * (wave & 1)) / 8 + (lane >> 5);
    const u32x4* pa = p + (RL_FEW_EB + min(lane & 31, T - 1)) * (P + 1);
    const u32x4* pb = p + (lane & (RL_FEW_EB - 1)) * (P + 1);
    f32x16 acc[1] = {};
    for (int s = 0; s < n; ++s)
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, pa[4 * s]), __builtin_bit_cast(f16x8, pb[4 * s]),
                                                        acc[0], 0, 0, 0);
    lds_barrier();                                     // the rows are read: their place takes the sums
    rl_finish<1, 1, RL_FEW_EB>(acc, reinterpret_cast<float*>(rows), 0, e0, T, E, out);
}

// Batches and chunks: 32 NT tokens x ER experts a workgroup. A stage is 64 k of every quarter of the tile's rows, read
// 128 bytes of a row per eight lanes and shared through LDS (16-byte chunk c of row r at c ^ (r % 8): eight rows' chunks
// of one step spread over all banks); the loads run D stages ahead in registers, about 128 KB per workgroup. Operands
// straight from memory in 32 x 32 tiles, as this kernel once did, touch 32 cache lines per load for a quarter of each
// and read twice as much. It is bound by the tiles' reads:
// 2,048 tokens, 384 experts, H 4096: 53.2 -> 20.6 us; 77 tokens, 288 experts: 19.8 -> 10.6. Larger tiles read less but
// leave more CUs idle; the lines are where the next size starts its second round on the 256 CUs (us at H 4096):
//   64 x 64 from 96 tiles: 96 of them (384 experts) 17.6, 32 x 32 17.3; 144: 18.7 and 24.9; 70 (288 experts): 17.3 and 14.2.
//   32 x 32 from 128 tiles: 144 of them 9.6, 32 x 16 12.8; 120: 9.5 and 9.6; 108 (288 experts): 10.9 and 9.5.
//   Up to 32 experts 32 x 32 always: a wider tile reads no less of z and its other columns are copies (8,192 tokens, 8
//   experts: 13.4, 64 x 64 17.7).
// Workgroups go to the 8 XCDs round-robin: with large tiles (at least 96 of them) the blocks of a token tile are renumbered
// onto one XCD, whose L2 then reads the tokens once (W, the smaller matrix, is read by all).
template <int NT, int ER, int D>
__global__ __launch_bounds__(RL_WAVES * 64, 2) void k_router_logits(const uint16_t* __restrict__ z,
                                                                    const uint16_t* __restrict__ W, int T, int H, int E,
                                                                    uint16_t* __restrict__ out)
{
    constexpr int TR = 32 * NT, R = TR + ER, NL = R / 16, NE = (ER + 31) / 32, NB = NT * NE;
    constexpr int ST = 4 * R * 8;                                       // a stage, in chunks: [quarter][row][chunk]
    constexpr int RED = RL_WAVES * NB * 1024 / 4;
    static_assert(D % 2 == 0, "stage s is in LDS half s % 2");
    __shared__ u32x4 lds[2 * ST > RED ? 2 * ST : RED];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5;
    const int neb = (E + ER - 1) / ER, xi = NT > 1 ? blockIdx.x >> 3 : blockIdx.x;
    const int t0 = (NT > 1 ? (blockIdx.x & 7) + 8 * (xi / neb) : xi / neb) * TR, e0 = xi % neb * ER;
    if (t0 >= T) return;
    const int kq = H / 4, ns = (kq + 63) / 64;
    // the thread's chunk of the NL pieces of a stage; rows past the last token or expert read the last one
    const int c = threadIdx.x & 7;
    const uint16_t* src[NL];
    int dst[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i)
    {
        const int rest = i * (RL_WAVES * 8) + (threadIdx.x >> 3), r = rest % R, q = rest / R;
        src[i] = (r < TR ? z + (size_t)min(t0 + r, T - 1) * H : W + (size_t)min(e0 + r - TR, E - 1) * H) + q * kq + 8 * c;
        dst[i] = rest * 8 + (c ^ (r & 7));
    }
    const u32x4 zero = {0u, 0u, 0u, 0u};
    u32x4 st[D][NL];
    auto fetch = [&](u32x4 (&f)[NL], int s) {
        const bool in = 64 * s + 8 * c < kq;            // past a quarter's end: operands of zeros, which add nothing
#pragma unroll
        for (int i = 0; i < NL; ++i) f[i] = in ? ldg4(src[i] + 64 * s) : zero;
    };
    auto store = [&](const u32x4 (&f)[NL], int g) {
#pragma unroll
        for (int i = 0; i < NL; ++i) lds[g * ST + dst[i]] = f[i];
    };
    f32x16 acc[NB] = {};
    const int q = wave >> 1, par = wave & 1;
    auto mul = [&](int g) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            const int ch = 2 * (2 * j + par) + h;
            auto at = [&](int r) { return __builtin_bit_cast(f16x8, lds[g * ST + (q * R + r) * 8 + (ch ^ (r & 7))]); };
            f16x8 a[NT], b[NE];
#pragma unroll
            for (int i = 0; i < NT; ++i) a[i] = at(32 * i + (lane & 31));
#pragma unroll
            for (int i = 0; i < NE; ++i) b[i] = at(TR + 32 * i + (lane & (ER < 32 ? ER - 1 : 31)));
#pragma unroll
            for (int i = 0; i < NB; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i / NE], b[i % NE], acc[i], 0, 0, 0);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(st[d], d);
    store(st[0], 0);
    fetch(st[0], D);
    lds_barrier();
    for (int s = 0; s < ns; s += D)
#pragma unroll
        for (int d = 0; d < D; ++d)
        {
            if (s + d >= ns) break;
            mul(d & 1);
            store(st[(d + 1) % D], (d + 1) & 1);
            fetch(st[(d + 1) % D], s + d + 1 + D);
            lds_barrier();
        }
    rl_finish<NB, NE, (ER < 32 ? ER : 32)>(acc, reinterpret_cast<float*>(lds), t0, e0, T, E, out);
}

int launch_router_logits(const void* z, const void* W, int T, int H, int E, void* logits, hipStream_t s)
{
    if (T < 0 || E <= 0 || H <= 0 || H % 64)
        return set_error(BMX_ERR_ARG, "bmx_router_logits: T (%d) >= 0, E (%d) > 0 and H (%d) a multiple of 64 required",
                         T, E, H);
    if (T == 0) return BMX_OK;
    if (!z || !W || !logits) return set_error(BMX_ERR_ARG, "bmx_router_logits: null pointer");
    if ((reinterpret_cast<uintptr_t>(z) | reinterpret_cast<uintptr_t>(W)) % 16)
        return set_error(BMX_ERR_ARG, "bmx_router_logits: z and the weight must be 16-byte aligned");
    auto tiles = [&](int tb, int eb) { return (long)((T + tb - 1) / tb) * ((E + eb - 1) / eb); };
    if (tiles(32, 32) > 0x7fffffffL) return set_error(BMX_ERR_ARG, "bmx_router_logits: too many tiles");
    const uint16_t* zp = static_cast<const uint16_t*>(z);
    const uint16_t* wp = static_cast<const uint16_t*>(W);
    uint16_t* lp = static_cast<uint16_t*>(logits);
    const dim3 block(RL_WAVES * 64);
    const size_t few = rl_few_lds(T, H);
    if (T <= 32 && few <= RL_FEW_LDS)
        hipLaunchKernelGGL(k_router_logits_few, dim3((unsigned)((E + RL_FEW_EB - 1) / RL_FEW_EB)), block,
                           std::max(few, (size_t)RL_WAVES * 4096), s, zp, wp, T, H, E, lp);
    else if (E > 32 && tiles(64, 64) >= 96)
        hipLaunchKernelGGL((k_router_logits<2, 64, 2>), dim3((unsigned)(8 * tiles(512, 64))), block, 0, s, zp, wp, T, H, E, lp);
    else if (tiles(32, 32) >= 128)
        hipLaunchKernelGGL((k_router_logits<1, 32, 4>), dim3((unsigned)tiles(32, 32)), block, 0, s, zp, wp, T, H, E, lp);
    else
        hipLaunchKernelGGL((k_router_logits<1, 16, 6>), dim3((unsigned)tiles(32, 16)), block, 0, s, zp, wp, T, H, E, lp);
    return check_launch("bmx_router_logits");
}

}  // namespace bmx
