// Fat-expert path (prefill): per-expert grouped GEMM with the EXL3 weights decoded into LDS and multiplied on
// MFMA, for experts that receive many routes (the reference's apply_exl3_batched_fat / run_batch,
// patches/vllm-exl3-host-dma.patch:182-201, runtime/dma_gemm.py:5-26, which reconstruct fp16 weights and run a
// 128x128 GEMM).
//
// Launches: mm_permute (sorted positions) -> k_fat_plan (expert records, row groups, tile lists) -> k_fat_prep
// (transformed inputs per row group) -> k_fat, k_fat16<0, 2>, k_mid<0> (gate/up) -> k_fat16<1, 4>, k_fat16<1, 2>, k_mid<1>
// (down) -> k_fat_combine; a tile size that the call cannot have is not launched.
//
// An expert's routes (sorted positions) are taken in row groups of 32, whose inputs are stored in MFMA operand order: per
// matrix and 32-element step one contiguous 2 KB, chunk g (8 elements: tile rows 0 and 1 of decode window g) of row r at
// 16 (32 g + r). A wave's operand load is then one contiguous KB, whichever kernel reads it.
//
// k_mid takes tiles of at most 96 routes (below). k_fat (8 waves, two per SIMD) and k_fat16 (16 waves) own a tile of 256
// (k_fat16 also 128) routes of one expert x 256 output columns, for calls with many of them:
//   gate/up (MODE 0): gate columns 128 c .. 128 c + 127 and the same up columns, so the epilogue holds both and
//                     applies the output transforms, SwiGLU and the down-input transform of that 128-block (the
//                     transforms act within 128-blocks);
//   down    (MODE 1): two 128-blocks of H; the epilogue applies the output transform and writes per-route rows.
// Per 32-row step (two tile rows) the inputs (buffer-to-LDS, FT_PA - 1 steps ahead) and the 32 trellis tiles of
// the columns (768-byte rows, buffer-to-LDS, FT_PT steps ahead) are staged in LDS by loader waves; every wave
// decodes 4 tiles of the next step into the MFMA B layout (fp16 weights, rounded as the reconstruct does) in
// between its v_mfma_f32_16x16x32_f16 over a (BM / 2) x 64 sub-tile (128 accumulators per lane), so one wave's
// decode runs while the other wave of its SIMD multiplies. The weights are decoded once per tile.
#include <algorithm>
#include <type_traits>

#include "mm_decode.h"

namespace mm {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int FT_BIG = 256;         // routes per tile (8 row blocks per row-wave)
constexpr int FT_MID = 96;          // routes per tile of k_mid
constexpr int FT_SMALL = 128;       // routes per tile of k_fat16<*, 2>

// Which tiles an expert's routes take. Tiles of 256 routes (and of 128, where the weights are rounded) cost the least per route
// once there are several rounds of workgroups of them (one fits a CU), FT_MID-route tiles leave fewer CUs idle before that and
// fewer rows empty. The kernels of the tile sizes add an expert's products in different orders, except those of 256 and 128.
//   a fused call: 256-route tiles where it has at least three rounds (FT_BIG_WORK workgroups) of them, the rest in FT_MID-route
//     tiles. 3 tiles (48 workgroups) of a 512-token call took 214 us of its 1,540 where FT_MID-route tiles took 60; at 64 tiles
//     (4,096 tokens) both GEMMs take 2.68 ms with them and 2.84 without, at 297 (16,384 tokens) 8.25 and 8.65.
//   the other entry points, whose rows must have the same bits whichever experts of a layer a call computes (a layer in one
//     call or in staging batches): by the expert's routes and the layer's. From 768 routes on 256-route tiles: a staging batch
//     of 16 experts holds few (12 took 189 us of its 470, as FT_MID-route tiles 50). In layers of at least FT_LARGE routes and
//     200 per expert, from a remainder of 129 routes on, and remainders of 97 to 128 routes in 128-route tiles (two FT_MID-route
//     tiles otherwise: 0.55 against 0.34 us per expert and column unit at H 5120); the shorter ones too where the layer has
//     under one and a half rounds of them (a launch of a few k_mid workgroups takes 99 + 50 us). mm_moe_prefill of 16,384
//     tokens by the first / by this rule, ms: H 5120 10.91 / 10.4 (64 hot experts), 10.94 / 10.05 (even routing), H 4096
//     10.50 / 9.60 (even); 16 staged experts 0.84 / 0.73. At 8,192 tokens staged experts take 0.48 ms by the first rule and
//     0.55 by this, the whole layer 5.5 and 5.3.
struct TileRule
{
    int min_tiles;      // 256-route tiles of the call
    int min_rows;       // routes of an expert that takes them
    int min_rest;       // remainder of c / 256 that takes one more
    int min_small;      // smallest remainder in a 128-route tile
    int fold;           // the shorter remainders of the layer that go with them
};
constexpr int FT_BIG_WORK = 3 * 256;
constexpr int FT_BIG_ROWS = 3 * FT_BIG;
constexpr int FT_REST = 193;        // two FT_MID tiles hold 192
constexpr int FT_REST_LARGE = 129;
constexpr int FT_LARGE = 80000;
constexpr int GRP_ROWS = 32;        // rows of a row group
constexpr int GRP_HALVES = 1024;    // one matrix's 32-element step of a row group
// 128-blocks per input transform workgroup (16,384 tokens, H 4096, 2.3 GB written: 783 us with 2, 844 with 4, 946 with 8;
// nontemporal stores of 4: 828 us, and 225 against 204 us at 4,096 tokens)
constexpr int PREP_BLOCKS = 2;
constexpr int FT_BN = 256;          // output columns per tile
constexpr int FT_WAVES = 8;
constexpr int FT_THREADS = 64 * FT_WAVES;
constexpr int FT16_THREADS = 1024;   // the sixteen-wave form
constexpr int FT_PA = 3;            // input ring stages (loads run FT_PA - 1 steps ahead)
constexpr int FT_PT = 5;            // trellis steps in flight
constexpr int FT_TS = FT_PT + 1;    // trellis ring slots
constexpr int FT_PLAN_MAX = 1024;   // active experts the plan kernel handles

// A tile of routes of one expert: rows row0 .. of record ai, whose inputs start at row group `group`.
struct FatTile
{
    int32_t ai, row0, group, pad;
};

struct FatArgs
{
    const ExpertRec* rec;         // [max_active] active experts (permutation order)
    const FatTile* tiles;         // this launch's tiles
    const int32_t* ntiles;        // [1]
    const uint16_t* xa;           // inputs in row groups: mode 0 [groups][H/32][gate, up][1024], mode 1 [groups][I/32][1024]
    const uint16_t* svh13;        // [E][2][I]
    const uint16_t* suh2;         // [E][I]
    const uint16_t* svh2;         // [E][H]
    const int32_t* route_at;      // [n] flat route index of each sorted position
    uint16_t* xd;                 // mode 0 output: the down inputs, in row groups
    float* Y;                     // mode 1 output [n_routes][H] (per route), fp32 or (YH) fp16 bits
    const float* xs;              // input sums [groups][nxs][NA][32] (affine decode), NA = 2 in mode 0, 1 in mode 1
    float* xds;                   // mode 0 output: sums of the down inputs [groups][nxds = I / 128][32]
    int H, I, K, N, nunits, nxs, nxds;
    float limit;
};

// Transformed inputs of every fat route (k_fat_prep): r16(FWHT(x16 * suh_m) * HAD) per 128-block (ft_core.h:96-102),
// where x16 is fp16 input as is, or bf16 / fp32 input rounded through bf16, in the row groups described above.
//
// 16 lanes hold a block, 8 elements per lane: lane 4 q + g of a block holds the elements k = 32 q + 2 g + j + 8 h + 16 t
// (j, h, t in {0, 1}) as v[4 t + 2 h + j], exactly chunk g of step q, so it stores them with one 16-byte write. The
// butterflies keep the reference's order and arithmetic (strides 1, 2, 4, ..., 64,
// (a, b) -> (a + b, a - b), ft_core.h:89-94): strides 1, 8, 16 pair elements within a lane; strides 2 and 4 pair
// lanes 4 q + g and 4 q + (g ^ 1 or 2), strides 32 and 64 lanes q ^ 1 and q ^ 2 of the block (DPP moves, all
// within the block's 16 lanes). The lane holding the upper element of a cross-lane pair forms partner - self as
// fma(-1, self, partner), the same single rounding.
__device__ __forceinline__ float xlane(float v, int pattern)
{
    if (pattern == 1) return xor_lane<1>(v);
    if (pattern == 2) return xor_lane<2>(v);
    if (pattern == 4) return xor_lane<4>(v);
    return xor_lane<8>(v);
}

// The 128-point transform of a block held by 16 lanes (lane 4 q + g of the block) with 8 elements each,
// v[4 t + 2 h + j] = element 32 q + 2 g + j + 8 h + 16 t. sgn = (g & 1, g & 2, q & 1, q & 2 ? -1 : 1).
struct Lane8Signs
{
    float s2, s4, s32, s64;
};
__device__ __forceinline__ Lane8Signs lane8_signs(int lane)
{
    const int g = lane & 3, q = (lane >> 2) & 3;
    return { (g & 1) ? -1.0f : 1.0f, (g & 2) ? -1.0f : 1.0f, (q & 1) ? -1.0f : 1.0f, (q & 2) ? -1.0f : 1.0f };
}
__device__ __forceinline__ void fwht128_lane8(float (&v)[8], const Lane8Signs& sg)
{
    // stride 1 (j)
#pragma unroll
    for (int i = 0; i < 8; i += 2)
    {
        const float a0 = v[i], a1 = v[i + 1];
        v[i] = a0 + a1;
        v[i + 1] = a0 - a1;
    }
    // strides 2, 4 (lanes g ^ 1, g ^ 2)
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_fmaf(sg.s2, v[i], xlane(v[i], 1));
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_fmaf(sg.s4, v[i], xlane(v[i], 2));
    // strides 8 (h), 16 (t)
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if ((i & 2) == 0)
        {
            const float a0 = v[i], a1 = v[i + 2];
            v[i] = a0 + a1;
            v[i + 2] = a0 - a1;
        }
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const float a0 = v[i], a1 = v[i + 4];
        v[i] = a0 + a1;
        v[i + 4] = a0 - a1;
    }
    // strides 32, 64 (lanes q ^ 1, q ^ 2)
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_fmaf(sg.s32, v[i], xlane(v[i], 4));
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_fmaf(sg.s64, v[i], xlane(v[i], 8));
}
// element index of v[i] in its 128-block for the lane (q, g) of the block
__device__ __forceinline__ int lane8_k(int lane, int i)
{
    return 32 * ((lane >> 2) & 3) + 2 * (lane & 3) + (i & 1) + 8 * ((i >> 1) & 1) + 16 * (i >> 2);
}

// One 16-lane group transforms one row of a row group: blocks b0 .. b1 - 1 of the token's row, both matrices (the
// input is read once), two blocks per pass, all loaded before any is used. SUMS: sum[m] += the values of matrix m.
template <int XD, bool SUMS>
__device__ __forceinline__ void fat_prep_row(const void* x, size_t row, const uint16_t* su0, uint16_t* dst, int H,
                                             int b0, int b1, float (&sum)[2])
{
    const int lane = threadIdx.x & 63;
    const int g = lane & 3, q = (lane >> 2) & 3;
    const Lane8Signs sg = lane8_signs(lane);
    // raw words of element pair (t, h): fp16 / bf16 input as one dword, fp32 as two
    using Raw = typename std::conditional<XD == MM_DTYPE_F32, uint2, uint32_t>::type;
    for (int f0 = b0; f0 < b1; f0 += 2)
    {
        Raw xr[2][4];
        uint32_t sr[2][2][4];
#pragma unroll
        for (int it = 0; it < 2; ++it)
        {
            const int k0 = min(f0 + it, b1 - 1) * 128 + 32 * q + 2 * g;
#pragma unroll
            for (int th = 0; th < 4; ++th)
            {
                const int k = k0 + 8 * (th & 1) + 16 * (th >> 1);
                if constexpr (XD == MM_DTYPE_F32)
                    xr[it][th] = *reinterpret_cast<const uint2*>(static_cast<const float*>(x) + row + k);
                else
                    xr[it][th] = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(x) + row + k);
                sr[it][0][th] = *reinterpret_cast<const uint32_t*>(su0 + k);
                sr[it][1][th] = *reinterpret_cast<const uint32_t*>(su0 + H + k);
            }
        }
#pragma unroll
        for (int it = 0; it < 2; ++it)
        {
            const int b = f0 + it;
            if (b >= b1) break;
            // th = 2 t + h: elements 8 h + 16 t (+ 0, 1) of the lane's column pair go to xv[4 t + 2 h + j]
            float xv[8];
#pragma unroll
            for (int th = 0; th < 4; ++th)
            {
                const int i = 4 * (th >> 1) + 2 * (th & 1);
                if constexpr (XD == MM_DTYPE_F16)
                {
                    xv[i] = h2f((uint16_t)(xr[it][th] & 0xffffu));
                    xv[i + 1] = h2f((uint16_t)(xr[it][th] >> 16));
                }
                else if constexpr (XD == MM_DTYPE_BF16)
                {
                    xv[i] = r16(__uint_as_float(xr[it][th] << 16));
                    xv[i + 1] = r16(__uint_as_float(xr[it][th] & 0xffff0000u));
                }
                else
                {
                    xv[i] = r16(bf16_value(__uint_as_float(xr[it][th].x)));
                    xv[i + 1] = r16(bf16_value(__uint_as_float(xr[it][th].y)));
                }
            }
#pragma unroll
            for (int m = 0; m < 2; ++m)
            {
                float v[8];
#pragma unroll
                for (int th = 0; th < 4; ++th)
                {
                    const int i = 4 * (th >> 1) + 2 * (th & 1);
                    v[i] = xv[i] * h2f((uint16_t)(sr[it][m][th] & 0xffffu));
                    v[i + 1] = xv[i + 1] * h2f((uint16_t)(sr[it][m][th] >> 16));
                }
                fwht128_lane8(v, sg);
                if constexpr (SUMS)
#pragma unroll
                    for (int i = 0; i < 8; ++i) sum[m] += r16(v[i] * HAD);
                uint4 o;
                o.x = (uint32_t)f2h(v[0] * HAD) | ((uint32_t)f2h(v[1] * HAD) << 16);
                o.y = (uint32_t)f2h(v[2] * HAD) | ((uint32_t)f2h(v[3] * HAD) << 16);
                o.z = (uint32_t)f2h(v[4] * HAD) | ((uint32_t)f2h(v[5] * HAD) << 16);
                o.w = (uint32_t)f2h(v[6] * HAD) | ((uint32_t)f2h(v[7] * HAD) << 16);
                *reinterpret_cast<uint4*>(dst + ((size_t)(4 * b + q) * 2 + m) * GRP_HALVES + g * 256) = o;
            }
        }
    }
}

// One workgroup per (row group, PREP_BLOCKS 128-blocks of the input row): wave w transforms rows 4 w .. 4 w + 3, so the
// workgroup's waves together write whole 512-byte runs of the row group. The token of a position is token_sorted's
// (a position of a token outside [0, T) is left unwritten), or order[pos] / topk.
template <bool SUMS>
__global__ __launch_bounds__(512) void k_fat_prep(const void* x, int x_dtype, const int32_t* order,
                                                  const int64_t* token_sorted, const ExpertRec* rec, const int2* groups,
                                                  const int32_t* ngroups, const uint16_t* suh13, uint16_t* xa, float* xs,
                                                  int topk, int T, int H)
{
    const int G = blockIdx.x, rl = threadIdx.x >> 4;
    if (G >= ngroups[0]) return;
    const int2 gi = groups[G];                       // record and first row
    const ExpertRec* r = rec + gi.x;
    if (gi.y + rl >= r->cnt) return;
    const int pos = r->first + gi.y + rl;
    const int64_t t = token_sorted ? token_sorted[pos] : (int64_t)(order[pos] / topk);
    if (t < 0 || t >= T) return;
    const int nb = H / 128, b0 = blockIdx.y * PREP_BLOCKS, b1 = min(nb, b0 + PREP_BLOCKS);
    const uint16_t* su0 = suh13 + (size_t)r->e * 2 * H;       // gate; up follows
    uint16_t* dst = xa + (size_t)G * 64 * H + rl * 8;          // a row group: 32 rows x 2 matrices x H
    float sum[2] = { 0.0f, 0.0f };
    if (x_dtype == MM_DTYPE_F16)
        fat_prep_row<MM_DTYPE_F16, SUMS>(x, (size_t)t * H, su0, dst, H, b0, b1, sum);
    else if (x_dtype == MM_DTYPE_BF16)
        fat_prep_row<MM_DTYPE_BF16, SUMS>(x, (size_t)t * H, su0, dst, H, b0, b1, sum);
    else
        fat_prep_row<MM_DTYPE_F32, SUMS>(x, (size_t)t * H, su0, dst, H, b0, b1, sum);
    if constexpr (!SUMS) return;
#pragma unroll
    for (int m = 0; m < 2; ++m)
    {
        sum[m] += xor_lane<1>(sum[m]);
        sum[m] += xor_lane<2>(sum[m]);
        sum[m] += xor_lane<4>(sum[m]);
        sum[m] += xor_lane<8>(sum[m]);
        if ((threadIdx.x & 15) == 0) xs[(((size_t)G * gridDim.y + blockIdx.y) * 2 + m) * GRP_ROWS + rl] = sum[m];
    }
}

// 256-route tiles of an expert with c routes; the rest (fewer than min_rest routes) goes to the other tiles.
__device__ __forceinline__ int fat_big_tiles(int c, int min_rest) { return c / FT_BIG + (c % FT_BIG >= min_rest ? 1 : 0); }

// Expert records, row groups and the tile lists of the experts with more than cap routes, one workgroup: thread a counts
// expert a's tiles and groups, the lists are then filled by all threads, each entry finding its expert by a binary search
// over the sums in LDS. totals = 256-route tiles, FT_MID-route tiles, row groups, 128-route tiles. The FT_MID-route list
// holds the tiles of
// three row groups first, then those of two, then those of one: the longest start first.
// CHOICE (a fused call that either path may take, cap 0): the active experts and routed positions that the decode path is to
// compute go to choice[0], [1]: all of them and no tile here, or none (see fused_path).
template <bool CHOICE>
__global__ __launch_bounds__(FT_PLAN_MAX) void k_fat_plan(const int32_t* counts, const int32_t* offsets,
                                                         const int32_t* active, const int32_t* nactive,
                                                         const int64_t* gate, const int64_t* up, const int64_t* down,
                                                         ExpertRec* rec, FatTile* big, FatTile* small, FatTile* mid,
                                                         int2* groups, int32_t* totals, int max_active, int cap, TileRule rule,
                                                         const int32_t* layer_counts, int32_t* choice, int E, int n)
{
    // lists: 256-route tiles; tiles of three, two and one row groups; row groups; 128-route tiles
    constexpr int NL = 6;
    __shared__ int s_w[NL][FT_PLAN_MAX / 64];
    __shared__ int s_off[NL][FT_PLAN_MAX + 1];             // exclusive sums
    const int a = threadIdx.x, lane = a & 63, wave = a >> 6;
    const int nact = min(nactive[0], max_active);
    int c = 0;
    if (a < nact)
    {
        const int e = active[a];
        c = counts[e];
        ExpertRec r{ e, c, offsets[e], 0, { gate[e], up[e], down[e] }, 0 };
        rec[a] = r;
    }
    if (c <= cap) c = 0;
    // exclusive sums of list i into s_off[i]
    auto scan = [&](int i, int v) {
        const int incl = wave_incl_scan(v);
        if (lane == 63) s_w[i][wave] = incl;
        __syncthreads();
        int base = 0, total = 0;
        for (int w = 0; w < FT_PLAN_MAX / 64; ++w)
        {
            if (w < wave) base += s_w[i][w];
            total += s_w[i][w];
        }
        s_off[i][a] = base + incl - v;
        if (a == 0) s_off[i][FT_PLAN_MAX] = total;
        return total;
    };
    if constexpr (CHOICE)
    {
        const int64_t records = scan(1, (c + 15) / 16), tiles = scan(2, (c + FT_MID - 1) / FT_MID);
        __syncthreads();
        const bool decode = 800 * records + 8 * (int64_t)n <= 900 * tiles + 10400;
        if (a == 0)
        {
            choice[0] = decode ? nact : 0;
            choice[1] = decode ? offsets[E] : 0;
        }
        if (decode) c = 0;
    }
    int nbig = c >= rule.min_rows ? fat_big_tiles(c, rule.min_rest) : 0;
    if (scan(0, nbig) < rule.min_tiles) nbig = 0;                 // uniform: too few to fill the GPU
    __syncthreads();
    const int tbig = scan(0, nbig);
    int rest = max(c - nbig * FT_BIG, 0), nsmall = 0, tsmall = 0;
    if (rule.min_small <= FT_SMALL)
    {
        // the shorter remainders of the whole layer, computed here or not
        int shorter = 0;
        if (a < E)
        {
            const int lc = max(layer_counts[a], 0);
            const int lr = lc - (lc >= rule.min_rows ? fat_big_tiles(lc, rule.min_rest) : 0) * FT_BIG;
            shorter = lr > 0 && lr < rule.min_small ? 1 : 0;
        }
        const bool fold = scan(1, shorter) <= rule.fold;
        nsmall = rest > 0 && rest <= FT_SMALL && (fold || rest >= rule.min_small) ? 1 : 0;
        tsmall = scan(5, nsmall);
    }
    if (nsmall) rest = 0;
    const int full = rest / FT_MID, r = rest % FT_MID;
    __syncthreads();
    const int t3 = scan(1, full + (r > 2 * GRP_ROWS ? 1 : 0));
    const int t2 = scan(2, r > GRP_ROWS && r <= 2 * GRP_ROWS ? 1 : 0);
    const int t1 = scan(3, r > 0 && r <= GRP_ROWS ? 1 : 0);
    const int tg = scan(4, (c + GRP_ROWS - 1) / GRP_ROWS);
    if (a == 0)
    {
        totals[0] = tbig;
        totals[1] = t3 + t2 + t1;
        totals[2] = tg;
        totals[3] = tsmall;
    }
    __syncthreads();
    // entry j of list i belongs to the last expert whose sum is at most j (later experts without entries share it)
    auto owner = [&](int i, int j) {
        int lo = 0, hi = FT_PLAN_MAX;
        while (hi - lo > 1)
        {
            const int m = (lo + hi) >> 1;
            if (s_off[i][m] <= j) lo = m; else hi = m;
        }
        return lo;
    };
    for (int j = a; j < tbig; j += FT_PLAN_MAX)
    {
        const int o = owner(0, j), row0 = (j - s_off[0][o]) * FT_BIG;
        big[j] = FatTile{ o, row0, s_off[4][o] + row0 / GRP_ROWS, 0 };
    }
    for (int j = a; j < tsmall; j += FT_PLAN_MAX)
    {
        const int o = owner(5, j), row0 = (s_off[0][o + 1] - s_off[0][o]) * FT_BIG;
        small[j] = FatTile{ o, row0, s_off[4][o] + row0 / GRP_ROWS, 0 };
    }
    for (int j = a; j < t3 + t2 + t1; j += FT_PLAN_MAX)
    {
        const int i = j < t3 ? 1 : j < t3 + t2 ? 2 : 3, k = j - (i == 1 ? 0 : i == 2 ? t3 : t3 + t2);
        const int o = owner(i, k);
        // the tiles of three row groups come first within an expert's rest; a shorter one follows them
        const int before = i == 1 ? k - s_off[1][o] : s_off[1][o + 1] - s_off[1][o];
        const int row0 = (s_off[0][o + 1] - s_off[0][o]) * FT_BIG + before * FT_MID;
        mid[j] = FatTile{ o, row0, s_off[4][o] + row0 / GRP_ROWS, 0 };
    }
    for (int j = a; j < tg; j += FT_PLAN_MAX)
    {
        const int o = owner(4, j);
        groups[j] = make_int2(o, (j - s_off[4][o]) * GRP_ROWS);
    }
}

// Work item of this workgroup. The grid is sized for the most tiles a call can have; the work = tiles x column units of
// this call is spread evenly over the 8 XCDs (workgroup b runs on XCD b % 8), and consecutive work items (the column
// units of one tile, then the next tile of the same expert) stay on one XCD, so they share its L2 for the inputs and
// the trellis.
__device__ __forceinline__ bool fat_work(const FatArgs& a, int& mt, int& nu)
{
    const int work = a.ntiles[0] * a.nunits, per_xcd = (work + 7) >> 3;
    const int L = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || L >= work) return false;
    mt = L / a.nunits;
    nu = L % a.nunits;
    return true;
}

// A wave-uniform pointer for a buffer descriptor (each half widened as uint32_t: readfirstlane returns int).
__device__ __forceinline__ void* uniform_ptr(const void* p)
{
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t l = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t h = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return reinterpret_cast<void*>((uintptr_t)((uint64_t)l | ((uint64_t)h << 32)));
}

// Epilogue of a fat tile from the transposed fp16 C tile in LDS (column c at c * CS halves, the raw GEMM outputs
// rounded to fp16): gate/up (MODE 0) applies the output transforms, SwiGLU and the down-input transform of the
// tile's 128-block and writes the down input in operand order; down (MODE 1) applies the output transform of its
// two 128-blocks and writes per-route rows. The C tile is complete (the caller's barrier) when this runs. sc = the scales of
// the tile's columns (gate/up: svh of gate, of up, suh of down, 128 each; down: svh of 256), route = the output rows of its
// positions (down).
template <int MODE, int CS, bool YH, int NW = FT_WAVES, bool SUMS = false>
__device__ __forceinline__ void fat_tile_epilogue(const FatArgs& a, const uint16_t* C, int rows,
                                                  int nu, size_t grp, int wave, int lane, const uint16_t* const (&sc)[3],
                                                  const int32_t* route)
{
    // Transforms in the layout of fwht128_lane8: per pass a wave takes 8 rows; lane (rpair, q, g) = (lane >> 4,
    // (lane >> 2) & 3, lane & 3) holds rows r0 + 2 rpair and r0 + 2 rpair + 1 (one dword of the transposed tile per
    // column) of the 8 columns lane8_k(lane, i) of each 128-block, so each butterfly stage is in-lane or a DPP
    // exchange within 16 lanes.
    const Lane8Signs sg = lane8_signs(lane);
    const int rpair = lane >> 4;
    int kk[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) kk[i] = lane8_k(lane, i);
    // column c at rows r, r + 1 (r even)
    auto rows2 = [&](int c, int r, float& v0, float& v1) {
        const uint32_t d = *reinterpret_cast<const uint32_t*>(C + (size_t)c * CS + r);
        v0 = h2f((uint16_t)(d & 0xffffu));
        v1 = h2f((uint16_t)(d >> 16));
    };
    if constexpr (MODE == 0)
    {
        const int c0 = nu * 128;
        float sgv[8], suv[8], sdv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
        {
            sgv[i] = h2f(sc[0][kk[i]]);
            suv[i] = h2f(sc[1][kk[i]]);
            sdv[i] = h2f(sc[2][kk[i]]);
        }
        // the lane's 8 elements are chunk g of step c0 / 32 + q of its row's group
        uint16_t* od = a.xd + (size_t)(c0 / 32 + ((lane >> 2) & 3)) * GRP_HALVES + 256 * (lane & 3);
        for (int r0 = 8 * wave; r0 < rows; r0 += 8 * NW)
        {
            const int r = r0 + 2 * rpair;
            float gv[2][8], uv[2][8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                rows2(kk[i], r, gv[0][i], gv[1][i]);
                rows2(128 + kk[i], r, uv[0][i], uv[1][i]);
            }
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2)
            {
                // the tile holds fp16 values, so the output transform's first rounding is exact
                fwht128_lane8(gv[h2], sg);
                fwht128_lane8(uv[h2], sg);
                float xv[8];
#pragma unroll
                for (int i = 0; i < 8; ++i)
                {
                    const float gg = r16((gv[h2][i] * HAD) * sgv[i]);
                    const float uu = r16((uv[h2][i] * HAD) * suv[i]);
                    xv[i] = r16(act_gu(gg, uu, a.limit)) * sdv[i];
                }
                fwht128_lane8(xv, sg);
                if constexpr (SUMS)
                {
                    // sum of the block's 128 rounded values over its 16 lanes
                    float sum = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) sum += r16(xv[i] * HAD);
                    sum += xor_lane<1>(sum);
                    sum += xor_lane<2>(sum);
                    sum += xor_lane<4>(sum);
                    sum += xor_lane<8>(sum);
                    const int rr = r + h2;
                    if ((lane & 15) == 0 && rr < rows)
                        a.xds[((grp + (rr >> 5)) * a.nxds + nu) * GRP_ROWS + (rr & 31)] = sum;
                }
                if (r + h2 < rows)
                {
                    uint4 o;
                    o.x = (uint32_t)f2h(xv[0] * HAD) | ((uint32_t)f2h(xv[1] * HAD) << 16);
                    o.y = (uint32_t)f2h(xv[2] * HAD) | ((uint32_t)f2h(xv[3] * HAD) << 16);
                    o.z = (uint32_t)f2h(xv[4] * HAD) | ((uint32_t)f2h(xv[5] * HAD) << 16);
                    o.w = (uint32_t)f2h(xv[6] * HAD) | ((uint32_t)f2h(xv[7] * HAD) << 16);
                    const int rr = r + h2;
                    *reinterpret_cast<uint4*>(od + (grp + (rr >> 5)) * 32 * a.I + 8 * (rr & 31)) = o;
                }
            }
        }
    }
    else
    {
        float svv[2][8];
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
            for (int i = 0; i < 8; ++i) svv[hb][i] = h2f(sc[hb][kk[i]]);
        for (int r0 = 8 * wave; r0 < rows; r0 += 8 * NW)
        {
            const int r = r0 + 2 * rpair;
            // output rows of the lane's two routes (a row past the tile's routes is not stored)
            const int y0 = r < rows ? route[r] : 0;
            const int y1 = r + 1 < rows ? route[r + 1] : 0;
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
            {
                const int c0 = (2 * nu + hb) * 128;
                float yv[2][8];
#pragma unroll
                for (int i = 0; i < 8; ++i) rows2(hb * 128 + kk[i], r, yv[0][i], yv[1][i]);
#pragma unroll
                for (int h2 = 0; h2 < 2; ++h2)
                {
                    fwht128_lane8(yv[h2], sg);
#pragma unroll
                    for (int i = 0; i < 8; ++i) yv[h2][i] = r16((yv[h2][i] * HAD) * svv[hb][i]);
                    if (r + h2 < rows)
                    {
                        const size_t yo = (size_t)(h2 ? y1 : y0) * a.H + c0;
                        // elements 2 p, 2 p + 1 are adjacent columns kk[2 p], kk[2 p] + 1
#pragma unroll
                        for (int p2 = 0; p2 < 4; ++p2)
                        {
                            if constexpr (YH)
                            {
                                // the output transform rounded y to fp16: the half stores are exact
                                const uint32_t w2 = (uint32_t)f2h(yv[h2][2 * p2]) | ((uint32_t)f2h(yv[h2][2 * p2 + 1]) << 16);
                                *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(a.Y) + yo + kk[2 * p2]) = w2;
                            }
                            else
                            {
                                *reinterpret_cast<float2*>(a.Y + yo + kk[2 * p2]) =
                                    make_float2(yv[h2][2 * p2], yv[h2][2 * p2 + 1]);
                            }
                        }
                    }
                }
            }
        }
    }
}

// The scales of column unit nu of expert e (fat_tile_epilogue).
template <int MODE>
__device__ __forceinline__ void fat_scales(const FatArgs& a, int e, int nu, const uint16_t* (&sc)[3])
{
    if constexpr (MODE == 0)
    {
        sc[0] = a.svh13 + ((size_t)e * 2 + 0) * a.I + nu * 128;
        sc[1] = a.svh13 + ((size_t)e * 2 + 1) * a.I + nu * 128;
        sc[2] = a.suh2 + (size_t)e * a.I + nu * 128;
    }
    else
    {
        sc[0] = sc[2] = a.svh2 + (size_t)e * a.H + nu * 256;
        sc[1] = sc[0] + 128;
    }
}

// Gate/up tiles of FT_BIG routes, MB = 8 row blocks of 16 per row-wave. 8 waves: wave (wm, wn) = (w >> 2,
// w & 3) multiplies row blocks wm, wm + 2, wm + 4, ... (rows 16 (2 i + wm) .. + 15) by column tiles 4 wn .. 4 wn + 3
// of 16, so in a tile with fewer routes the two waves of a SIMD keep about the same number of row blocks
// (0.7 % off the 16k layer against contiguous halves); every wave loads an
// eighth of the inputs and waves 0 .. 3 also the trellis (chunk w: tile row w >> 1 of matrix w & 1),
// which runs further ahead; wave w decodes column tiles 2 (w & 3), 2 (w & 3) + 1 of sub-block w >> 2 in both tile
// rows (chunks w >> 2 and 2 + (w >> 2)). Rows past the tile's routes multiply what their row group holds (zeros past the
// last group) and are not stored.
__global__ __launch_bounds__(FT_THREADS, 1) void k_fat(FatArgs a)
{
    constexpr int MB = 8, BM = FT_BIG;
    constexpr int NA = 2;                                        // input matrices (gate, up share the tile)
    constexpr int SEG = NA * 64;                                 // bytes of one route's step (gate, up)
    constexpr int A_STAGE = BM * SEG;                            // one step's inputs
    constexpr int LA = A_STAGE / 1024 / FT_WAVES;                // input loads (1 KB each) per wave and step
    constexpr int T_SLOT = 4 * 1024;                             // one step's trellis: 4 chunks of 8 tiles
    constexpr int B_BUF = 16 * 64 * 16;                          // decoded B of one step: 16 tiles x 64 lanes
    constexpr int A_BYTES = FT_PA * A_STAGE, T_BYTES = FT_TS * T_SLOT;
    constexpr int MAIN = A_BYTES + T_BYTES + 2 * B_BUF;
    constexpr int CS = BM + 2;                                   // transposed C tile: column stride in halves
    constexpr int SMEM = MAIN > FT_BN * CS * 2 ? MAIN : FT_BN * CS * 2;
    static_assert(SMEM <= 160 * 1024, "LDS");
    static_assert(((CS / 2) & 1) == 1, "odd dword stride: conflict-free column reads");
    static_assert(BM == 32 * MB, "two row-waves");
    __shared__ __align__(16) uint8_t smem[SMEM];
    uint8_t* Aring = smem;
    uint8_t* Tring = smem + A_BYTES;
    uint8_t* Bdec = smem + A_BYTES + T_BYTES;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int mt, nu;
    if (!fat_work(a, mt, nu)) return;
    const FatTile* tp = a.tiles + mt;
    const ExpertRec* rp = a.rec + tp->ai;
    const int row0 = tp->row0;
    const int rows = __builtin_amdgcn_readfirstlane(min(BM, rp->cnt - row0));
    const int pos0 = __builtin_amdgcn_readfirstlane(rp->first + row0);
    const int e = __builtin_amdgcn_readfirstlane(rp->e);
    const size_t grp = (size_t)__builtin_amdgcn_readfirstlane(tp->group);
    const int S = a.K / 32;

    const bool tloader = wave < 4;
    // trellis loader (waves 0 .. 3): chunk q = wave of step s is tile row 2 s + (q >> 1) of matrix q & 1, 8 tiles =
    // 768 bytes, 12 bytes per lane stored 16 bytes apart.
    // Steps past the end reload the last row into the free slot, so every step issues one load.
    const int tq = wave & 3;
    const uint32_t row_bytes = (uint32_t)(a.N / 16) * 96, wbytes = (uint32_t)(a.K / 16) * row_bytes;
    const void* wbase = (const void*)(uintptr_t)((tq & 1) ? rp->w[1] : rp->w[0]);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(wbase), (short)0, (int)wbytes,
                                                                          0x00020000);
    const uint32_t wcol = (uint32_t)nu * 768;
    auto load_trellis = [&](int s) {
        const uint32_t tr = (uint32_t)(2 * min(s, S - 1) + (tq >> 1));
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, Tring + (size_t)(s % FT_TS) * T_SLOT + (size_t)tq * 1024, 12,
                                                 tr * row_bytes + wcol + (uint32_t)lane * 12, 0, 0, 0);
    };
    // inputs (every wave): LA loads of 1 KB each (half of one matrix's step of a row group). Row groups past the tile's
    // routes and steps past the end read out of range (zero, no memory access).
    const uint32_t gbytes = (uint32_t)NA * a.K * GRP_ROWS * 2;          // a row group
    const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(a.xa + grp * (gbytes / 2)), (short)0, (int)((uint32_t)((rows + 31) / GRP_ROWS) * gbytes), 0x00020000);
    auto load_input = [&](int s, int u) {
        const int st = s % FT_PA;
        const uint32_t ks = s < S ? (uint32_t)s * (NA * 2048) : 0x40000000u; // the range is below 2^30
        const int li = wave * LA + u;                                  // 0 .. A_STAGE / 1024 - 1
        const uint32_t voff = (uint32_t)(li / (2 * NA)) * gbytes + (uint32_t)(li % (2 * NA)) * 1024 + (uint32_t)lane * 16;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, Aring + (size_t)st * A_STAGE + (size_t)li * 1024, 16, voff + ks, 0, 0, 0);
    };

    // ---- decode: lane (col, g) decodes states i0 .. i0+3 of column col in a tile
    const int col = lane & 15, g = lane >> 4;
    const int i0 = 32 * (col & 7) + 8 * g + 4 * (col >> 3);
    const int eb = 3 * i0 + 11;
    const int blo = eb >> 5, bhi = (blo + 23) % 24;
    const int llo = 4 * (blo / 3) + blo % 3, lhi = 4 * (bhi / 3) + bhi % 3;
    const uint32_t sh = 31u - (uint32_t)(eb & 31);
    // Wave w decodes column tiles 2 (w & 3) and 2 (w & 3) + 1 of sub-block w >> 2 (chunks w >> 2 and 2 + (w >> 2):
    // tile rows 0 and 1 of the step) and stores each column tile's 8 k-values per lane, tile row 0 in the low 8
    // bytes and row 1 in the high 8, as one 16-byte write (lane-contiguous: no LDS bank conflicts). Decoded tile k
    // of the wave (k = 0 .. 3) is tile row k & 1 of column tile 2 (w & 3) + (k >> 1): trellis words at
    // tword + (k & 1) * 512 + (k >> 1) * 32.
    const int db = wave >> 2, dc = 2 * (wave & 3);
    const uint32_t* tword = reinterpret_cast<const uint32_t*>(Tring + (size_t)db * 1024 + (size_t)dc * 128);
    uint8_t* bdst = Bdec + ((size_t)(db * 8 + dc) * 64 + lane) * 16;
    // ---- MFMA: rows 16 (2 i + wm) + col of input matrix wn >> 1, B tiles 4 wn .. + 3
    const int wm = wave >> 2, wn = wave & 3;
    const uint8_t* bsrc = Bdec + ((size_t)(wn * 4) * 64 + lane) * 16;
    int aoff[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
    {
        const int r = 16 * (2 * i + wm) + col;
        aoff[i] = ((r >> 5) * NA + (wn >> 1)) * 2048 + (g * 32 + (r & 31)) * 16;
    }
    float4_t acc[MB][4];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{ 0.f, 0.f, 0.f, 0.f };

    // Loads in issue order, per wave: inputs of step 0, [trellis of steps 0 .. FT_PT - 1], inputs of step 1, then
    // in step s [the trellis of step s + FT_PT] and the inputs of step s + 2 (LA loads, in between the MFMAs);
    // [..] = waves 0 .. 3 only. At the top of step s the inputs of step s (issued in step s - 2, or before the loop)
    // are complete once at most LA (+ 1 trellis load for waves 0 .. 3) loads are outstanding: that is exactly what
    // step s - 1 issued after them (step 0: more than that came after). The trellis of step s + 1 is older than
    // the inputs of step s (FT_PT - 1 > 2 steps earlier, or before them in the prologue, with more than LA + 1 loads
    // after it), so it is complete too. One barrier per step then publishes the loads and the tiles decoded in step
    // s - 1.
    static_assert(FT_PA == 3 && FT_PT >= 4, "issue order above");
#pragma unroll
    for (int u = 0; u < LA; ++u) load_input(0, u);
    asm volatile("" ::: "memory");                                // keep the issue order
    if (tloader)
        for (int s = 0; s < FT_PT; ++s) load_trellis(s);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < LA; ++u) load_input(1, u);
    if (tloader) wait_vmcnt<LA + FT_PT - 1>(); else wait_vmcnt<LA>();          // trellis of step 0
    lds_barrier();
#pragma unroll
    for (int v = 0; v < 2; ++v)
    {
        const half4_t r0 = decode4<true>(tword[v * 32 + lhi], tword[v * 32 + llo], sh);
        const half4_t r1 = decode4<true>(tword[512 + v * 32 + lhi], tword[512 + v * 32 + llo], sh);
        *reinterpret_cast<half8_t*>(bdst + v * 1024) = half8_t{ r0[0], r0[1], r0[2], r0[3], r1[0], r1[1], r1[2], r1[3] };
    }
    // Row blocks of this wave that hold routes of the tile (uniform; blocks i < nvb): in a partial tile a wave skips
    // the MFMAs and input reads of its empty row blocks (their accumulators stay zero and are never stored); loads
    // and decode, which serve the whole workgroup, run either way. Full waves take the scheduled variant.
    const int nvb = max(0, min(MB, ((rows + 15) / 16 - wm + 1) / 2));
    auto main_loop = [&](auto part_tag) {
        constexpr bool PART = decltype(part_tag)::value;
        for (int s = 0; s < S; ++s)
        {
            if (tloader) wait_vmcnt<LA + 1>(); else wait_vmcnt<LA>();
            lds_barrier();
            if (tloader) load_trellis(s + FT_PT);
            // one step: the trellis words of step s + 1 and the operands of step s first, then per row block its 4
            // MFMAs, one tile of step s + 1 decoded after every MB / 4 blocks
            // slot offset as one scalar, so each read is a per-lane base plus an immediate
            const uint32_t toff = (uint32_t)__builtin_amdgcn_readfirstlane(((s + 1) % FT_TS) * T_SLOT);
            const uint8_t* thp = reinterpret_cast<const uint8_t*>(tword + lhi) + toff;
            const uint8_t* tlp = reinterpret_cast<const uint8_t*>(tword + llo) + toff;
            uint32_t th[4], tl[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                th[u] = *reinterpret_cast<const uint32_t*>(thp + (u & 1) * 2048 + (u >> 1) * 128);
                tl[u] = *reinterpret_cast<const uint32_t*>(tlp + (u & 1) * 2048 + (u >> 1) * 128);
            }
            const uint8_t* as = Aring + (size_t)(s % FT_PA) * A_STAGE;
            const uint8_t* bs = bsrc + (size_t)(s & 1) * B_BUF;
            uint8_t* bd = bdst + (size_t)((s + 1) & 1) * B_BUF;
            // every operand of the step is read before the step's LDS writes (input loads, decoded tiles): the
            // compiler keeps LDS accesses that may alias in program order, so reads placed after a write would each
            // wait a full LDS round trip
            half8_t B[4], A[MB];
#pragma unroll
            for (int j = 0; j < 4; ++j) B[j] = *reinterpret_cast<const half8_t*>(bs + j * 1024);
#pragma unroll
            for (int i = 0; i < MB; ++i)
                if (!PART || i < nvb) A[i] = *reinterpret_cast<const half8_t*>(as + aoff[i]);
            // tile 0 is decoded before the first MFMA: the decode runs while the workgroup's operand reads of the
            // step are still being served (about 2 % off the layer against decoding it after the MFMAs of row
            // blocks 0 .. MB / 4 - 1); tiles 1 .. 3 follow row blocks MB / 4 - 1, MB / 2 - 1, 3 MB / 4 - 1, and
            // each column tile is stored once both of its tile rows are decoded
            half4_t d0 = decode4<true>(th[0], tl[0], sh);
#pragma unroll
            for (int i = 0; i < MB; ++i)
            {
                if (!PART || i < nvb)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i], B[j], acc[i][j], 0, 0, 0);
                if (i % (MB / LA) == 0) load_input(s + FT_PA - 1, i / (MB / LA));
                if (i % (MB / 4) == MB / 4 - 1 && i / (MB / 4) < 3)
                {
                    const int u = i / (MB / 4) + 1;
                    const half4_t d = decode4<true>(th[u], tl[u], sh);
                    if (u & 1)
                        *reinterpret_cast<half8_t*>(bd + (u >> 1) * 1024) =
                            half8_t{ d0[0], d0[1], d0[2], d0[3], d[0], d[1], d[2], d[3] };
                    else
                        d0 = d;
                }
            }
            // schedule: the LDS reads first, the decode of tile 0, then one MFMA followed by two VALU
            // instructions (the rest of the decode, which needs about that many per MFMA), so a wave keeps its MFMA
            // pipe busy between its own decode instructions
            if constexpr (!PART)
            {
                __builtin_amdgcn_sched_group_barrier(0x0100, 4 + MB + 8, 0);
                __builtin_amdgcn_sched_group_barrier(0x0002, 16, 0);
#pragma unroll
                for (int k = 0; k < 4 * MB; ++k)
                {
                    __builtin_amdgcn_sched_group_barrier(0x0008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x0002, 2, 0);
                }
            }
        }
    };
    if (nvb == MB)
        main_loop(std::false_type{});
    else
        main_loop(std::true_type{});
    wait_vmcnt<0>();
    lds_barrier();

    // ---- epilogue through a transposed fp16 C tile in LDS (column c at c * CS halves; the output transforms
    // round y to fp16 first)
    uint16_t* C = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int c = (wn * 4 + j) * 16 + col, r = 16 * (2 * i + wm) + 4 * g;
            uint32_t* d = reinterpret_cast<uint32_t*>(C + (size_t)c * CS + r);
            d[0] = (uint32_t)f2h(acc[i][j][0]) | ((uint32_t)f2h(acc[i][j][1]) << 16);
            d[1] = (uint32_t)f2h(acc[i][j][2]) | ((uint32_t)f2h(acc[i][j][3]) << 16);
        }
    __syncthreads();
    const uint16_t* sc[3];
    fat_scales<0>(a, e, nu, sc);
    fat_tile_epilogue<0, CS, false>(a, C, rows, nu, grp, wave, lane, sc, a.route_at + pos0);
}

// Sixteen-wave form of the tile (four waves per SIMD, at most 64 accumulators per lane): MBW = row blocks per wave, BM =
// 64 MBW routes (4: 256, down only; 2: 128). Wave (wm, wn) = (w >> 2, w & 3) multiplies row blocks wm, wm + 4, ... (rows
// 16 (4 i + wm) .. + 15) by column tiles 4 wn .. 4 wn + 3, so each SIMD (waves w, w + 4, w + 8, w + 12) holds
// one column group over every row block of the tile. Inputs: buffer-to-LDS, two steps ahead in a three-stage ring,
// input load li of a step (1 KB) issued by wave li % 16; trellis as k_fat (waves 0 .. 3); wave w decodes column
// tile w & 7 of sub-block w >> 3 in both tile rows (one 16-byte store per lane and step).
template <int MODE, int MBW, bool YH = false>
__global__ __launch_bounds__(FT16_THREADS, 1) void k_fat16(FatArgs a)
{
    constexpr int NW = 16;
    constexpr int BM = 64 * MBW;
    constexpr int NA = MODE == 0 ? 2 : 1;
    constexpr int SEG = NA * 64;
    constexpr int A_STAGE = BM * SEG;
    constexpr int NL = A_STAGE / 1024;                           // input loads of a step
    constexpr int T_SLOT = 4 * 1024;
    constexpr int B_BUF = 16 * 64 * 16;
    constexpr int A_BYTES = FT_PA * A_STAGE, T_BYTES = FT_TS * T_SLOT;
    constexpr int MAIN = A_BYTES + T_BYTES + 2 * B_BUF;
    constexpr int CS = BM + 2;
    constexpr int SMEM = MAIN > FT_BN * CS * 2 ? MAIN : FT_BN * CS * 2;
    static_assert(SMEM <= 160 * 1024, "LDS");
    static_assert(((CS / 2) & 1) == 1, "odd dword stride: conflict-free column reads");
    static_assert(NL >= 4 && NL <= 2 * NW, "the trellis loaders also load inputs; at most two input loads per wave");
    __shared__ __align__(16) uint8_t smem[SMEM];
    uint8_t* Aring = smem;
    uint8_t* Tring = smem + A_BYTES;
    uint8_t* Bdec = smem + A_BYTES + T_BYTES;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int mt, nu;
    if (!fat_work(a, mt, nu)) return;
    const FatTile* tp = a.tiles + mt;
    const ExpertRec* rp = a.rec + tp->ai;
    const int row0 = tp->row0;
    const int rows = __builtin_amdgcn_readfirstlane(min(BM, rp->cnt - row0));
    const int pos0 = __builtin_amdgcn_readfirstlane(rp->first + row0);
    const int e = __builtin_amdgcn_readfirstlane(rp->e);
    const size_t grp = (size_t)__builtin_amdgcn_readfirstlane(tp->group);
    const int S = a.K / 32;

    const bool tloader = wave < 4;
    const int tq = wave & 3;
    const uint32_t row_bytes = (uint32_t)(a.N / 16) * 96, wbytes = (uint32_t)(a.K / 16) * row_bytes;
    const void* wbase = (const void*)(uintptr_t)(MODE == 0 ? ((tq & 1) ? rp->w[1] : rp->w[0]) : rp->w[2]);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(wbase), (short)0, (int)wbytes,
                                                                          0x00020000);
    const uint32_t wcol = MODE == 0 ? (uint32_t)nu * 768 : (uint32_t)(2 * nu + (tq & 1)) * 768;
    auto load_trellis = [&](int s) {
        const uint32_t tr = (uint32_t)(2 * min(s, S - 1) + (tq >> 1));
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, Tring + (size_t)(s % FT_TS) * T_SLOT + (size_t)tq * 1024, 12,
                                                 tr * row_bytes + wcol + (uint32_t)lane * 12, 0, 0, 0);
    };
    const uint32_t gbytes = (uint32_t)NA * a.K * GRP_ROWS * 2;
    const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(a.xa + grp * (gbytes / 2)), (short)0, (int)((uint32_t)((rows + 31) / GRP_ROWS) * gbytes), 0x00020000);
    // input load li = wave + 16 u of a step; this wave issues na of them (uniform)
    const int na = wave < NL ? (wave + NW < NL ? 2 : 1) : 0;
    auto load_input = [&](int s, int u) {
        const int st = s % FT_PA;
        const uint32_t ks = s < S ? (uint32_t)s * (NA * 2048) : 0x40000000u;
        const int li = wave + NW * u;
        const uint32_t voff = (uint32_t)(li / (2 * NA)) * gbytes + (uint32_t)(li % (2 * NA)) * 1024 + (uint32_t)lane * 16;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, Aring + (size_t)st * A_STAGE + (size_t)li * 1024, 16, voff + ks, 0, 0, 0);
    };
    auto load_inputs = [&](int s) {
        if (na > 0) load_input(s, 0);
        if (na > 1) load_input(s, 1);
    };

    const int col = lane & 15, g = lane >> 4;
    const int i0 = 32 * (col & 7) + 8 * g + 4 * (col >> 3);
    const int eb = 3 * i0 + 11;
    const int blo = eb >> 5, bhi = (blo + 23) % 24;
    const int llo = 4 * (blo / 3) + blo % 3, lhi = 4 * (bhi / 3) + bhi % 3;
    const uint32_t sh = 31u - (uint32_t)(eb & 31);
    const int db = wave >> 3, dc = wave & 7;
    const uint32_t* tword = reinterpret_cast<const uint32_t*>(Tring + (size_t)db * 1024 + (size_t)dc * 128);
    uint8_t* bdst = Bdec + ((size_t)(db * 8 + dc) * 64 + lane) * 16;
    const int wm = wave >> 2, wn = wave & 3;
    const uint8_t* bsrc = Bdec + ((size_t)(wn * 4) * 64 + lane) * 16;
    int aoff[MBW];
#pragma unroll
    for (int i = 0; i < MBW; ++i)
    {
        const int r = 16 * (4 * i + wm) + col;
        aoff[i] = ((r >> 5) * NA + (MODE == 0 ? (wn >> 1) : 0)) * 2048 + (g * 32 + (r & 31)) * 16;
    }
    float4_t acc[MBW][4];
#pragma unroll
    for (int i = 0; i < MBW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{ 0.f, 0.f, 0.f, 0.f };

    // Issue order per wave: inputs of step 0, [trellis of steps 0 .. FT_PT - 1], inputs of step 1, then in step s
    // [the trellis of step s + FT_PT] and the inputs of step s + 2 ([..] = waves 0 .. 3). At the top of step s the
    // wave's inputs of step s are complete once at most na (+ 1) loads are outstanding (what step s - 1 issued
    // after them; step 0: more came after); the trellis of step s + 1 was issued before them.
    auto wait_step = [&]() {
        const int k = na + (tloader ? 1 : 0);
        if (k >= 3) wait_vmcnt<3>();
        else if (k == 2) wait_vmcnt<2>();
        else if (k == 1) wait_vmcnt<1>();
        else if (na == 0 && tloader) wait_vmcnt<FT_PT - 2>();
    };
    load_inputs(0);
    asm volatile("" ::: "memory");
    if (tloader)
        for (int s = 0; s < FT_PT; ++s) load_trellis(s);
    asm volatile("" ::: "memory");
    load_inputs(1);
    if (tloader)
    {
        if (na == 2) wait_vmcnt<2 + FT_PT - 1>();
        else wait_vmcnt<1 + FT_PT - 1>();
    }
    lds_barrier();
    {
        const half4_t r0 = decode4<true>(tword[lhi], tword[llo], sh);
        const half4_t r1 = decode4<true>(tword[512 + lhi], tword[512 + llo], sh);
        *reinterpret_cast<half8_t*>(bdst) = half8_t{ r0[0], r0[1], r0[2], r0[3], r1[0], r1[1], r1[2], r1[3] };
    }
    const int nb16 = (rows + 15) >> 4;
    const int nvb = max(0, min(MBW, (nb16 - wm + 3) >> 2));
    auto main_loop = [&](auto part_tag) {
        constexpr bool PART = decltype(part_tag)::value;
        for (int s = 0; s < S; ++s)
        {
            wait_step();
            lds_barrier();
            if (tloader) load_trellis(s + FT_PT);
            const uint32_t toff = (uint32_t)__builtin_amdgcn_readfirstlane(((s + 1) % FT_TS) * T_SLOT);
            const uint8_t* thp = reinterpret_cast<const uint8_t*>(tword + lhi) + toff;
            const uint8_t* tlp = reinterpret_cast<const uint8_t*>(tword + llo) + toff;
            const uint32_t th0 = *reinterpret_cast<const uint32_t*>(thp), tl0 = *reinterpret_cast<const uint32_t*>(tlp);
            const uint32_t th1 = *reinterpret_cast<const uint32_t*>(thp + 2048);
            const uint32_t tl1 = *reinterpret_cast<const uint32_t*>(tlp + 2048);
            const uint8_t* as = Aring + (size_t)(s % FT_PA) * A_STAGE;
            const uint8_t* bs = bsrc + (size_t)(s & 1) * B_BUF;
            uint8_t* bd = bdst + (size_t)((s + 1) & 1) * B_BUF;
            half8_t B[4], A[MBW];
#pragma unroll
            for (int j = 0; j < 4; ++j) B[j] = *reinterpret_cast<const half8_t*>(bs + j * 1024);
#pragma unroll
            for (int i = 0; i < MBW; ++i)
                if (!PART || i < nvb) A[i] = *reinterpret_cast<const half8_t*>(as + aoff[i]);
            const half4_t d0 = decode4<true>(th0, tl0, sh);
#pragma unroll
            for (int i = 0; i < MBW; ++i)
            {
                if (!PART || i < nvb)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i], B[j], acc[i][j], 0, 0, 0);
                if (i == 0) load_inputs(s + FT_PA - 1);
                if (i == MBW / 2 - 1)
                {
                    const half4_t d1 = decode4<true>(th1, tl1, sh);
                    *reinterpret_cast<half8_t*>(bd) = half8_t{ d0[0], d0[1], d0[2], d0[3], d1[0], d1[1], d1[2], d1[3] };
                }
            }
            if constexpr (!PART)
            {
                __builtin_amdgcn_sched_group_barrier(0x0100, 4 + MBW + 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x0002, 8, 0);
#pragma unroll
                for (int k = 0; k < 4 * MBW; ++k)
                {
                    __builtin_amdgcn_sched_group_barrier(0x0008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x0002, 1, 0);
                }
            }
        }
    };
    if (nvb == MBW)
        main_loop(std::false_type{});
    else
        main_loop(std::true_type{});
    wait_vmcnt<0>();
    lds_barrier();

    uint16_t* C = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
    for (int i = 0; i < MBW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int c = (wn * 4 + j) * 16 + col, r = 16 * (4 * i + wm) + 4 * g;
            uint32_t* d = reinterpret_cast<uint32_t*>(C + (size_t)c * CS + r);
            d[0] = (uint32_t)f2h(acc[i][j][0]) | ((uint32_t)f2h(acc[i][j][1]) << 16);
            d[1] = (uint32_t)f2h(acc[i][j][2]) | ((uint32_t)f2h(acc[i][j][3]) << 16);
        }
    __syncthreads();
    const uint16_t* sc[3];
    fat_scales<MODE>(a, e, nu, sc);
    fat_tile_epilogue<MODE, CS, YH, NW>(a, C, rows, nu, grp, wave, lane, sc, a.route_at + pos0);
}

typedef float float16_t __attribute__((ext_vector_type(16)));

// k_mid's LDS: the four waves' rings (mid_depth steps of the trellis and the inputs) and, over them once they are done, the
// partial sums of one row group and its C tile. One array: with a second one the compiler gives their accesses alias
// scopes and then waits for every load to LDS (vmcnt 0) before each read.
constexpr int mid_depth(int rb) { return rb == 3 ? 2 : 3; }
constexpr int mid_slot(int rb) { return 2048 + rb * 2048; }
constexpr int MID_C_AT = 2 * 32 * 128 * 4;
constexpr int MID_RINGS = std::max({ 4 * mid_depth(1) * mid_slot(1), 4 * mid_depth(2) * mid_slot(2),
                                     4 * mid_depth(3) * mid_slot(3), MID_C_AT + FT_BN * (GRP_ROWS + 2) * 2 });
// what the epilogue needs from memory, loaded while the rings fill: scales [3][128], output rows, input sums [2]
constexpr int MID_SC_AT = MID_RINGS, MID_ROUTE_AT = MID_SC_AT + 3 * 256, MID_XS_AT = MID_ROUTE_AT + FT_MID * 4;
constexpr int MID_SMEM = MID_XS_AT + 2 * FT_MID * 4;
static_assert(2 * MID_SMEM <= 160 * 1024, "two workgroups (two waves per SIMD) share a CU's LDS");

// Tiles of up to FT_MID = 96 routes x 256 output columns, for experts (and remainders of experts) with too few routes to
// fill a 256-route tile. A workgroup is four waves: two column blocks of 128 (MODE 0: gate and up of one block, MODE
// 1: two blocks) x two halves of K, and no barrier until the epilogue, which adds the halves. A wave streams its trellis rows (768 bytes) and
// its inputs (a row group's step is one contiguous KB per operand) into a private LDS ring, and decodes each tile once,
// in registers, for all its routes: v_mfma_f32_32x32x16_f16 over 32 routes x 32 columns, whose k-half h of operand mm
// holds decode window 2 mm + h of both tile rows of the step, so the operand chunks are those of the row groups.
template <int MODE, int RB, bool EXACT, bool YH>
__device__ __forceinline__ void mid_tile(const FatArgs& a, uint8_t* smem, int rows, int pos0, int e, size_t grp, int nu,
                                         const ExpertRec* rp)
{
    constexpr int BM = RB * GRP_ROWS;
    constexpr int NA = MODE == 0 ? 2 : 1;
    constexpr int DEPTH = mid_depth(RB);
    constexpr int T_SLOT = 2048, SLOT = mid_slot(RB);
    constexpr int NL = 2 + 2 * RB;                                // loads of a step
    constexpr int CS = GRP_ROWS + 2;                              // C tile of one row group (fat_tile_epilogue)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = wave & 1, kh = wave >> 1;
    const int S = a.K / 64, step0 = kh * S;                       // steps of this wave's half of K (a.K / 32 is even)

    const uint32_t row_bytes = (uint32_t)(a.N / 16) * 96, wbytes = (uint32_t)(a.K / 16) * row_bytes;
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr((const void*)(uintptr_t)rp->w[MODE == 0 ? sub : 2]), (short)0, (int)wbytes, 0x00020000);
    const uint32_t wcol = MODE == 0 ? (uint32_t)nu * 768 : (uint32_t)(2 * nu + sub) * 768;
    const uint32_t gbytes = (uint32_t)NA * a.K * GRP_ROWS * 2;
    const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(a.xa + grp * (gbytes / 2)), (short)0, (int)((uint32_t)((rows + 31) / GRP_ROWS) * gbytes), 0x00020000);
    uint8_t* ring = smem + wave * (DEPTH * SLOT);
    // step s into a slot (past the end: the last step again, into a free slot): both trellis rows, 12 bytes per lane 16
    // apart, then the operands mm of each row group (one past the tile's routes reads zeros)
    auto load_step = [&](int s, int slot) {
        uint8_t* d = ring + slot * SLOT;
        s = step0 + min(s, S - 1);
        const uint32_t o = (uint32_t)(2 * s) * row_bytes + wcol;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, d, 12, (uint32_t)lane * 12, o, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, d + 1024, 12, (uint32_t)lane * 12, o + row_bytes, 0, 0);
        const uint32_t ao = (uint32_t)s * (NA * 2048) + (MODE == 0 ? (uint32_t)sub * 2048 : 0);
#pragma unroll
        for (int r = 0; r < RB; ++r)
        {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, d + T_SLOT + r * 2048, 16, (uint32_t)lane * 16, ao + r * gbytes, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, d + T_SLOT + r * 2048 + 1024, 16, (uint32_t)lane * 16 + 1024,
                                                     ao + r * gbytes, 0, 0);
        }
    };

    // decode: lane (n = lane & 15, ct = (lane >> 4) & 1, h = lane >> 5) decodes window 2 mm + h of column n of tile
    // 2 cp + ct
    const int n = lane & 15, h = lane >> 5;
    int llo[2], lhi[2];
    uint32_t sh[2];
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
    {
        const int i0 = 32 * (n & 7) + 8 * (2 * mm + h) + 4 * (n >> 3), eb = 3 * i0 + 11;
        const int blo = eb >> 5, bhi = (blo + 23) % 24;
        llo[mm] = 4 * (4 * (blo / 3) + blo % 3) + 128 * ((lane >> 4) & 1);
        lhi[mm] = 4 * (4 * (bhi / 3) + bhi % 3) + 128 * ((lane >> 4) & 1);
        sh[mm] = 31u - (uint32_t)(eb & 31);
    }

    float16_t acc[RB][4];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[r][c][v] = 0.0f;
    // trellis words and operands of half mm of the step in a slot
    uint32_t W[2][4][2][2];
    half8_t A[2][RB];
    auto read_half = [&](int slot, auto mm_tag) {
        constexpr int mm = decltype(mm_tag)::value;
        const uint8_t* t0 = ring + slot * SLOT;
#pragma unroll
        for (int cp = 0; cp < 4; ++cp)
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                W[mm][cp][t][0] = *reinterpret_cast<const uint32_t*>(t0 + lhi[mm] + cp * 256 + t * 1024);
                W[mm][cp][t][1] = *reinterpret_cast<const uint32_t*>(t0 + llo[mm] + cp * 256 + t * 1024);
            }
#pragma unroll
        for (int r = 0; r < RB; ++r)
            A[mm][r] = *reinterpret_cast<const half8_t*>(t0 + T_SLOT + r * 2048 + mm * 1024 + lane * 16);
    };
    auto compute_half = [&](auto mm_tag) {
        constexpr int mm = decltype(mm_tag)::value;
#pragma unroll
        for (int cp = 0; cp < 4; ++cp)
        {
            const half4_t b0 = decode4<EXACT>(W[mm][cp][0][0], W[mm][cp][0][1], sh[mm]);
            const half4_t b1 = decode4<EXACT>(W[mm][cp][1][0], W[mm][cp][1][1], sh[mm]);
            const half8_t B = { b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3] };
#pragma unroll
            for (int r = 0; r < RB; ++r)
                acc[r][cp] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[mm][r], B, acc[r][cp], 0, 0, 0);
        }
    };
    const std::integral_constant<int, 0> h0;
    const std::integral_constant<int, 1> h1;
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) load_step(j, j);
    {
        // (every thread's loads in one round trip with the rings')
        const int tid = threadIdx.x;
        const uint16_t* sc[3];
        fat_scales<MODE>(a, e, nu, sc);
        constexpr int NSC = MODE == 0 ? 3 : 2;
        uint32_t scw = 0;
        if (tid < NSC * 64) scw = reinterpret_cast<const uint32_t*>(tid < 64 ? sc[0] : tid < 128 ? sc[1] : sc[2])[tid & 63];
        int32_t ro = 0;
        if (MODE == 1 && tid < rows) ro = a.route_at[pos0 + tid];
        float xsum = 0.0f;
        const int xr = tid & 127, xm = tid >> 7;               // row, column block
        if (!EXACT && xr < rows)
            for (int b = 0; b < a.nxs; ++b)
                xsum += a.xs[(((grp + (xr >> 5)) * a.nxs + b) * NA + (MODE == 0 ? xm : 0)) * GRP_ROWS + (xr & 31)];
        if (tid < NSC * 64) reinterpret_cast<uint32_t*>(smem + MID_SC_AT)[tid] = scw;
        if (MODE == 1 && tid < rows) reinterpret_cast<int32_t*>(smem + MID_ROUTE_AT)[tid] = ro;
        if (!EXACT && xr < BM) reinterpret_cast<float*>(smem + MID_XS_AT)[xm * FT_MID + xr] = xsum * kbias_f();
    }
    wait_vmcnt<(DEPTH - 1) * NL>();
    constexpr bool PIPE = RB < 3;
    if constexpr (PIPE) read_half(0, h0);
    int slot = 0;
    for (int s = 0; s < S; ++s)
    {
        // the second half's reads run during the first half's decode, the next step's first reads during the second's
        if constexpr (PIPE) read_half(slot, h1);
        else read_half(slot, h0);
        compute_half(h0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!PIPE) read_half(slot, h1);
        // step s + 1 is complete once at most the loads of the steps after it are outstanding; this step's reads are
        // complete before its slot is filled again
        wait_vmcnt<(DEPTH - 2) * NL>();
        wait_lgkm0();
        load_step(s + DEPTH, slot);
        slot = slot + 1 == DEPTH ? 0 : slot + 1;
        if constexpr (PIPE) read_half(slot, h0);
        compute_half(h1);
        __builtin_amdgcn_sched_barrier(0);
    }
    wait_vmcnt<0>();
    __syncthreads();
    float4_t* red = reinterpret_cast<float4_t*>(smem) + sub * 1024 + lane;
    uint16_t* C = reinterpret_cast<uint16_t*>(smem + MID_C_AT);
    const float* xs_row = reinterpret_cast<const float*>(smem + MID_XS_AT) + sub * FT_MID;
    const uint16_t* sc0 = reinterpret_cast<const uint16_t*>(smem + MID_SC_AT);
    const uint16_t* const sc[3] = { sc0, sc0 + 128, sc0 + 256 };
    const int32_t* route = reinterpret_cast<const int32_t*>(smem + MID_ROUTE_AT);
    // one row group at a time: the second half's sums through LDS, then the C tile (lane (column lane & 31, h) of a 32 x
    // 32 block holds rows 8 (v >> 2) + 4 h + (v & 3); the affine decode's sums become KINV S + KBIAS (sum of the row's
    // inputs)), then the epilogue, 8 rows per wave
#pragma unroll
    for (int r = 0; r < RB; ++r)
    {
        if (r * GRP_ROWS >= rows) break;
        if (kh == 1)
#pragma unroll
            for (int cp = 0; cp < 4; ++cp)
#pragma unroll
                for (int v = 0; v < 16; v += 4)
                    red[(cp * 4 + v / 4) * 64] = float4_t{ acc[r][cp][v], acc[r][cp][v + 1], acc[r][cp][v + 2], acc[r][cp][v + 3] };
        __syncthreads();
        if (kh == 0)
#pragma unroll
            for (int v = 0; v < 16; v += 4)
            {
                const int rr = 2 * v + 4 * h;
                float4_t xs = { 0.f, 0.f, 0.f, 0.f };
                if constexpr (!EXACT) xs = *reinterpret_cast<const float4_t*>(&xs_row[r * GRP_ROWS + rr]);
#pragma unroll
                for (int cp = 0; cp < 4; ++cp)
                {
                    const float4_t o = red[(cp * 4 + v / 4) * 64];
                    uint32_t* d = reinterpret_cast<uint32_t*>(C + (size_t)(sub * 128 + cp * 32 + (lane & 31)) * CS + rr);
                    float y[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                    {
                        const float sum = acc[r][cp][v + i] + o[i];
                        y[i] = EXACT ? sum : fmaf(kinv_f(), sum, xs[i]);
                    }
                    d[0] = (uint32_t)f2h(y[0]) | ((uint32_t)f2h(y[1]) << 16);
                    d[1] = (uint32_t)f2h(y[2]) | ((uint32_t)f2h(y[3]) << 16);
                }
            }
        __syncthreads();
        fat_tile_epilogue<MODE, CS, YH, 4, !EXACT>(a, C, min(rows - r * GRP_ROWS, GRP_ROWS), nu, grp + r, wave, lane, sc,
                                                   route + r * GRP_ROWS);
    }
}

template <int MODE, bool EXACT, bool YH = false>
__global__ __launch_bounds__(256, 2) void k_mid(FatArgs a)
{
    __shared__ __align__(16) uint8_t smem[MID_SMEM];
    // workgroup b runs on XCD b % 8: tile t's column units go to XCD t % 8 one after another (they share the inputs), so the
    // XCDs get the same mix of long and short tiles
    const int b = blockIdx.x >> 3, mt = b / a.nunits * 8 + (int)(blockIdx.x & 7), nu = b % a.nunits;
    if (mt >= a.ntiles[0]) return;
    const FatTile* tp = a.tiles + mt;
    const ExpertRec* rp = a.rec + tp->ai;
    const int row0 = tp->row0;
    const int rows = __builtin_amdgcn_readfirstlane(min(FT_MID, rp->cnt - row0));
    const int pos0 = __builtin_amdgcn_readfirstlane(rp->first + row0);
    const int e = __builtin_amdgcn_readfirstlane(rp->e);
    const size_t grp = (size_t)__builtin_amdgcn_readfirstlane(tp->group);
    if (rows > 2 * GRP_ROWS)
        mid_tile<MODE, 3, EXACT, YH>(a, smem, rows, pos0, e, grp, nu, rp);
    else if (rows > GRP_ROWS)
        mid_tile<MODE, 2, EXACT, YH>(a, smem, rows, pos0, e, grp, nu, rp);
    else
        mid_tile<MODE, 1, EXACT, YH>(a, smem, rows, pos0, e, grp, nu, rp);
}

// (skip: where not 0, the decode path has computed the call)
// Weighted combine of the fat routes: out[t] = (accumulate ? out[t] : 0) + sum_j w_j y_j over the routes j of
// token t whose expert has more than cap routes, fp32 fma in ascending j (with cap 0 this is mm_combine). The
// per-route rows y_j are fp16 (the down GEMM writes them so: its output transform rounds every value to fp16).
__global__ __launch_bounds__(256) void k_fat_combine(float* __restrict__ out, const uint16_t* __restrict__ Y,
                                                     const int64_t* __restrict__ ids, const float* __restrict__ w,
                                                     const int32_t* __restrict__ counts, int T, int k, int H, int E,
                                                     int cap, int accumulate, const int32_t* skip)
{
    if (skip && skip[0] != 0) return;
    const int t = blockIdx.y;
    const int h = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (t >= T || h >= H) return;
    float4 acc = accumulate ? *reinterpret_cast<const float4*>(out + (size_t)t * H + h) : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j = 0; j < k; ++j)
    {
        const int s = t * k + j;
        const int64_t e = ids[s];
        if (e < 0 || e >= E || counts[e] <= cap) continue;
        const float wj = w[s];
        const uint2 yb = *reinterpret_cast<const uint2*>(Y + (size_t)s * H + h);
        const float4 y = make_float4(h2f((uint16_t)(yb.x & 0xffffu)), h2f((uint16_t)(yb.x >> 16)),
                                     h2f((uint16_t)(yb.y & 0xffffu)), h2f((uint16_t)(yb.y >> 16)));
        acc.x = fmaf(wj, y.x, acc.x);
        acc.y = fmaf(wj, y.y, acc.y);
        acc.z = fmaf(wj, y.z, acc.z);
        acc.w = fmaf(wj, y.w, acc.w);
    }
    *reinterpret_cast<float4*>(out + (size_t)t * H + h) = acc;
}

// ------------------------------------------------------------------------------- sorted-route form
// The reference's fat entry takes the routes already sorted by expert (token_sorted, weight_sorted and per-expert
// counts, patches/vllm-exl3-host-dma.patch:182-201). Selection, token lists and the combine of that form:

// One block: counts (effective) = counts_in[e] for experts with more than cap routes that are not skipped and whose
// range lies within the n positions, else 0; offsets = exclusive sums of counts_in (clamped to n), offsets[E] =
// the routed positions, offsets[E + 1] = n; active = the selected experts in ascending id, nactive their number.
__global__ __launch_bounds__(FT_PLAN_MAX) void k_fatb_setup(const int32_t* counts_in, const uint8_t* skip, int E, int n,
                                                           int cap, int32_t* counts, int32_t* offsets, int32_t* active,
                                                           int32_t* nactive)
{
    __shared__ int s_w[2][FT_PLAN_MAX / 64];
    const int e = threadIdx.x, lane = e & 63, wave = e >> 6;
    const int c = e < E ? max(counts_in[e], 0) : 0;
    const int ic = wave_incl_scan(c);
    if (lane == 63) s_w[0][wave] = ic;
    __syncthreads();
    int base = 0, total = 0;
    for (int w = 0; w < FT_PLAN_MAX / 64; ++w)
    {
        if (w < wave) base += s_w[0][w];
        total += s_w[0][w];
    }
    const long long off = (long long)base + ic - c;
    const bool sel = e < E && c > cap && !(skip && skip[e]) && off + c <= n;
    const int f = wave_incl_scan(sel ? 1 : 0);
    if (lane == 63) s_w[1][wave] = f;
    __syncthreads();
    int fb = 0, nf = 0;
    for (int w = 0; w < FT_PLAN_MAX / 64; ++w)
    {
        if (w < wave) fb += s_w[1][w];
        nf += s_w[1][w];
    }
    if (e < E)
    {
        offsets[e] = (int)min(off, (long long)n);
        counts[e] = sel ? c : 0;
        if (sel) active[fb + f - 1] = e;
    }
    if (e == 0)
    {
        const int routed = min(total, n);
        offsets[E] = routed;
        offsets[E + 1] = n;
        counts[E] = n - routed;
        nactive[0] = nf;
    }
}

__device__ __forceinline__ int fatb_expert(const int32_t* offsets, int E, int pos)
{
    int lo = 0, hi = E;
    while (hi - lo > 1)
    {
        const int mid = (lo + hi) >> 1;
        if (offsets[mid] <= pos) lo = mid; else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(256) void k_fill_i32(int32_t* p, int n, int v)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

// Per position of a selected expert: FILL = 0 counts the position's token (tcount[t]++) and writes order[pos] =
// pos (the grouped GEMM's output row); FILL = 1 appends the position to its token's list (any order within a
// token: the combine visits a list in ascending position).
template <int FILL>
__global__ __launch_bounds__(256) void k_fatb_tokens(const int64_t* token_sorted, const int32_t* counts,
                                                     const int32_t* offsets, int32_t* order, int32_t* tcount,
                                                     const int32_t* toff, int32_t* tpos, int T, int E, int n)
{
    for (int pos = blockIdx.x * blockDim.x + threadIdx.x; pos < n; pos += gridDim.x * blockDim.x)
    {
        if (FILL == 0) order[pos] = pos;
        if (pos >= offsets[E]) continue;
        const int e = fatb_expert(offsets, E, pos);
        if (counts[e] <= 0 || pos >= offsets[e] + counts[e]) continue;
        const int64_t t = token_sorted[pos];
        if (t < 0 || t >= T) continue;
        if (FILL == 0)
            atomicAdd(&tcount[t], 1);
        else
            tpos[toff[t] + atomicAdd(&tcount[t], 1)] = pos;
    }
}

// One block: toff[0 .. T] = exclusive sums of tcount[0 .. T-1] (each thread sums a contiguous chunk).
__global__ __launch_bounds__(1024) void k_scan_i32(const int32_t* tcount, int32_t* toff, int T)
{
    __shared__ int s_w[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (T + 1023) / 1024, i0 = min(tid * per, T), i1 = min(i0 + per, T);
    int sum = 0;
    for (int i = i0; i < i1; ++i) sum += tcount[i];
    const int inc = wave_incl_scan(sum);
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    int base = 0, total = 0;
    for (int w = 0; w < 16; ++w)
    {
        if (w < wave) base += s_w[w];
        total += s_w[w];
    }
    int run = base + inc - sum;
    for (int i = i0; i < i1; ++i)
    {
        toff[i] = run;
        run += tcount[i];
    }
    if (tid == 0) toff[T] = total;
}

// out[t] += sum over the token's selected positions p, in ascending p, of fp32(weight_sorted[p]) * Y[p] (fp32 fma).
__global__ __launch_bounds__(256) void k_fatb_combine(float* __restrict__ out, const uint16_t* __restrict__ Y,
                                                      const uint16_t* __restrict__ wsorted, const int32_t* __restrict__ toff,
                                                      const int32_t* __restrict__ tpos, int T, int H)
{
    const int t = blockIdx.y;
    const int h = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (t >= T || h >= H) return;
    const int b = toff[t], m = toff[t + 1] - b;
    if (m <= 0) return;
    float4 acc = *reinterpret_cast<const float4*>(out + (size_t)t * H + h);
    int prev = -1;
    for (int i = 0; i < m; ++i)
    {
        int p = 0x7fffffff;
        for (int j = 0; j < m; ++j)
        {
            const int q = tpos[b + j];
            if (q > prev && q < p) p = q;
        }
        prev = p;
        const float wj = h2f(wsorted[p]);
        const uint2 yb = *reinterpret_cast<const uint2*>(Y + (size_t)p * H + h);
        const float4 y = make_float4(h2f((uint16_t)(yb.x & 0xffffu)), h2f((uint16_t)(yb.x >> 16)),
                                     h2f((uint16_t)(yb.y & 0xffffu)), h2f((uint16_t)(yb.y >> 16)));
        acc.x = fmaf(wj, y.x, acc.x);
        acc.y = fmaf(wj, y.y, acc.y);
        acc.z = fmaf(wj, y.z, acc.z);
        acc.w = fmaf(wj, y.w, acc.w);
    }
    *reinterpret_cast<float4*>(out + (size_t)t * H + h) = acc;
}

// ------------------------------------------------------------------------------------------------- host

struct FatWs
{
    int32_t* counts;      // [E + 1]   permutation
    int32_t* offsets;     // [E + 2]
    int32_t* order;       // [n]
    int32_t* active;      // [E]
    int32_t* nactive;     // [1]
    void* pws;            // permutation workspace
    size_t pws_bytes;
    ExpertRec* rec;       // [min(n, E)]
    FatTile* big;         // 256-route tiles
    FatTile* small;       // 128-route tiles
    FatTile* mid;         // FT_MID-route tiles
    int2* groups;         // row groups: record, first row
    int32_t* totals;      // [4] entries of the lists
    int max_big, max_small, max_mid, max_groups;
    uint16_t* xa;         // [max_groups][H / 32][2][GRP_HALVES]
    uint16_t* xd;         // [max_groups][I / 32][GRP_HALVES]
    float* xs;            // [max_groups][prep slices][2][GRP_ROWS] input sums
    float* xds;           // [max_groups][I / 128][GRP_ROWS] down-input sums
    int nxs;
    float* Y;             // [n][H]
    size_t plan_bytes;    // up to xa: permutation, records and lists
    size_t bytes;
};

static FatWs fat_carve(void* base, int n, int E, int H, int I)
{
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t na = (size_t)(n < E ? n : E);
    const size_t pwsb = mm_permute_workspace(n, E);
    // an expert of c routes has at most c / min_rest 256-route tiles, one 128-route tile of more than FT_MID routes, c / FT_MID
    // + 1 others and c / GRP_ROWS + 1 row groups
    FatWs w;
    w.max_big = n / FT_REST_LARGE;
    w.max_small = (int)na;
    w.max_mid = n / FT_MID + (int)na;
    w.max_groups = n / GRP_ROWS + (int)na;
    const size_t ng = (size_t)w.max_groups;
    w.nxs = (H / 128 + PREP_BLOCKS - 1) / PREP_BLOCKS;
    constexpr int NS = 17;
    const size_t sizes[NS] = { al((size_t)(E + 1) * 4), al((size_t)(E + 2) * 4), al((size_t)n * 4), al((size_t)E * 4),
                               al(4), al(pwsb), al(na * sizeof(ExpertRec)), al(w.max_big * sizeof(FatTile)),
                               al(w.max_small * sizeof(FatTile)),
                               al(w.max_mid * sizeof(FatTile)), al(ng * sizeof(int2)), al(16),
                               al(ng * GRP_ROWS * 2 * H * 2), al(ng * GRP_ROWS * I * 2), al((size_t)n * H * 4),
                               al(ng * w.nxs * 2 * GRP_ROWS * 4), al(ng * (I / 128) * GRP_ROWS * 4) };
    char* p = static_cast<char*>(base);
    char* at[NS];
    size_t off = 0;
    for (int i = 0; i < NS; ++i)
    {
        at[i] = p ? p + off : nullptr;
        off += sizes[i];
    }
    w.counts = (int32_t*)at[0]; w.offsets = (int32_t*)at[1]; w.order = (int32_t*)at[2]; w.active = (int32_t*)at[3];
    w.nactive = (int32_t*)at[4]; w.pws = at[5]; w.pws_bytes = pwsb; w.rec = (ExpertRec*)at[6];
    w.big = (FatTile*)at[7]; w.small = (FatTile*)at[8]; w.mid = (FatTile*)at[9]; w.groups = (int2*)at[10];
    w.totals = (int32_t*)at[11]; w.xa = (uint16_t*)at[12]; w.xd = (uint16_t*)at[13]; w.Y = (float*)at[14];
    w.xs = (float*)at[15]; w.xds = (float*)at[16];
    w.plan_bytes = 0;
    for (int i = 0; i < 12; ++i) w.plan_bytes += sizes[i];
    w.bytes = off;
    return w;
}

static int fat_check(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* ids, void* ws,
                     size_t ws_bytes, const char* who, bool check_ws = true)
{
    MM_CHECK_ARG(L && L->gate_ptr && L->up_ptr && L->down_ptr && L->suh13 && L->svh13 && L->suh2 && L->svh2,
                 "%s: incomplete layer", who);
    MM_CHECK_ARG(L->E > 0 && L->E <= FT_PLAN_MAX && L->H % 256 == 0 && L->I % 128 == 0 && L->H > 0 && L->I > 0,
                 "%s: need 0 < E <= %d, H a multiple of 256 and I of 128", who, FT_PLAN_MAX);
    MM_CHECK_ARG((size_t)(L->H / 16) * (L->I / 16) * 96 < ((size_t)1 << 31), "%s: matrix larger than 2 GiB", who);
    MM_CHECK_ARG((size_t)FT_BIG * 2 * L->H * 2 < ((size_t)1 << 30), "%s: H too large", who);
    MM_CHECK_ARG(x && ids, "%s: null pointer", who);
    MM_CHECK_ARG(x_dtype == MM_DTYPE_F16 || x_dtype == MM_DTYPE_BF16 || x_dtype == MM_DTYPE_F32,
                 "%s: x_dtype must be MM_DTYPE_F16, MM_DTYPE_BF16 or MM_DTYPE_F32", who);
    MM_CHECK_ARG(T > 0 && topk > 0 && (size_t)T * topk < ((size_t)1 << 30), "%s: bad T/topk", who);
    if (!check_ws) return MM_OK;
    const size_t need = fat_carve(nullptr, T * topk, L->E, L->H, L->I).bytes;
    MM_CHECK_ARG(ws && ws_bytes >= need, "%s: workspace too small (%zu < %zu)", who, ws_bytes, need);
    return MM_OK;
}

// How a call's experts are taken: the fused call by the layer's codebook evaluation, the others with fp16-rounded weights.
struct FatMode
{
    bool exact;
    TileRule rule;
};
static FatMode fat_mode(const mm_layer_t* L, int n, bool fused)
{
    const int units = L->I / 128, tiles = (FT_BIG_WORK + units - 1) / units, none = FT_SMALL + 1;
    if (fused) return { (L->flags & MM_LAYER_EXACT) != 0, TileRule{ tiles, 0, FT_REST, none, 0 } };
    if (n >= FT_LARGE && n / 200 >= L->E) return { true, TileRule{ 0, 0, FT_REST_LARGE, FT_MID + 1, tiles / 2 } };
    return { true, TileRule{ 0, FT_BIG_ROWS, FT_REST, none, 0 } };
}

// Expert records, row groups and tile lists of the sorted positions in ws (counts, offsets, active, nactive filled).
// layer_counts: the routes of every expert of the layer, whether the call computes it or not.
static void fat_plan(const mm_layer_t* L, int n, int cap, const FatWs& ws, hipStream_t s, const FatMode& mode,
                     const int32_t* layer_counts, int32_t* choice)
{
    const int E = L->E, na = n < E ? n : E;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(1), dim3(FT_PLAN_MAX), 0, s, ws.counts, ws.offsets, ws.active, ws.nactive, L->gate_ptr,
                           L->up_ptr, L->down_ptr, ws.rec, ws.big, ws.small, ws.mid, ws.groups, ws.totals, na, cap, mode.rule,
                           layer_counts, choice, E, n);
    };
    if (choice) launch(k_fat_plan<true>);
    else launch(k_fat_plan<false>);
}

// Input transform and both GEMMs of a plan: Y rows of every position of an active expert with more than cap routes.
// token_sorted: the positions' tokens, or null (order[pos] / topk).
static int fat_gemms(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* token_sorted, int n,
                     const FatWs& ws, hipStream_t s, bool yh, const FatMode& mode)
{
    const bool exact = mode.exact;
    auto prep = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)ws.max_groups, (unsigned)ws.nxs), dim3(512), 0, s, x, x_dtype, ws.order,
                           token_sorted, ws.rec, ws.groups, ws.totals + 2, L->suh13, ws.xa, ws.xs, topk, T, L->H);
    };
    if (exact) prep(k_fat_prep<false>);
    else prep(k_fat_prep<true>);
    // tiles of 128 and of 256 routes the call can have
    const int max_small = mode.rule.min_small <= FT_SMALL ? ws.max_small : 0;
    const int most_big = n / mode.rule.min_rest;
    const int max_big = most_big >= mode.rule.min_tiles && n >= mode.rule.min_rows ? most_big : 0;
    auto grid = [](int tiles, int units) { return dim3((unsigned)(((size_t)tiles * units + 7) & ~(size_t)7)); };    // >= 8 per_xcd
    auto mid_grid = [](int tiles, int units) { return dim3((unsigned)(((size_t)tiles + 7) / 8 * 8 * units)); };
    FatArgs g{ ws.rec, ws.big, ws.totals, ws.xa, L->svh13, L->suh2, L->svh2, ws.order, ws.xd, ws.Y,
               ws.xs, ws.xds, L->H, L->I, L->H, L->I, L->I / 128, ws.nxs, L->I / 128, L->limit };
    FatArgs gm = g;
    gm.tiles = ws.mid;
    gm.ntiles = ws.totals + 1;
    FatArgs gs = g;
    gs.tiles = ws.small;
    gs.ntiles = ws.totals + 3;
    FatArgs d = g;
    d.xa = ws.xd; d.K = L->I; d.N = L->H; d.nunits = L->H / 256;
    d.xs = ws.xds; d.nxs = g.nxds;
    FatArgs dm = d;
    dm.tiles = ws.mid;
    dm.ntiles = ws.totals + 1;
    FatArgs ds = d;
    ds.tiles = ws.small;
    ds.ntiles = ws.totals + 3;
    // gate/up: 256-route tiles on the 8-wave kernel, down on the 16-wave kernel (same bits; measured on the 16k layer:
    // gate/up equal, down 2.76-2.85 against 2.92-2.94 ms)
    if (max_big > 0) hipLaunchKernelGGL(k_fat, grid(max_big, g.nunits), dim3(FT_THREADS), 0, s, g);
    if (max_small > 0) hipLaunchKernelGGL((k_fat16<0, FT_SMALL / 64>), grid(max_small, g.nunits), dim3(FT16_THREADS), 0, s, gs);
    if (exact) hipLaunchKernelGGL((k_mid<0, true>), mid_grid(ws.max_mid, g.nunits), dim3(256), 0, s, gm);
    else hipLaunchKernelGGL((k_mid<0, false>), mid_grid(ws.max_mid, g.nunits), dim3(256), 0, s, gm);
    if (yh)
    {
        if (max_big > 0)
            hipLaunchKernelGGL((k_fat16<1, FT_BIG / 64, true>), grid(max_big, d.nunits), dim3(FT16_THREADS), 0, s, d);
        if (max_small > 0)
            hipLaunchKernelGGL((k_fat16<1, FT_SMALL / 64, true>), grid(max_small, d.nunits), dim3(FT16_THREADS), 0, s, ds);
        if (exact) hipLaunchKernelGGL((k_mid<1, true, true>), mid_grid(ws.max_mid, d.nunits), dim3(256), 0, s, dm);
        else hipLaunchKernelGGL((k_mid<1, false, true>), mid_grid(ws.max_mid, d.nunits), dim3(256), 0, s, dm);
    }
    else
    {
        if (max_big > 0)
            hipLaunchKernelGGL((k_fat16<1, FT_BIG / 64>), grid(max_big, d.nunits), dim3(FT16_THREADS), 0, s, d);
        if (max_small > 0)
            hipLaunchKernelGGL((k_fat16<1, FT_SMALL / 64>), grid(max_small, d.nunits), dim3(FT16_THREADS), 0, s, ds);
        if (exact) hipLaunchKernelGGL((k_mid<1, true>), mid_grid(ws.max_mid, d.nunits), dim3(256), 0, s, dm);
        else hipLaunchKernelGGL((k_mid<1, false>), mid_grid(ws.max_mid, d.nunits), dim3(256), 0, s, dm);
    }
    return check_launch("fat path");
}

// Permutation, plan, input transform and both GEMMs: Y rows of every route whose expert has more than cap routes.
static int fat_run(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* ids, int cap,
                   const FatWs& ws, hipStream_t s, bool yh, bool fused)
{
    const int n = T * topk, E = L->E;
    int rc = permute_launch(ids, nullptr, n, topk, E, ws.counts, ws.offsets, ws.order, nullptr, nullptr, nullptr,
                            ws.active, ws.nactive, ws.pws, ws.pws_bytes, s);
    if (rc) return rc;
    const FatMode mode = fat_mode(L, n, fused);
    fat_plan(L, n, cap, ws, s, mode, ws.counts, nullptr);
    return fat_gemms(L, x, x_dtype, T, topk, nullptr, n, ws, s, yh, mode);
}

static int fat_combine(const mm_layer_t* L, int T, int topk, const int64_t* ids, const float* w, int cap, int accumulate,
                       float* out, const FatWs& ws, hipStream_t s, const int32_t* skip)
{
    const dim3 grid((unsigned)((L->H / 4 + 255) / 256), (unsigned)T);
    hipLaunchKernelGGL(k_fat_combine, grid, dim3(256), 0, s, out, reinterpret_cast<const uint16_t*>(ws.Y), ids, w,
                       ws.counts, T, topk, L->H, L->E, cap, accumulate, skip);
    return check_launch("fat layer");
}

// fat_run and the weighted combine of its rows.
static int fat_layer(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* ids, const float* w,
                     int cap, int accumulate, float* out, const FatWs& ws, hipStream_t s, bool fused)
{
    const int r = fat_run(L, x, x_dtype, T, topk, ids, cap, ws, s, true, fused);
    return r ? r : fat_combine(L, T, topk, ids, w, cap, accumulate, out, ws, s, nullptr);
}

// Workspace of the sorted-route form: the fat sections for n positions, then the token lists.
struct FatbWs
{
    FatWs f;
    int32_t* tcount;     // [T]
    int32_t* toff;       // [T + 1]
    int32_t* tpos;       // [n]
    size_t bytes;
};

static FatbWs fatb_carve(void* base, int n, int T, int E, int H, int I)
{
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    FatbWs w;
    w.f = fat_carve(base, n, E, H, I);
    char* p = base ? static_cast<char*>(base) + w.f.bytes : nullptr;
    const size_t s0 = al((size_t)T * 4), s1 = al((size_t)(T + 1) * 4), s2 = al((size_t)n * 4);
    w.tcount = (int32_t*)p;
    w.toff = p ? (int32_t*)(p + s0) : nullptr;
    w.tpos = p ? (int32_t*)(p + s0 + s1) : nullptr;
    w.bytes = w.f.bytes + s0 + s1 + s2;
    return w;
}

// ------------------------------------------------------------------------------------ the fused-MoE call

// A call runs as a whole on one path. The decode path cuts the experts' rows into equal runs over the whole GPU, but decodes
// an expert once per 16 of its routes (a record); k_mid decodes a tile as fast for one route as for 32 and takes up to 96, but
// is slower per tile and needs many to fill the GPU, and its call has more launches. Whole calls, us on the decode path / on the
// grouped GEMM, H 4096, I 2048, n routes over E experts, routing uniform (u), Zipf (z) or on 8 experts (8):
//   E 8:   n 256 104 / 133 u, 113 / 155 z; 512 175 / 163, 168 / 169; 1,024 281 / 172, 289 / 174
//   E 16:  n 256 116 / 119 u, 123 / 138 z; 400 152 / 135, 146 / 164; 1,024 287 / 175, 288 / 187
//   E 64:  n 600 276 / 304 u, 316 / 313 z; 768 290 / 308, 345 / 326; 1,020 376 / 309, 408 / 361
//   E 128: n 800 470 / 535 u, 488 / 518 z; 1,024 488 / 532, 539 / 531; 1,600 586 / 552, 679 / 574
//   E 256: n 1,024 861 / 957 u, 731 / 763 z; 2,048 932 / 993, 1,043 / 946; 3,200 1,104 / 1,002, 1,341 / 1,054
//   E 384: n 1,024 1,141 / 1,326 u, 879 / 907 z, 249 / 174 8; 2,048 1,295 / 1,414, 1,252 / 1,146, 475 / 225
//   H 2048, I 1024, E 64: n 800 109 / 119 u, 118 / 129 z; 1,024 134 / 121, 138 / 146.  H 1024, I 512, E 32: n 512 52 / 63 u
// Both paths cost an expert's decode per record or tile, and the grouped GEMM about 40 us more in launches, which is 220
// routes of the decode path at H 4096, I 2048. So up to GV_ROUTE_MAX routes the decode path (routed in-kernel) takes 10 routes
// per expert and those, at least 384; what the host cannot see is left there: tokens that agree on a few of many experts. Above, the permutation is needed in any case, and while experts
// get few routes (7 each on average; 9 to 1,280 routes) the plan kernel chooses on the device by records and tiles: decode path
// 40 + 3.05 records + n / 33 us, grouped GEMM 80 + 3.45 tiles us, within 5 % of the above. The launches of the path not taken
// find no work (25-30 us in all), so calls of small layers, in the end faster than that, are not given the choice (E H I below
// 2^30: 512 experts, H 2048, I 512, 2,500 routes take 290 us on the grouped GEMM and 330 chosen). With more routes the experts
// are busy enough for the grouped GEMM.
enum class FusedPath { DECODE, CHOICE, GEMM };
constexpr int64_t FUSED_LAUNCHES = (int64_t)220 * 4096 * 2048;
static int fused_most_decode(int E, int H, int I)
{
    return (int)std::min<int64_t>(GV_ROUTE_MAX, std::max<int64_t>(384, 10 * E + FUSED_LAUNCHES / ((int64_t)H * I)));
}
static int fused_most_choice(int E, int H, int I)
{
    return (int64_t)E * H * I >= (int64_t)1 << 30 ? std::min(9 * E, std::max(7 * E, 1280)) : 0;
}
static FusedPath fused_path(int n, int E, int H, int I)
{
    if (n <= GV_ROUTE_MAX) return n <= fused_most_decode(E, H, I) ? FusedPath::DECODE : FusedPath::GEMM;
    return n <= fused_most_choice(E, H, I) && decode_fits(n, E, H, I) ? FusedPath::CHOICE : FusedPath::GEMM;
}

// Workspace of a call that either path may take: the grouped GEMM's, with the decode workspace over its inputs and rows (one of
// the two is used, and the decode path's launches come first), then the choice.
struct FusedWs
{
    FatWs f;
    void* dws;
    size_t dws_bytes;
    int32_t* choice;      // [2]
    size_t bytes;
};

static FusedWs fused_carve(void* base, int n, int E, int H, int I, size_t decode_bytes)
{
    FusedWs w;
    w.f = fat_carve(base, n, E, H, I);
    w.dws_bytes = decode_bytes;
    const size_t most = std::max(w.f.bytes, w.f.plan_bytes + w.dws_bytes);      // multiples of 256
    char* p = static_cast<char*>(base);
    w.dws = p ? p + w.f.plan_bytes : nullptr;
    w.choice = p ? (int32_t*)(p + most) : nullptr;
    w.bytes = most + 256;
    return w;
}

// Bytes a call of n routes needs.
static size_t fused_bytes(int n, int E, int H, int I)
{
    switch (fused_path(n, E, H, I))
    {
    case FusedPath::DECODE: return mm_gemv_workspace(n, E, H, I);
    case FusedPath::CHOICE: return fused_carve(nullptr, n, E, H, I, mm_gemv_workspace(n, E, H, I)).bytes;
    default: return fat_carve(nullptr, n, E, H, I).bytes;
    }
}

}  // namespace mm

using namespace mm;

extern "C" {

size_t mm_fused_moe_workspace(int T, int topk, int E, int H, int I, int cap)
{
    if (T <= 0 || topk <= 0 || E <= 0 || H <= 0 || I <= 0 || cap < 0) return 0;
    const int n = T * topk;
    // enough for every smaller call too, whichever path it takes
    size_t bytes = decode_workspace_upto(std::min(n, fused_most_decode(E, H, I)), E, H, I);
    const int choice = std::min(n, fused_most_choice(E, H, I));
    if (choice > GV_ROUTE_MAX)
        bytes = std::max(bytes, fused_carve(nullptr, choice, E, H, I, decode_workspace_upto(choice, E, H, I)).bytes);
    return n > fused_most_decode(E, H, I) ? std::max(bytes, fat_carve(nullptr, n, E, H, I).bytes) : bytes;
}

int mm_fused_moe(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* ids, const float* w,
                 int cap, float* out, void* workspace, size_t workspace_bytes, mm_stream_t stream)
{
    const int rc = fat_check(L, x, x_dtype, T, topk, ids, workspace, 0, "mm_fused_moe", false);
    if (rc) return rc;
    MM_CHECK_ARG(w && out && cap >= 1, "mm_fused_moe: null pointer or cap < 1");
    MM_CHECK_ARG(topk <= 16, "mm_fused_moe: topk must be at most 16");
    const int n = T * topk, E = L->E;
    const size_t need = fused_bytes(n, E, L->H, L->I);
    MM_CHECK_ARG(workspace && workspace_bytes >= need, "mm_fused_moe: workspace too small (%zu < %zu)", workspace_bytes,
                 need);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const FusedPath path = fused_path(n, E, L->H, L->I);
    if (path == FusedPath::DECODE)
        return moe_decode_launch(L, x, x_dtype, 0, T, topk, ids, w, n, out, workspace, workspace_bytes, stream,
                                 "mm_fused_moe");
    if (path == FusedPath::GEMM)
        return fat_layer(L, x, x_dtype, T, topk, ids, w, 0, 0, out, fat_carve(workspace, n, E, L->H, L->I), s, true);
    const FusedWs ws = fused_carve(workspace, n, E, L->H, L->I, mm_gemv_workspace(n, E, L->H, L->I));
    int r = permute_launch(ids, nullptr, n, topk, E, ws.f.counts, ws.f.offsets, ws.f.order, nullptr, nullptr, nullptr,
                           ws.f.active, ws.f.nactive, ws.f.pws, ws.f.pws_bytes, s);
    if (r) return r;
    const FatMode mode = fat_mode(L, n, true);
    fat_plan(L, n, 0, ws.f, s, mode, ws.f.counts, ws.choice);
    // the decode path's launches first: the grouped GEMM's inputs lie over their workspace
    r = moe_decode_launch(L, x, x_dtype, 0, T, topk, ids, w, n, out, ws.dws, ws.dws_bytes, stream, "mm_fused_moe",
                          ws.f.offsets, ws.f.order, ws.f.active, ws.choice, ws.choice + 1);
    if (r) return r;
    r = fat_gemms(L, x, x_dtype, T, topk, nullptr, n, ws.f, s, true, mode);
    return r ? r : fat_combine(L, T, topk, ids, w, 0, 0, out, ws.f, s, ws.choice + 1);
}

size_t mm_prefill_workspace(int n, int E, int H, int I)
{
    if (n <= 0 || E <= 0 || H <= 0 || I <= 0) return 0;
    return fat_carve(nullptr, n, E, H, I).bytes;
}

int mm_grouped_gemm(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* ids, int cap,
                    float* Y, void* workspace, size_t workspace_bytes, mm_stream_t stream)
{
    const int rc = fat_check(L, x, x_dtype, T, topk, ids, workspace, workspace_bytes, "mm_grouped_gemm");
    if (rc) return rc;
    MM_CHECK_ARG(Y && cap >= 0, "mm_grouped_gemm: null Y or negative cap");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    FatWs ws = fat_carve(workspace, T * topk, L->E, L->H, L->I);
    ws.Y = Y;
    return fat_run(L, x, x_dtype, T, topk, ids, cap, ws, s, false, false);
}

int mm_moe_prefill(const mm_layer_t* L, const void* x, int x_dtype, int T, int topk, const int64_t* ids, const float* w,
                   int cap, int accumulate, float* out, void* workspace, size_t workspace_bytes, mm_stream_t stream)
{
    const int rc = fat_check(L, x, x_dtype, T, topk, ids, workspace, workspace_bytes, "mm_moe_prefill");
    if (rc) return rc;
    MM_CHECK_ARG(w && out && cap >= 0, "mm_moe_prefill: null pointer or negative cap");
    return fat_layer(L, x, x_dtype, T, topk, ids, w, cap, accumulate, out, fat_carve(workspace, T * topk, L->E, L->H, L->I),
                     reinterpret_cast<hipStream_t>(stream), false);
}

size_t mm_fat_batched_workspace(int n, int T, int E, int H, int I)
{
    if (n <= 0 || T <= 0 || E <= 0 || H <= 0 || I <= 0) return 0;
    return fatb_carve(nullptr, n, T, E, H, I).bytes;
}

int mm_fat_batched(const mm_layer_t* L, const void* x, int x_dtype, int T, int n, const int64_t* token_sorted,
                   const uint16_t* weight_sorted, const int32_t* counts, const uint8_t* skip, int cap, float* out,
                   void* workspace, size_t workspace_bytes, mm_stream_t stream)
{
    MM_CHECK_ARG(n > 0, "mm_fat_batched: need n > 0 sorted positions");
    MM_CHECK_ARG(L && L->gate_ptr && L->up_ptr && L->down_ptr && L->suh13 && L->svh13 && L->suh2 && L->svh2,
                 "mm_fat_batched: incomplete layer");
    MM_CHECK_ARG(L->E > 0 && L->E <= FT_PLAN_MAX && L->H % 256 == 0 && L->I % 128 == 0 && L->H > 0 && L->I > 0,
                 "mm_fat_batched: need 0 < E <= %d, H a multiple of 256 and I of 128", FT_PLAN_MAX);
    MM_CHECK_ARG((size_t)(L->H / 16) * (L->I / 16) * 96 < ((size_t)1 << 31), "mm_fat_batched: matrix larger than 2 GiB");
    MM_CHECK_ARG(x_dtype == MM_DTYPE_F16 || x_dtype == MM_DTYPE_BF16 || x_dtype == MM_DTYPE_F32,
                 "mm_fat_batched: x_dtype must be MM_DTYPE_F16, MM_DTYPE_BF16 or MM_DTYPE_F32");
    MM_CHECK_ARG(x && token_sorted && weight_sorted && counts && out && cap >= 0, "mm_fat_batched: null pointer or negative cap");
    MM_CHECK_ARG(T > 0 && n < (1 << 30) && T < (1 << 30), "mm_fat_batched: bad T/n");
    const FatbWs ws = fatb_carve(workspace, n, T, L->E, L->H, L->I);
    MM_CHECK_ARG(workspace && workspace_bytes >= ws.bytes, "mm_fat_batched: workspace too small (%zu < %zu)",
                 workspace_bytes, ws.bytes);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int E = L->E;
    const unsigned pg = (unsigned)std::min((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fatb_setup, dim3(1), dim3(FT_PLAN_MAX), 0, s, counts, skip, E, n, cap, ws.f.counts,
                       ws.f.offsets, ws.f.active, ws.f.nactive);
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)std::min((T + 255) / 256, 1024)), dim3(256), 0, s, ws.tcount, T, 0);
    hipLaunchKernelGGL(k_fatb_tokens<0>, dim3(pg), dim3(256), 0, s, token_sorted, ws.f.counts, ws.f.offsets, ws.f.order,
                       ws.tcount, ws.toff, ws.tpos, T, E, n);
    hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, s, ws.tcount, ws.toff, T);
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)std::min((T + 255) / 256, 1024)), dim3(256), 0, s, ws.tcount, T, 0);
    hipLaunchKernelGGL(k_fatb_tokens<1>, dim3(pg), dim3(256), 0, s, token_sorted, ws.f.counts, ws.f.offsets, ws.f.order,
                       ws.tcount, ws.toff, ws.tpos, T, E, n);
    const FatMode mode = fat_mode(L, n, false);
    fat_plan(L, n, cap, ws.f, s, mode, counts, nullptr);
    int r = fat_gemms(L, x, x_dtype, T, 1, token_sorted, n, ws.f, s, true, mode);
    if (r) return r;
    const dim3 grid((unsigned)((L->H / 4 + 255) / 256), (unsigned)T);
    hipLaunchKernelGGL(k_fatb_combine, grid, dim3(256), 0, s, out, reinterpret_cast<const uint16_t*>(ws.f.Y),
                       weight_sorted, ws.toff, ws.tpos, T, L->H);
    return check_launch("mm_fat_batched");
}

}  // extern "C"
