// attn_prompt.hip -- fp32 flash attention of many query rows on the gfx950 fp16
// matrix cores.
//
// Reference semantics (cogito-ml/cogito):
//   src/cuda/flash_attn_kernels.c:261-396  online softmax; GQA: query head h
//                                           reads KV head h * Hk / H; masked
//                                           scores are -FLT_MAX
//
// Two launches.  k_prompt_pack turns K and V once per call into MFMA operand
// fragments: per (sequence, KV head, 32-key tile) a record of 1 KiB blocks, a
// block holding the 16 bytes of each lane in lane order, so that the attention
// copies a record linearly and reads LDS without bank conflicts.  A value
// becomes hi + lo / 2^12 fp16, each rounded to nearest, after a power-of-two
// scaling per key row: off by at most 2^-23 of itself or 2^-52 of the row's
// maximum.  k_prompt_attn then runs 64 query rows a block (4 waves of 16 rows)
// over the tiles of one KV head: scores S^T = K Q^T and O^T = V^T P^T on
// v_mfma_f32_16x16x32_f16, Q and P as such pairs too (P times its key's V
// multiplier, scaled by a power of two that follows the largest contribution of
// each query row), the products hi hi in one fp32 sum, hi lo + lo hi in
// another, added at the end (lo lo, at most 2^-22 of the product, is left out).
// Three such products cost 3/16 of one on the fp32 matrix instructions, and 32
// products are summed per rounding instead of 2: the error against 64 bits is
// below that of k_attn's fp32 products (1021 causal rows of 32 heads over 8 of
// 128: 1.9e-7 against 3.2e-7; 1000 rows of 12 heads of 64 over 1900 keys 2.8e-7
// against 4.1e-7; 700 windowed rows of 16/2 heads of 96 2.1e-7 against 3.6e-7).
// lo times 2^12 and its own sums cost 2 us of 80 at the first of these sizes;
// without them a value below 2^-17 of its row's maximum loses bits (dims of O
// 2^-30 of the others': an error of 3e-3).  In the S^T orientation a lane holds
// one query row and 8 keys of a tile, which is the B operand of P^T: P never
// moves.
//
// Rows are ordered by position, heads fastest, so that a block's causal range
// ends early; tiles that no row of the block sees are skipped.  Measured at
// that size: 724 us for k_attn (scalar K loads a row apart, every tile of the
// causal mask), 80 us for the call here.  A call whose inputs the operands
// cannot hold costs this time before k_attn's.  Waiting bounds it, two waves a
// SIMD that meet at a barrier every tile: 238 vector instructions a wave and
// tile beside 48 MFMAs keep the VALU 25 % and the matrix cores 16 % busy.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "cgx_internal.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kTile = 32;                 // keys per record
constexpr int kBlock = 1024;              // bytes of a fragment block

inline hipStream_t stream() { return (hipStream_t)cgx_stream(); }

int launch_check(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        cgx_set_error("%s launch failed: %s", what, hipGetErrorString(e));
        return -1;
    }
    return 0;
}

enum { kMaskNone = 0, kMaskWindow = 2, kMaskCustom = 3, kMaskCausal = 5 };   // CGK_MASK_*

constexpr int P = 2;                      // parts of a value: hi, lo
// Blocks of a record: K fragments [key half][32-dim chunk][part], the keys' K
// and V multipliers (2 x 32 floats), then V fragments [16-dim tile][part].
template <int DP>
constexpr int kRecBlocks = 4 * (DP / 32) * P + 1;
template <int DP>
constexpr int kRecK = 2 * (DP / 32) * P;      // blocks before the multipliers

struct PackArgs {
    const float* K;              // [B][Nk][Hk][D]
    const float* V;
    int B, Nk, Hk, D, tiles;     // tiles: records per (sequence, KV head)
    unsigned* flag;              // set by an input that k_attn has to take
    uint8_t* rec;
};

struct PromptArgs {
    const float* Q;              // [B][Nq][H][D]
    const uint8_t* rec;
    int B, Nq, Nk, H, Hk, D, tiles;
    float scale;
    int mask_kind, window;
    const float* mask;           // custom additive [Nq][Nk]
    int splits, chunks;
    int first;                   // row chunks taken from the long end first
    int vec;                     // rows of O stored 16 bytes at a time
    float* O;                    // [B][Nq][H][D]
    float* part_o;               // [splits][B*Nq*H][D]
    float* part_ml;              // [splits][B*Nq*H][2]
    float* lse;                  // [B][H][Nq] or nullptr
    unsigned* flag;              // as in PackArgs
};

__device__ __forceinline__ int head_begin(int hk, int H, int Hk) { return (hk * H + Hk - 1) / Hk; }

// The flag is a word of host memory, written by the first inputs of a call that
// k_attn has to take, read once the stream is idle.
__device__ __forceinline__ void refuse(unsigned* flag) {
    __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Position p (0..31) of a V fragment row holds this key of the tile: the keys
// whose scores a lane of group p / 8 holds after S^T = K Q^T.
__device__ __forceinline__ int key_of_pos(int p) {
    const int g = p >> 3, j = p & 7;
    return j < 4 ? 4 * g + j : 16 + 4 * g + j - 4;
}

// Ends of the range of row maxima that the packed path takes; other inputs run
// k_attn (see PromptArgs::flag).  Q times scale and K below 2^50: a score in a
// row's held units, without Q's power of two, stays below 2^74.  V from 2^-100
// (or zero): a key's weight times its V multiplier is no subnormal.  A Q row is
// scaled up by at most 2^60: the lowest value, -FLT_MAX in held units, stands
// for a score below -2^67, so that a hidden key weighs nothing beside a visible
// one, and a score of queries too small for the scaling is off by at most 2^-28.
constexpr float kMaxQK = 0x1p50f, kMinV = 0x1p-100f;
constexpr int kMaxQExp = 60;

// Exponent e such that |v| * 2^e < 2^15 for |v| <= m, m finite (m = 0: 0).
__device__ __forceinline__ int scale_exp(float m) {
    const int ex = (int)(__float_as_uint(m) >> 23);            // 0 .. 254
    return m > 0.0f ? 141 - (ex > 1 ? ex : 1) : 0;             // 2^(ex-127) <= m < 2^(ex-126)
}

// hi + lo / kLo fp16 of 8 values below 2^15, each rounded to nearest.
constexpr float kLo = 4096.0f;             // |v - hi| <= 2^3: lo stays in range
__device__ __forceinline__ void split8(const float (&v)[8], f16x8& hi, f16x8& lo) {
#pragma unroll
    for (int i = 0; i < 8; i++) hi[i] = (_Float16)v[i];
#pragma unroll
    for (int i = 0; i < 8; i++) lo[i] = (_Float16)((v[i] - (float)hi[i]) * kLo);
}

// One block per (32-key tile, KV head, sequence).  A thread takes 8-dim units
// of one key (8 threads a key) for K, and 8-key units of one dim for V,
// through LDS.
template <int DP>
__global__ __launch_bounds__(kThreads) void k_prompt_pack(PackArgs a) {
    constexpr int CB = DP / 32, UNITS = DP / 8;
    constexpr int UPT = (UNITS + 7) / 8;               // units per thread
    __shared__ float s_v[kTile][DP + 1];
    const int tile = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
    const int nk = a.Nk;
    uint8_t* rec = a.rec + (((size_t)b * a.Hk + hk) * a.tiles + tile) * (kRecBlocks<DP> * kBlock);
    const int key = threadIdx.x >> 3, part = threadIdx.x & 7;
    const int kk = tile * kTile + key;
    const bool live = kk < nk;
    float* mul = (float*)(rec + kRecK<DP> * kBlock);
    float kv[UPT][8], vv[UPT][8];
    float km = 0.0f, vm = 0.0f;
    const size_t row = (((size_t)b * nk + (live ? kk : 0)) * a.Hk + hk) * a.D;
    float bad = 0.0f;
#pragma unroll
    for (int i = 0; i < UPT; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int d = 8 * (part + 8 * i) + j;
            const bool in = live && d < a.D;
            kv[i][j] = in ? a.K[row + d] : 0.0f;
            vv[i][j] = in ? a.V[row + d] : 0.0f;
            km = fmaxf(km, fabsf(kv[i][j]));
            vm = fmaxf(vm, fabsf(vv[i][j]));
            // x * 0 is NaN for an infinity or a NaN
            bad += kv[i][j] * 0.0f + vv[i][j] * 0.0f;
        }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        km = fmaxf(km, __shfl_xor(km, o));
        vm = fmaxf(vm, __shfl_xor(vm, o));
    }
    if (bad != bad || km >= kMaxQK || (vm > 0.0f && vm < kMinV)) refuse(a.flag);
    const int ek = scale_exp(km), ev = scale_exp(vm);
#pragma unroll
    for (int i = 0; i < UPT; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            kv[i][j] = ldexpf(kv[i][j], ek);
            vv[i][j] = ldexpf(vv[i][j], ev);
        }
    km = ldexpf(1.0f, -ek);
    vm = ldexpf(1.0f, -ev);
    if (part == 0) {
        mul[key] = km;
        mul[kTile + key] = vm;
    }
    const int kh = key >> 4;
#pragma unroll
    for (int i = 0; i < UPT; i++) {
        const int u = part + 8 * i;
        if (u >= UNITS) continue;
        const int c = u >> 2, g = u & 3, lane = (key & 15) + 16 * g;
        f16x8 hi, lo;
        split8(kv[i], hi, lo);
        f16x8* p = (f16x8*)(rec + (size_t)((kh * CB + c) * P) * kBlock) + lane;
        p[0] = hi;
        p[64] = lo;
#pragma unroll
        for (int j = 0; j < 8; j++) s_v[key][8 * u + j] = vv[i][j];
    }
    __syncthreads();
    uint8_t* vrec = rec + (size_t)(kRecK<DP> + 1) * kBlock;
    for (int e = threadIdx.x; e < (DP / 16) * 64; e += kThreads) {
        const int t = e >> 6, lane = e & 63, d = 16 * t + (lane & 15), g = lane >> 4;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = s_v[key_of_pos(8 * g + j)][d];
        f16x8 hi, lo;
        split8(x, hi, lo);
        f16x8* p = (f16x8*)(vrec + (size_t)(t * P) * kBlock) + lane;
        p[0] = hi;
        p[64] = lo;
    }
}

// Maximum / sum over the four lane groups (lanes 16 and 32 apart).  The
// maximum as a median with an infinity that the compiler cannot see: fmaxf
// first quiets values that come from a lane exchange.  No instruction here is
// written in inline asm: between an MFMA and a write of its C operand the
// hardware needs wait states, which the compiler inserts only around
// instructions that it knows.
__device__ __forceinline__ float max2(float a, float b) {
    float inf = __builtin_inff();
    asm("" : "+s"(inf));
    return __builtin_amdgcn_fmed3f(a, b, inf);
}
__device__ __forceinline__ float groups_max(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = max2(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return max2(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float groups_sum(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// split8 with the conversions back to fp32 as instructions of their own (the
// empty asm hides the value's origin): the compiler's v_fma_mix for the
// remainder runs at half rate.
__device__ __forceinline__ void split8_fast(const float (&v)[8], f16x8& hi, f16x8& lo) {
    f16x2 h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        h[i] = __builtin_convertvector((f32x2){v[2 * i], v[2 * i + 1]}, f16x2);
        float a = (float)h[i][0], b = (float)h[i][1];
        asm volatile("" : "+v"(a), "+v"(b));
        l[i] = __builtin_convertvector(
            (f32x2){(v[2 * i] - a) * kLo, (v[2 * i + 1] - b) * kLo}, f16x2);
    }
    hi = __builtin_bit_cast(f16x8, h);
    lo = __builtin_bit_cast(f16x8, l);
    asm volatile("" : "+v"(lo));
}

// Barrier that orders LDS accesses only: the next tile's loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr float kGrow = 8.0f;              // in binades

// Each iteration runs the products of the next tile's scores beside the
// softmax of this tile's, which do not depend on each other, so that the
// matrix cores and the VALU work at the same time within a wave (the call at
// the size above, before lo had sums of its own, 91 us with one tile at a time,
// 84 with its operand reads grouped, 82 so).  LDS holds the K part of tile
// t + 1 and the V part of tile t, both double buffered, behind one barrier a
// tile.  O is rescaled only where a row's maximum grows by more than kGrow or
// its contributions leave the room kept for them (83 -> 80 us).  128 rows a
// block do not fit the registers (head_dim 64, 4 x 1021 causal rows of 32
// heads: 175 us with spills, 164 with 64 rows).
template <int DP>
__global__ __launch_bounds__(kThreads, 2) void k_prompt_attn(PromptArgs a) {
    constexpr int CB = DP / 32, TD = DP / 16;
    constexpr int NB = kRecBlocks<DP>;              // 1 KiB blocks of a record
    constexpr int KB = kRecK<DP> + 1, VB = NB - KB; // K and multiplier blocks; V blocks
    constexpr int KS = (KB + kWaves - 1) / kWaves, VS = (VB + kWaves - 1) / kWaves;
    __shared__ __attribute__((aligned(16))) uint8_t s_k[2][KS * kWaves * kBlock];
    __shared__ __attribute__((aligned(16))) uint8_t s_v[2][VS * kWaves * kBlock];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = lane & 15, g = lane >> 4;
    const int hk = blockIdx.y, split = blockIdx.x;
    // the last rows first (they see the most keys under a causal mask); when
    // all blocks are resident at once, the second block of each CU from the
    // short end, so that the two add up to similar lengths
    const int b = (int)blockIdx.z % a.B, rank = (int)blockIdx.z / a.B;
    const int chunk = rank < a.first ? a.chunks - 1 - rank : rank - a.first;
    const int nk = a.Nk;
    const int h0 = head_begin(hk, a.H, a.Hk), G = head_begin(hk + 1, a.H, a.Hk) - h0;
    const int R = G * a.Nq;
    const int row0 = chunk * 16 * kWaves;
    if (row0 >= R) return;                             // uniform over the block

    // ---- the block's rows and the tiles they see
    const int rlast = min(row0 + 16 * kWaves, R) - 1;
    const int qa = row0 / G, qb = rlast / G;
    int klo = 0, khi = nk;
    if (a.mask_kind == kMaskCausal) khi = min(nk, qb + 1);
    // (a row that sees no key averages all of them, as in the reference)
    if (a.mask_kind == kMaskWindow && a.window >= 0 && qb - a.window < nk) {
        klo = max(0, qa - a.window);
        khi = (int)min((long long)nk, (long long)qb + a.window + 1);
    }
    // (a split without tiles leaves the lowest maximum and a zero sum)
    const int tn = (nk + kTile - 1) / kTile;
    const int t0 = max(klo / kTile, (int)((long long)tn * split / a.splits));
    const int t1 = min((khi + kTile - 1) / kTile, (int)((long long)tn * (split + 1) / a.splits));

    const uint8_t* rec = a.rec + ((size_t)b * a.Hk + hk) * a.tiles * (NB * kBlock);
    // a wave's blocks of a tile's K part and of its V part (past the end of a
    // part: its last block again; past the last tile: the last tile)
    f32x4 kst[KS], vst[VS];
    auto fetch_k = [&](int t) {
        const uint8_t* src = rec + (size_t)min(t, t1 - 1) * (NB * kBlock) + 16 * lane;
#pragma unroll
        for (int i = 0; i < KS; i++) kst[i] = *(const f32x4*)(src + min(wave + i * kWaves, KB - 1) * kBlock);
    };
    auto fetch_v = [&](int t) {
        const uint8_t* src = rec + (size_t)min(t, t1 - 1) * (NB * kBlock) + KB * kBlock + 16 * lane;
#pragma unroll
        for (int i = 0; i < VS; i++) vst[i] = *(const f32x4*)(src + min(wave + i * kWaves, VB - 1) * kBlock);
    };
    auto put_k = [&](int buf) {
#pragma unroll
        for (int i = 0; i < KS; i++)
            *(f32x4*)(&s_k[buf][(wave + i * kWaves) * kBlock + 16 * lane]) = kst[i];
    };
    auto put_v = [&](int buf) {
#pragma unroll
        for (int i = 0; i < VS; i++)
            *(f32x4*)(&s_v[buf][(wave + i * kWaves) * kBlock + 16 * lane]) = vst[i];
    };
    if (t0 < t1) {
        fetch_k(t0);
        fetch_v(t0);
    }

    // ---- Q operands: row 16 wave + n of the block, scaled, hi + lo
    f16x8 qh[CB], ql[CB];
    const int r = row0 + 16 * wave + n;
    const bool rok = r < R;
    const int rq = (rok ? r : rlast) / G, rh = h0 + (rok ? r : rlast) % G;
    const float* qp = a.Q + (((size_t)b * a.Nq + rq) * a.H + rh) * a.D;
    float qv[CB][8];
    float m = 0.0f, bad = 0.0f;
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int d = 32 * c + 8 * g + j;
            qv[c][j] = d < a.D ? qp[d] * a.scale : 0.0f;
            m = fmaxf(m, fabsf(qv[c][j]));
            bad += qv[c][j] * 0.0f;
        }
    m = groups_max(m);
    if (m >= kMaxQK) bad = __builtin_nanf("");
    const int e = min(scale_exp(m), kMaxQExp);
    const float qmul = ldexpf(1.0f, -e);
#pragma unroll
    for (int c = 0; c < CB; c++) {
#pragma unroll
        for (int j = 0; j < 8; j++) qv[c][j] = ldexpf(qv[c][j], e);
        split8(qv[c], qh[c], ql[c]);
    }
    if (bad != bad) refuse(a.flag);

    // scores are held without the row's Q multiplier (a power of two), under a
    // custom mask, which any value may enter, as they are: x times unit is the
    // score, and the softmax's exponent is (x - m) unit log2(e)
    const float unit = a.mask_kind == kMaskCustom ? 1.0f : qmul;
    float m_run = -__builtin_inff(), l_run = 0.0f;
    int er = 16;                   // O is held times 2^(141 - er)
    f32x4 o[TD], ox[TD];           // products hi hi; hi lo + lo hi, times kLo
    float x[8];                    // this tile's scores
#pragma unroll
    for (int t = 0; t < TD; t++) o[t] = ox[t] = (f32x4)(0.0f);
    // the wave's first and last query positions (mask-free tiles)
    const int wr0 = min(row0 + 16 * wave, rlast), wr1 = min(wr0 + 15, rlast);
    const int qmin = wr0 / G, qmax = wr1 / G;
    // the last tile that some row of this wave sees
    int tw1 = t1;
    if (a.mask_kind == kMaskCausal) tw1 = min(t1, qmax / kTile + 1);

    f32x4 s[2], sx[2];
    auto scores = [&](int buf) {
        f16x8 kf[2][CB][P];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int c = 0; c < CB; c++)
#pragma unroll
                for (int p = 0; p < P; p++)
                    kf[i][c][p] = ((const f16x8*)(s_k[buf] + ((i * CB + c) * P + p) * kBlock))[lane];
#pragma unroll
        for (int i = 0; i < 2; i++) s[i] = sx[i] = (f32x4)(0.0f);
#pragma unroll
        for (int c = 0; c < CB; c++) {
#pragma unroll
            for (int i = 0; i < 2; i++)
                s[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[i][c][0], qh[c], s[i], 0, 0, 0);
#pragma unroll
            for (int p = 0; p < P; p++)
#pragma unroll
                for (int i = 0; i < 2; i++)
                    sx[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        kf[i][c][p], p ? qh[c] : ql[c], sx[i], 0, 0, 0);
        }
    };
    // the K (0) or V (1) multipliers of the tile in K buffer `buf`
    auto multipliers = [&](int buf, int which, float (&m)[8]) {
        const float* mul = (const float*)(s_k[buf] + (KB - 1) * kBlock) + which * kTile;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float4 v = *(const float4*)(mul + 16 * i + 4 * g);
            m[4 * i] = v.x; m[4 * i + 1] = v.y; m[4 * i + 2] = v.z; m[4 * i + 3] = v.w;
        }
    };
    // the products' sums times the keys' multipliers, masked
    auto finish_scores = [&](int t, const float (&kmu)[8]) {
        const int kt = t * kTile;
        bool full = kt + kTile <= nk;
        switch (a.mask_kind) {
            case kMaskCausal: full = full && kt + kTile - 1 <= qmin; break;
            case kMaskWindow:
                full = full && (long long)kt >= (long long)qmax - a.window &&
                       (long long)kt + kTile - 1 <= (long long)qmin + a.window;
                break;
            case kMaskCustom: full = false; break;
            default: break;
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            x[j] = fmaf(sx[j >> 2][j & 3], 1.0f / kLo, s[j >> 2][j & 3]) * kmu[j];
        if (full) return;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int kk = kt + (j < 4 ? 4 * g + j : 12 + 4 * g + j);
            const int q = rq;
            bool vis = true;
            float v = x[j];
            if (a.mask_kind == kMaskCausal) vis = kk <= q;
            else if (a.mask_kind == kMaskWindow) vis = abs(kk - q) <= a.window;
            else if (a.mask_kind == kMaskCustom && kk < nk)
                v = v * qmul + a.mask[(size_t)q * nk + kk];
            x[j] = kk >= nk ? -__builtin_inff() : (vis ? v : -FLT_MAX);
        }
    };

    float vmu[8];                  // this tile's V multipliers
    if (t0 < t1) {
        put_k(0);
        put_v(0);
        fetch_k(t0 + 1);
        lds_barrier();
        float kmu[8];
        multipliers(0, 0, kmu);
        multipliers(0, 1, vmu);
        scores(0);
        finish_scores(t0, kmu);
        put_k(1);
    }
    for (int t = t0; t < t1; t++) {
        const int buf = (t - t0) & 1;
        lds_barrier();             // K of t + 1 and V of t are in LDS
        fetch_v(t + 1);
        fetch_k(t + 2);
        if (t < tw1) {             // (beyond it every row of this wave is masked)
            // ---- the next tile's products beside this tile's softmax
            scores(buf ^ 1);
            f16x8 ph, pl;
            const float c = unit * 1.44269504088896340736f;
            float mx = m_run;
#pragma unroll
            for (int j = 0; j < 8; j++) mx = fmaxf(mx, x[j]);
            // a maximum that has grown by no more than kGrow keeps its
            // place (weights up to 2^kGrow), and O its scale
            const float m_top = groups_max(mx);
            const float m_new = (m_top - m_run) * c > kGrow ? m_top : m_run;
            const float m_use = m_new == -__builtin_inff() ? 0.0f : m_new;
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * c);
            float sum = 0.0f, pm = 0.0f;
            float y[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float p = __builtin_amdgcn_exp2f((x[j] - m_use) * c);
                sum += p;
                y[j] = p * vmu[j];
                pm = fmaxf(pm, fabsf(y[j]));
            }
            l_run = l_run * alpha + sum;
            m_run = m_new;
            pm = groups_max(pm);
            // scale of the row's contributions: what earlier ones have
            // decayed to, or the tile's largest with room for 3 bits more
            const int ex = min((int)(__float_as_uint(pm) >> 23), 254);
            const int ea = (int)(__float_as_uint(alpha) >> 23) - 127 + (alpha < 1.0f ? 1 : 0);
            const int eo = max(er + ea, 16);
            const int en = ex > eo ? ex + 3 : eo;
            const float f = ldexpf(alpha, er - en);
            er = en;
            const float up = ldexpf(1.0f, 141 - en);
#pragma unroll
            for (int j = 0; j < 8; j++) y[j] *= up;
            split8_fast(y, ph, pl);
            if (__ballot(f != 1.0f)) {
#pragma unroll
                for (int tt = 0; tt < TD; tt++) {
                    o[tt] *= f;
                    ox[tt] *= f;
                }
            }
            // ---- O += P V; products of one accumulator stand four apart
            const uint8_t* vb = s_v[buf];
#pragma unroll
            for (int t4 = 0; t4 < TD; t4 += 4) {
                f16x8 vf[4][P];
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int p = 0; p < P; p++)
                        if (t4 + i < TD) vf[i][p] = ((const f16x8*)(vb + ((t4 + i) * P + p) * kBlock))[lane];
#pragma unroll
                for (int p = 0; p < P + 1; p++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (t4 + i < TD) {
                            f32x4& acc = p ? ox[t4 + i] : o[t4 + i];
                            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                vf[i][p == 2 ? P - 1 : 0], p == 1 ? pl : ph, acc, 0, 0, 0);
                        }
            }
        }
        // (nobody reads these buffers before the next barrier)
        put_v(buf ^ 1);
        put_k(buf);
        if (t + 1 < tw1) {
            float kmu[8];
            multipliers(buf ^ 1, 0, kmu);
            multipliers(buf ^ 1, 1, vmu);
            finish_scores(t + 1, kmu);
        }
    }

    // ---- O rows: lane (n, g) holds dims 16 tt + 4 g .. + 3 of its rows
    const size_t nrow = (size_t)a.B * a.Nq * a.H;
    const float L = groups_sum(l_run);
    // the row's maximum score (a masked one stays the lowest value)
    const float M = m_run > -FLT_MAX ? m_run * unit : m_run;
    const size_t orow = ((size_t)b * a.Nq + rq) * a.H + rh;
    const float down = ldexpf(1.0f, er - 141);
    float* dst = a.splits == 1 ? a.O + orow * a.D : a.part_o + ((size_t)split * nrow + orow) * a.D;
#pragma unroll
    for (int tt = 0; tt < TD; tt++) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = fmaf(ox[tt][i], 1.0f / kLo, o[tt][i]) * down;
            if (a.splits == 1) v[i] = L > 0.0f ? v[i] / L : 0.0f;
        }
        const int d = 16 * tt + 4 * g;
        if (!rok) continue;
        if (a.vec) {
            *(float4*)(dst + d) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (d + i < a.D) dst[d + i] = v[i];
        }
    }
    if (a.splits == 1) {
        if (rok && g == 0 && a.lse) {
            a.lse[((size_t)b * a.H + rh) * a.Nq + rq] =
                L > 0.0f ? M + logf(L) : -__builtin_inff();
        }
    } else if (rok && g == 0) {
        *(float2*)&a.part_ml[((size_t)split * nrow + orow) * 2] = make_float2(M, L);
    }
}

template <int DP>
int launch_all(const PackArgs& pk, const PromptArgs& a) {
    hipLaunchKernelGGL(k_prompt_pack<DP>, dim3(pk.tiles, pk.Hk, pk.B), dim3(kThreads), 0, stream(),
                       pk);
    if (launch_check("k_prompt_pack")) return -1;
    hipLaunchKernelGGL(k_prompt_attn<DP>, dim3(a.splits, a.Hk, a.chunks * a.B), dim3(kThreads), 0,
                       stream(), a);
    return launch_check("k_prompt_attn");
}

unsigned* g_flag = nullptr;    // host memory that the kernels write (PackArgs::flag)
int g_min_mega = 150;     // the packed path's least work (cgk_attn_prompt_pays), in 1e6

}  // namespace

// Whether the packed path takes an attention over fp32 K/V.  It costs a pass
// over K and V and a second launch; k_attn's time grows with the rows (in
// blocks of 32 per KV head), the keys and the head_dim.  Both measured, us a
// call with host work (k_attn / packed), by that product:
//   59e6   32 rows of 32/8 heads of 128, 449 keys        48 / 47
//   118e6  64 rows of the same                           49 / 48
//   134e6  16 rows, 2042 keys                            55 / 53
//   150e6  3 x 16 rows of 12 heads of 64, 2042 keys      59 / 57
//   200e6  64 rows of 16/2 heads of 96, 2042 keys        82 / 41
//   268e6  32 rows of 32/8 heads of 128, 2042 keys       88 / 52
//   401e6  3 x 16 rows of 16 heads of 128, 2042 keys    141 / 95
// Below the line the two are within 2 us; k_attn needs no scratch there.
// head_dim 32 and below stays with k_attn, whose error was the smaller one
// (2.4e-7 against 3.0e-7 with lo unscaled).
extern "C" int cgk_attn_prompt_pays(int B, int Nq, int Nk, int H, int Hk, int D) {
    const double rows = ((long long)((H + Hk - 1) / Hk) * Nq + 31) / 32 * 32.0;
    return D > 32 && D <= 128 && (double)B * Hk * rows * Nk * D >= 1e6 * g_min_mega;
}

extern "C" int cgx_flash_packed_min(int mega) {
    const int old = g_min_mega;
    if (mega >= 0) g_min_mega = mega;
    return old;
}

// Flash forward.  Returns 0, -1 on an error, or 1 when the call has to take
// k_attn (no scratch memory, a grid too large, stream capture).
extern "C" int cgk_attn_prompt_f32(const float* Q, const float* K, const float* V, int B, int Nq,
                                   int Nk, int H, int Hk, int D, float scale, int mask_kind,
                                   int window, const float* mask, float* O, float* lse) {
    if (cgx_is_capturing()) return 1;
    const int DP = (D + 31) / 32 * 32, tiles = (Nk + kTile - 1) / kTile;
    const long long R = (long long)((H + Hk - 1) / Hk) * Nq;
    PackArgs pk;
    PromptArgs a;
    memset(&pk, 0, sizeof(pk));
    memset(&a, 0, sizeof(a));
    // 64 rows a block; key splits until there are two blocks a CU, of at least
    // 8 tiles each
    const long long chunks = (R + 63) / 64, blocks = chunks * Hk * B;
    long long splits = 512 / blocks;
    if (splits > tiles / 8) splits = tiles / 8;
    if (splits < 1) splits = 1;
    if (Hk > 65535 || chunks * B > 65535 || R + 128 > 0x7fffffff) return 1;
    const long long first = blocks * splits <= 512 ? 256 / (splits * Hk * B) : chunks;
    const size_t nrow = (size_t)B * Nq * H;
    pk.rec = (uint8_t*)cgx_scratch_try(CGX_SLOT_WS4, (size_t)(4 * (DP / 32) * P + 1) * kBlock *
                                                         tiles * Hk * B);
    if (!g_flag && hipHostMalloc((void**)&g_flag, 64, hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        g_flag = nullptr;
    }
    bool room = pk.rec && g_flag;
    if (room && splits > 1) {
        a.part_o = (float*)cgx_scratch_try(CGX_SLOT_WS2, (size_t)splits * nrow * D * 4);
        a.part_ml = (float*)cgx_scratch_try(CGX_SLOT_WS3, (size_t)splits * nrow * 2 * 4);
        room = a.part_o && a.part_ml;
    }
    if (!room) return 1;           // the fp32 kernel needs less
    // no earlier call's kernels run any more: each is waited for (flash_run)
    *(volatile unsigned*)g_flag = 0;
    pk.K = K; pk.V = V;
    pk.B = a.B = B;
    pk.Nk = a.Nk = Nk;
    pk.Hk = a.Hk = Hk;
    pk.D = a.D = D;
    pk.tiles = a.tiles = tiles;
    pk.flag = a.flag = g_flag;
    a.Q = Q; a.Nq = Nq; a.H = H;
    a.rec = pk.rec;
    a.scale = scale;
    a.mask_kind = mask_kind; a.window = window; a.mask = mask;
    a.splits = (int)splits;
    a.chunks = (int)chunks;
    a.first = first < 1 ? 1 : (first > chunks ? (int)chunks : (int)first);
    a.vec = D == DP && !((uintptr_t)O & 15);
    a.O = O;
    a.lse = lse;
    const int rc = DP == 64 ? launch_all<64>(pk, a)
                 : DP == 96 ? launch_all<96>(pk, a) : launch_all<128>(pk, a);
    if (rc || splits == 1) return rc;
    return cgk_attn_combine(a.part_o, a.part_ml, (int)splits, (int)nrow, D, Nq, H, O, lse);
}

extern "C" int cgk_attn_prompt_refused(void) { return *(volatile unsigned*)g_flag != 0; }
