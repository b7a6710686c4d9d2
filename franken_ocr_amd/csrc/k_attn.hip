// k_attn.hip — causal prefill attention (decoder.rs:568-640 prefill_attention,
// :1282-1340 chunk_prefill_attention) on the bf16 matrix cores at f32 precision.
//
// A chunk's cs queries (global positions c0 .. c0 + cs - 1) attend keys
// [0, t] of the f32 prefix, per head, softmax(q.k * 1/sqrt(128)) . v.
//
// An f32 operand x is the exact sum of three bf16 values, x = x1 + x2 + x3
// (x1 = bf16(x), x2 = bf16(x - x1), x3 = x - x1 - x2: 8 + 8 + 8 bits of
// mantissa, each residual exact), and a product x.y is the six MFMAs
// x1y1 + x1y2 + x2y1 + x2y2 + x1y3 + x3y1, exact products summed in f32. The
// three terms left out are at most 2^-24 of |x||y|, an f32 product's unit
// roundoff. Measured against 64 bits the attention is nearer than in f32 MFMAs
// (1024 rows 1.4e-7, 2.4e-7), and six bf16 MFMAs take 6/16 of their matrix
// time. Values that have no such split (infinities, NaN, |x| so large that
// bf16(x) is infinite, nonzero |x| below 2^-100, whose last terms bf16 does
// not reach) are found while staging, and scores far from zero afterwards;
// their ranges take f32 MFMAs from memory (attend_f32).
//
// Block = 4 waves on one head and 128 query rows (32 per wave); the block
// walks its key range in tiles of 32 keys. The tile's K and V are split by
// the threads that load them and staged in LDS in MFMA fragment order (25 KB
// each, with 28 KB of Q terms two blocks per CU, at 256 VGPRs): K while the block's P.V of the tile
// before runs, V while its scores run, so each load has a phase of MFMAs to
// land in and one buffer of each is enough. Per wave S^T = K . Q^T (A = 32
// keys x 16 dims from LDS, B = 16 dims x 32 query rows from registers, the
// split Q held for the whole range), so lane (hf = lane / 32, j = lane % 32)
// holds row j's scores of the keys 8 (r / 4) + 4 hf + r % 4, r = 0..15, which
// is the B operand P^T of the P.V product if V's keys are taken in that order:
// the probabilities never leave their registers. O^T = V^T . P^T
// accumulates over one tile from zero and is added to the rescaled running
// output in one fma per value.
//
// The scores are kept in base-2 units: the kernel's scale is
// log2(e) / sqrt(128), so exp(s / sqrt(128) - max) is exp2 of the scaled
// score minus its max (the hardware v_exp_f32, about 1 ulp).
//
// Long prefixes are split into key ranges over more blocks (split-K); each
// writes its running max, denominator and unnormalised output, and a merge
// kernel folds them (log-sum-exp). A row whose keys all lie in other ranges
// contributes max -inf and nothing else. The ranges hold equal numbers of
// tiles, as many as make the least estimated time (attn_pick_splits; the
// causal chunk's row tiles need different numbers of tiles).
#include "focr_internal.hpp"
#include "k_common.hpp"

namespace focr {
namespace {

constexpr int kD = 128;          // head_dim
constexpr int kKT = 32;          // keys per LDS tile
constexpr int kRT = 128;         // query rows per block
constexpr int kBlocksPerCu = 2;  // the kernel's residency (LDS 77 KB, 256 VGPRs)
constexpr int kCuLds = 160 * 1024;
constexpr float kLog2e = 1.4426950408889634f;
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

struct AttnArgs {
    const float* q;  // row i, head h at q + i * ldq + h * hq
    const float* k;  // key j, head h at k + j * ldk + h * hk
    const float* v;
    float* out;      // single range: normalised context, out + i * ldo + h * ho
    float* part_o;   // split: [split][head][row][kD] unnormalised
    float* part_ml;  // split: [split][head][row][2] (base-2 max, denominator)
    int ldq, hq, ldk, hk, ldv, hv, ldo, ho;
    int cs, c0, c1, heads, split_len, nsplit;
    float scale;     // log2(e) / sqrt(head_dim)
};

// Key ranges of the row tile that holds chunk row `row`: it sees the keys
// [0, min(c1, c0 + the tile's last row + 1)).
__device__ __forceinline__ int attn_ranges(const AttnArgs& a, int row) {
    return (min(a.c1, a.c0 + (row / kRT + 1) * kRT) + a.split_len - 1) / a.split_len;
}

// Lane l's value and lane (l ^ 32)'s, in both (gfx950's v_permlane32_swap of
// a value with itself).
__device__ __forceinline__ float perm32(float v, float& other) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    other = __uint_as_float(r[1]);
    return __uint_as_float(r[0]);
}

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2bf));
}

// x - (the low / high bf16 of w) in one instruction: v_dot2_f32_bf16 with
// (-1, 0) or (0, -1). The differences taken here are exact. The constants are
// kept opaque: as an inline constant the instruction takes -1.0 for both.
__device__ __forceinline__ uint32_t opaque(uint32_t c) {
    asm("" : "+s"(c));
    return c;
}
__device__ __forceinline__ float sub_lo(float x, uint32_t w) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, w), __builtin_bit_cast(v2bf, opaque(0x0000bf80u)), x,
                                           false);
}
__device__ __forceinline__ float sub_hi(float x, uint32_t w) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, w), __builtin_bit_cast(v2bf, opaque(0xbf800000u)), x,
                                           false);
}

// The three bf16 terms of a and b, packed (a low, b high): w1, w2, w3.
__device__ __forceinline__ uint3 split2(float a, float b) {
    const uint32_t w1 = pk_bf16(a, b);
    const float ar = sub_lo(a, w1), br = sub_hi(b, w1);
    const uint32_t w2 = pk_bf16(ar, br);
    return make_uint3(w1, w2, pk_bf16(sub_lo(ar, w2), sub_hi(br, w2)));
}

// chk turns NaN or infinite (and stays so) where a first term is infinite or
// NaN: values that have no split. times (two equal bf16) lowers the limit: with
// 2^23 chk overflows from first terms of 2^104, or of 2^100 where they add up.
__device__ __forceinline__ float chk_terms(float chk, uint32_t w1, uint32_t times) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, w1), __builtin_bit_cast(v2bf, times), chk, false);
}
__device__ __forceinline__ bool not_finite(float x) { return !(fabsf(x) < INFINITY); }

// Below kMinSplit the third term runs out of bf16's range (its last bit is at
// 2^-133; the least term of 2^-100 is at 2^-123, still a normal number), so
// nonzero values below it have no split either. low_abs keeps the least
// magnitude that a thread stages, a v_min3 a pair; only where that is small is
// it seen whether the value is an ordinary zero. (An exact test of every value
// is three instructions a pair.)
constexpr float kMinSplit = 0x1p-100f;
__device__ __forceinline__ float low_abs(float low, float a, float b) {
    asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(low) : "v"(a), "v"(b));
    return low;
}
__device__ __forceinline__ bool too_low(float x) { return x != 0.0f && fabsf(x) < kMinSplit; }

struct Split8 {
    v4u w[3];  // terms 1, 2, 3 of eight values
    __device__ __forceinline__ void pair(int i, float a, float b, float& chk, uint32_t times = 0u) {
        const uint3 t = split2(a, b);
        chk = chk_terms(chk, t.x, times);
        w[0][i] = t.x;
        w[1][i] = t.y;
        w[2][i] = t.z;
    }
};

__device__ __forceinline__ v8bf bf8(const v4u& w) { return __builtin_bit_cast(v8bf, w); }

__device__ __forceinline__ v16f mfma_bf16(const v4u& a, const v4u& b, const v16f& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf8(a), bf8(b), c, 0, 0, 0);
}

// Mask the tile's scores (row j's keys 8 (r / 4) + 4 hf + r % 4) where it needs
// a mask, and move the row's running max: m_run becomes the new max, corr what
// the sums so far are scaled by; returns what the scaled scores are taken
// against (0 while the row has no key: every probability is 0).
__device__ __forceinline__ float softmax_max(v16f& sm, const AttnArgs& a, int kb, int ke, int t, int wrow0, int hf,
                                             float& m_run, float& corr) {
    if (kb + kKT > ke || kb + kKT - 1 > a.c0 + wrow0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = kb + 8 * (r >> 2) + 4 * hf + (r & 3);
            sm[r] = key <= t && key < ke ? sm[r] : -INFINITY;
        }
    }
    float tmax = sm[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, sm[r]);
    float other;
    tmax = perm32(tmax, other);
    const float m_new = fmaxf(m_run, fmaxf(tmax, other) * a.scale);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    corr = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    return m_use;
}

// Scores further from zero than this (base 2, as m_run) are left to the f32
// products: the fast path's exponent, one fma of the unrounded product, is off
// the rounded maximum by half an ulp of it, 2^-5 here, which all of a row's
// probabilities share and the denominator takes out again. From 2^31 on it
// would be past the exponents' range.
constexpr float kFarScore = 0x1p20f;
constexpr uint32_t kVLimit = 0x4b004b00u;  // 2^23 twice: V from 2^104, where a probability above 1 could overflow

// A wave's whole key range on f32 MFMAs from memory, for blocks whose values
// have no split and for rows whose scores are far from zero: infinities and
// NaN come out as the f32 products give them, and a range's largest score has
// the probability 1 exactly. The results have the fast path's layout.
__device__ __forceinline__ void attend_f32(const AttnArgs& a, int h, int ks, int ke, int t, int wrow0, int qrow,
                                           int lane, v16f (&oacc)[4], float& m_run, float& l_run) {
    const int hf = lane >> 5, j = lane & 31;
    const float* qp = a.q + static_cast<size_t>(qrow) * a.ldq + static_cast<size_t>(h) * a.hq + hf;
    const float* kh = a.k + static_cast<size_t>(h) * a.hk + hf;
    const float* vh = a.v + static_cast<size_t>(h) * a.hv + j;
#pragma unroll
    for (int d = 0; d < 4; ++d) oacc[d] = v16f(0.0f);
    m_run = -INFINITY;
    l_run = 0.0f;
    if (wrow0 >= a.cs) return;
    for (int kb = ks; kb < min(ke, a.c0 + wrow0 + 32); kb += kKT) {
        const float* kp = kh + static_cast<size_t>(min(kb + j, a.c1 - 1)) * a.ldk;
        // (the dot in four chains, the tile's outputs from zero: a value goes
        // through no more roundings than in the other forms)
        v16f sc[4] = {v16f(0.0f), v16f(0.0f), v16f(0.0f), v16f(0.0f)};
#pragma unroll 2
        for (int s = 0; s < kD / 4; s += 2)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                sc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(kp[32 * c + s], qp[32 * c + s], sc[c], 0, 0, 0);
        v16f sm = (sc[0] + sc[1]) + (sc[2] + sc[3]);
        float corr;
        const float m_use = softmax_max(sm, a, kb, ke, t, wrow0, hf, m_run, corr);
        float tsum = 0.0f;
        v16f o[4] = {v16f(0.0f), v16f(0.0f), v16f(0.0f), v16f(0.0f)};
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float p = __builtin_amdgcn_exp2f(sm[r] * a.scale - m_use);
            tsum += p;
            const float* vr = vh + static_cast<size_t>(min(kb + 8 * (r >> 2) + 4 * hf + (r & 3), a.c1 - 1)) * a.ldv;
#pragma unroll
            for (int d = 0; d < 4; ++d)
                o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[32 * d], p, o[d], 0, 0, 0);
        }
        l_run = l_run * corr + tsum;
#pragma unroll
        for (int d = 0; d < 4; ++d) oacc[d] = oacc[d] * corr + o[d];
    }
}

// LDS slots of 16 bytes (8 values). K: chunk c of 8 dims of a key at
// c * kKRow + key, a fragment (16 dims) two chunks; V: fragments of 64 slots.
constexpr int kKRow = kKT + 1;                   // one slot of padding: see the staging below
constexpr int kKTerm = (kD / 8) * kKRow;         // one term of a tile
constexpr int kQLds = 7;                         // Q fragments kept in LDS (all in registers spills)
constexpr int kVFrag = 64;
constexpr int kORow = kD / 4 + 1;                // a row of f32
constexpr int kVTerm = 2 * (kD / 32) * kVFrag;   // 2 steps of 16 keys x 4 blocks of 32 dims

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kBlocksPerCu))) void attn_prefill_kernel(
    const AttnArgs a) {
    __shared__ v4u smem[3 * kKTerm + 3 * kVTerm + 4 * kQLds * 64];
    __shared__ int bad[2];  // a K / V tile held values without a split (kept once set)
    v4u* const lk = smem;
    v4u* const lv = lk + 3 * kKTerm;
    // before and after the key loop: 32 rows of f32 per wave, one row's slots padded by one
    static_assert(4 * 32 * kORow <= 3 * kKTerm + 3 * kVTerm + 4 * kQLds * 64, "the waves' rows fit the staging");
    static_assert(kBlocksPerCu * (sizeof(smem) + sizeof(bad)) <= kCuLds, "the blocks of a CU fit its LDS");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int hf = lane >> 5, j = lane & 31;
    // the block's head, row tile and key range: blockIdx.x / heads counts the
    // ranges that have keys, the last row tile's first (they are the most and
    // the longest); heads vary fastest, so the XCDs (block id % 8) share every
    // row tile's work
    const int h = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.heads));
    int tile = (a.cs - 1) / kRT, split = static_cast<int>(blockIdx.x / static_cast<unsigned>(a.heads));
    for (; tile > 0; --tile) {
        const int ns = attn_ranges(a, tile * kRT);
        if (split < ns) break;
        split -= ns;
    }
    const int row0 = tile * kRT;                  // block's first chunk row
    const int wrow0 = row0 + wave * 32;           // this wave's first chunk row
    const int wrow = wrow0 + j;                   // this lane's chunk row
    const int qrow = wrow < a.cs ? wrow : a.cs - 1;
    const int t = a.c0 + wrow;                    // its global position
    // keys this block needs: [0, min(c1, c0 + row0 + kRT)), this split's part
    const int kmax = min(a.c1, a.c0 + row0 + kRT);
    const int ks = split * a.split_len;
    const int ke = min(ks + a.split_len, kmax);
    if (threadIdx.x < 2) bad[threadIdx.x] = 0;

    // K staging: thread = 8 dims (chunk kc) of keys kr and kr + 16. With the
    // chunks' rows of slots padded by one, the eight lanes of a write (one
    // key, eight chunks) and of a read (eight keys of one chunk) fall on
    // different banks.
    const int kc = threadIdx.x & 15, kr = threadIdx.x >> 4;
    // V staging: wave = the 8 keys of one fragment half (step wave / 2, half
    // wave % 2: keys 16 step + 4 half + {0..3, 8..11}), lane = dims 2 lane
    // and 2 lane + 1. Slot of dim d: half * 32 + (d % 32 with bit 0 flipped
    // by bit 3), for the same reason.
    const int vkey0 = 16 * (wave >> 1) + 4 * (wave & 1);
    const int koff = 4 * (kr * a.ldk + 8 * kc);
    const float* kh = a.k + static_cast<size_t>(h) * a.hk;
    const float* vh = a.v + static_cast<size_t>(h) * a.hv;
    // Buffer loads relative to the tile, which cost no address arithmetic in
    // vector registers: K rows past the prefix read as zero (the bounds check
    // of a buffer load), V rows are one per load, so a scalar offset clamped
    // to the prefix; a tile past the prefix reads as zero.
    auto tile_rsrc = [&](const float* base, int ld, int kb) {
        const int rows = min(a.c1 - kb, kKT);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + static_cast<size_t>(kb) * ld), 0,
                                                 rows > 0 ? 4 * ((rows - 1) * ld + kD) : 0, 0x00027000);
    };
    v4f pk[4];
    v2f pv[8];
    auto load_k = [&](int kb) {
        const auto r = tile_rsrc(kh, a.ldk, kb);
#pragma unroll
        for (int p = 0; p < 4; ++p)
            pk[p] = __builtin_bit_cast(
                v4f, __builtin_amdgcn_raw_buffer_load_b128(r, koff + (p >> 1) * 64 * a.ldk + 16 * (p & 1), 0, 0));
    };
    auto load_v = [&](int kb) {
        const auto r = tile_rsrc(vh, a.ldv, kb);
        const int last = max(a.c1 - kb, 1) - 1;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            pv[i] = __builtin_bit_cast(
                v2f, __builtin_amdgcn_raw_buffer_load_b64(r, 8 * lane,
                                                          4 * a.ldv * min(vkey0 + (i & 3) + 8 * (i >> 2), last), 0));
    };
    auto store_k = [&]() {
        float chk = 0.0f, low = INFINITY;
#pragma unroll
        for (int p = 0; p < 4; ++p) low = low_abs(low_abs(low, pk[p].x, pk[p].y), pk[p].z, pk[p].w);
        if (low < kMinSplit) {
#pragma unroll
            for (int p = 0; p < 4; ++p)
                if (too_low(pk[p].x) || too_low(pk[p].y) || too_low(pk[p].z) || too_low(pk[p].w)) chk = NAN;
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            Split8 s;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s.pair(i, pk[2 * p + (i >> 1)][2 * (i & 1)], pk[2 * p + (i >> 1)][2 * (i & 1) + 1], chk);
#pragma unroll
            for (int m = 0; m < 3; ++m) lk[m * kKTerm + kc * kKRow + kr + 16 * p] = s.w[m];
        }
        if (chk != chk) bad[0] = 1;
    };
    auto store_v = [&]() {
        float chk = 0.0f, low = INFINITY;
        const uint32_t limit = opaque(kVLimit);
#pragma unroll
        for (int i = 0; i < 8; ++i) low = low_abs(low, pv[i].x, pv[i].y);
        if (low < kMinSplit) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (too_low(pv[i].x) || too_low(pv[i].y)) chk = NAN;
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            Split8 s;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s.pair(i, pv[2 * i][e], pv[2 * i + 1][e], chk, limit);
            const int d = (2 * lane + e) & 31;
            const int slot = ((wave >> 1) * 4 + (lane >> 4)) * kVFrag + (wave & 1) * 32 + (d ^ ((d >> 3) & 1));
#pragma unroll
            for (int m = 0; m < 3; ++m) lv[m * kVTerm + slot] = s.w[m];
        }
        if (not_finite(chk)) bad[1] = 1;
    };

    load_k(ks);
    // The wave's Q rows through LDS (two rows a load; a lane's own row read
    // from memory would touch a line per row and piece), then the three terms
    // of q[row j][16 s + 8 hf .. + 7], s = 0..7.
    v4u* const rows = smem + wave * 32 * kORow;
    const float* qh = a.q + static_cast<size_t>(h) * a.hq + 4 * j;
#pragma unroll
    for (int i = 0; i < 16; ++i)
        rows[(2 * i + hf) * kORow + j] =
            *reinterpret_cast<const v4u*>(qh + static_cast<size_t>(min(wrow0 + 2 * i + hf, a.cs - 1)) * a.ldq);
    Split8 qf[8];
    float qchk = 0.0f, qlow = INFINITY;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const v4f x0 = __builtin_bit_cast(v4f, rows[j * kORow + 4 * s + 2 * hf]);
        const v4f x1 = __builtin_bit_cast(v4f, rows[j * kORow + 4 * s + 2 * hf + 1]);
        qlow = low_abs(low_abs(qlow, x0.x, x0.y), x0.z, x0.w);
        qlow = low_abs(low_abs(qlow, x1.x, x1.y), x1.z, x1.w);
        qf[s].pair(0, x0.x, x0.y, qchk);
        qf[s].pair(1, x0.z, x0.w, qchk);
        qf[s].pair(2, x1.x, x1.y, qchk);
        qf[s].pair(3, x1.z, x1.w, qchk);
    }
    if (qlow < kMinSplit) {
#pragma unroll 1
        for (int i = 0; i < kD; i += 4) {
            const v4f x = __builtin_bit_cast(v4f, rows[j * kORow + i / 4]);
            if (too_low(x.x) || too_low(x.y) || too_low(x.z) || too_low(x.w)) qchk = NAN;
        }
    }
    // the third terms of steps 0 .. kQLds - 1 stay in LDS (all in registers spills)
    v4u* lqw = lv + 3 * kVTerm + wave * kQLds * 64 + lane;
    v16f oacc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) oacc[d] = v16f(0.0f);
    float m_run = -INFINITY, l_run = 0.0f;  // l_run: this lane's keys only
    __syncthreads();  // every wave has its Q rows, and bad[] is cleared
#pragma unroll
    for (int s = 0; s < kQLds; ++s) lqw[64 * s] = qf[s].w[2];
    if (qchk != qchk) bad[0] = 1;
    store_k();
    load_v(ks);

    bool no_split = false;    // block-uniform
    unsigned long long far = 0;  // lanes whose scores were far from zero
    for (int kb = ks; kb < ke; kb += kKT) {
        const bool live = wrow0 < a.cs && kb <= a.c0 + wrow0 + 31;  // wave-uniform: some row sees some key
        __syncthreads();  // K(kb) staged; every wave is done with V of the tile before
        if ((no_split = __builtin_amdgcn_readfirstlane(bad[0]) != 0)) break;
        store_v();
        // (past the range's last tile too: rows of the prefix that nobody
        // uses; a conditional load would keep its registers all round the loop)
        load_k(kb + kKT);
        uint32_t pw[3][8] = {};  // the probabilities' terms, two per word
        float corr = 1.0f;
        if (live) {
            // the large products and the five smaller ones summed apart: eight
            // roundings at the score's own size. Each fragment of the next
            // step is read as soon as this step's last MFMA on it is out.
            v16f sm = v16f(0.0f), sl = v16f(0.0f);
            const v4u* kf = lk + hf * kKRow + j;
            v4u k1 = kf[0], k2 = kf[kKTerm], k3 = kf[2 * kKTerm], q3 = lqw[0];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int n = 2 * (s < 7 ? s + 1 : 7) * kKRow;
                sl = mfma_bf16(k3, qf[s].w[0], sl);
                __builtin_amdgcn_sched_barrier(0);
                k3 = kf[2 * kKTerm + n];
                sm = mfma_bf16(k1, qf[s].w[0], sm);
                sl = mfma_bf16(k1, q3, sl);
                sl = mfma_bf16(k1, qf[s].w[1], sl);
                __builtin_amdgcn_sched_barrier(0);
                k1 = kf[n];
                if (s < 7) q3 = s + 1 < kQLds ? lqw[64 * (s + 1)] : qf[s + 1].w[2];
                sl = mfma_bf16(k2, qf[s].w[1], sl);
                sl = mfma_bf16(k2, qf[s].w[0], sl);
                __builtin_amdgcn_sched_barrier(0);
                k2 = kf[kKTerm + n];
            }
            sm = sm + sl;
            const float m_use = softmax_max(sm, a, kb, ke, t, wrow0, hf, m_run, corr);
            far |= __builtin_amdgcn_ballot_w64(fabsf(m_use) > kFarScore);
            float tsum = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(sm[2 * i], a.scale, -m_use));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(sm[2 * i + 1], a.scale, -m_use));
                tsum += p0;
                tsum += p1;
                const uint3 w = split2(p0, p1);
                pw[0][i] = w.x;
                pw[1][i] = w.y;
                pw[2][i] = w.z;
            }
            l_run = l_run * corr + tsum;
        }
        __syncthreads();  // V(kb) staged; every wave is done with K(kb)
        if ((no_split = __builtin_amdgcn_readfirstlane(bad[1]) != 0)) break;
        store_k();
        load_v(kb + kKT);
        if (!live) continue;
        const v4u* vf = lv + hf * 32 + (j ^ ((j >> 3) & 1));
        v4u v1 = vf[0], v2 = vf[kVTerm], v3 = vf[2 * kVTerm];
        v16f o = v16f(0.0f);
#pragma unroll
        for (int i = 0; i < 8; ++i) {  // (32 dims d, 16 keys s) in turn, the smallest products first
            const int d = i >> 1, s = i & 1, nx = i < 7 ? i + 1 : 7;
            const int n = ((nx & 1) * 4 + (nx >> 1)) * kVFrag;
            const v4u p1 = {pw[0][4 * s], pw[0][4 * s + 1], pw[0][4 * s + 2], pw[0][4 * s + 3]};
            const v4u p2 = {pw[1][4 * s], pw[1][4 * s + 1], pw[1][4 * s + 2], pw[1][4 * s + 3]};
            const v4u p3 = {pw[2][4 * s], pw[2][4 * s + 1], pw[2][4 * s + 2], pw[2][4 * s + 3]};
            o = mfma_bf16(v3, p1, o);
            __builtin_amdgcn_sched_barrier(0);
            v3 = vf[2 * kVTerm + n];
            o = mfma_bf16(v2, p2, o);
            o = mfma_bf16(v2, p1, o);
            __builtin_amdgcn_sched_barrier(0);
            v2 = vf[kVTerm + n];
            o = mfma_bf16(v1, p3, o);
            o = mfma_bf16(v1, p2, o);
            o = mfma_bf16(v1, p1, o);
            __builtin_amdgcn_sched_barrier(0);
            v1 = vf[n];
            if (s == 1) {
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[d][r] = fmaf(oacc[d][r], corr, o[r]);
                o = v16f(0.0f);
            }
        }
    }
    // a score that overflowed (a sum of first terms can where the f32 dot does
    // not, and the two sums with opposite signs) shows as a denominator that is
    // not finite, or as a row with keys and no maximum
    far |= __builtin_amdgcn_ballot_w64(not_finite(l_run) || (m_run == -INFINITY && ks <= t));
    if (no_split || far) attend_f32(a, h, ks, ke, t, wrow0, qrow, lane, oacc, m_run, l_run);
    float other;
    l_run = perm32(l_run, other) + other;
    __syncthreads();  // the staging becomes the waves' output rows
    if (wrow0 >= a.cs) return;
    // lane (hf, j) holds O[row j][32d + 8 (r / 4) + 4 hf + r % 4] in
    // oacc[d][r]: through LDS to rows, two rows a store
    const float inv = a.nsplit == 1 ? 1.0f / l_run : 1.0f;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            rows[j * kORow + 8 * d + 2 * q + hf] = __builtin_bit_cast(
                v4u, v4f{oacc[d][4 * q] * inv, oacc[d][4 * q + 1] * inv, oacc[d][4 * q + 2] * inv,
                         oacc[d][4 * q + 3] * inv});
    const size_t pidx = (static_cast<size_t>(split) * a.heads + h) * a.cs;
    if (a.nsplit > 1 && hf == 0 && wrow < a.cs)
        *reinterpret_cast<float2*>(a.part_ml + (pidx + wrow) * 2) = make_float2(m_run, l_run);
    float* op = a.nsplit > 1 ? a.part_o + pidx * kD : a.out + static_cast<size_t>(h) * a.ho;
    const int ld = a.nsplit > 1 ? kD : a.ldo;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = wrow0 + 2 * i + hf;
        if (row < a.cs)
            *reinterpret_cast<v4u*>(op + static_cast<size_t>(row) * ld + 4 * j) = rows[(2 * i + hf) * kORow + j];
    }
}

// Combine lane l's value with lanes l ^ 16, l ^ 32, l ^ 48 (the four 16-lane
// rows): gfx950's v_permlane16_swap / v_permlane32_swap of a value with itself
// put both partners of an xor-16 (xor-32) pair in each lane (VALU; the
// shuffle form went through ds_bpermute at LDS latency). The pairs combine as
// the xor butterfly did: (r0 op r1) op (r2 op r3) in every lane.
__device__ __forceinline__ float perm16_lo(float v, float& hi) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    hi = __uint_as_float(r[1]);
    return __uint_as_float(r[0]);
}
__device__ __forceinline__ float wave16_max(float v) {
    float b;
    const float a = perm16_lo(v, b);
    v = fmaxf(a, b);
    const float c = perm32(v, b);
    return fmaxf(c, b);
}
__device__ __forceinline__ float wave16_sum(float v) {
    float b;
    const float a = perm16_lo(v, b);
    v = a + b;
    const float c = perm32(v, b);
    return c + b;
}

// ---- few rows and keys: f32 matrix cores ------------------------------------
// A call of a few key ranges is one chain of latencies: query rows, first tile,
// its products, output, merge. The kernel above puts 128 query rows, their
// splits and a pass through LDS for the output into that chain; this one has
// 64 rows a block, 16 a wave, and exact f32 products on v_mfma_f32_16x16x4, so
// its chain is shorter and its matrix time 16/6. Whole calls, this kernel and the
// one above, us: 16 rows 5.3, 8.1; 64 rows 10.1, 11.8; 128 rows 11.4, 18.6; 192
// rows 13.3, 15.1; 64 rows after 448 keys 12.6, 16.3; 128 after 128 12.8, 15.3,
// after 384 17.9, 18.7. Past that it loses: 256 rows 17.0, 16.4; 16 after 500
// 16.8, 14.9; 256 after 256 22.9, 20.7; 64 after 960 32.5, 19.7.
// Scores come as S^T = K Q^T (A = 16 keys x 4 dims from LDS, B = 4 dims x 16
// query rows in registers), so lane (g, j) holds row j's scores of keys 16 n +
// 4 g + r, the B operand of the P V product; dims in the order 8 (4 g + r') + m
// leave each lane 32 consecutive dims of its row. Ranges and partials are those
// of the kernel above, so the merge is shared.
constexpr int kSmRT = 64;                  // query rows per block
constexpr int kSmKeys = 512;               // keys of a call at most
constexpr int kSmBlocksPerCu = 3;          // residency (LDS 34 KB, 143 VGPRs)
constexpr int kLdsRow = kD + 4;            // padded LDS row (floats)
constexpr int kSub = kKT / 16;             // 16-key MFMA subtiles per tile
constexpr int kPieces = kKT * kD / 4 / 256;  // float4 of one matrix per thread and tile

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kSmBlocksPerCu))) void attn_prefill_small_kernel(
    const AttnArgs a) {
    extern __shared__ float4 lds_kv4[];  // K tile then V tile, [kKT][kLdsRow] floats each
    float* lk = reinterpret_cast<float*>(lds_kv4);
    float* lv = lk + kKT * kLdsRow;
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, j = lane & 15;
    const int h = blockIdx.y;
    const int split = blockIdx.z;
    const int row0 = blockIdx.x * kSmRT;         // block's first chunk row
    const int wrow = row0 + wave * 16 + j;       // this lane's chunk row
    const int qrow = wrow < a.cs ? wrow : a.cs - 1;
    const int t = a.c0 + wrow;                    // its global position
    // keys this block needs: [0, min(c1, c0 + row0 + kSmRT)), this split's part
    const int kmax = min(a.c1, a.c0 + row0 + kSmRT);
    const int ks = split * a.split_len;
    const int ke = min(ks + a.split_len, kmax);
    // a range past these rows' last key; the merge goes by tiles of kRT
    // rows, so it finds an empty range; block-uniform
    if (ks >= ke) {
        if (wrow < a.cs && g == 0 && ks < min(a.c1, a.c0 + (row0 / kRT + 1) * kRT))
            *reinterpret_cast<float2*>(
                a.part_ml + ((static_cast<size_t>(split) * a.heads + h) * a.cs + wrow) * 2) =
                make_float2(-INFINITY, 0.0f);
        return;
    }

    // Q fragment: qf[s] = q[row j][32g + s], s = 0..31
    float qf[32];
    {
        const float4* qp = reinterpret_cast<const float4*>(a.q + static_cast<size_t>(qrow) * a.ldq +
                                                           static_cast<size_t>(h) * a.hq + 32 * g);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const v4f x = *reinterpret_cast<const v4f*>(qp + u);
            qf[4 * u] = x.x;
            qf[4 * u + 1] = x.y;
            qf[4 * u + 2] = x.z;
            qf[4 * u + 3] = x.w;
        }
    }
    v4f oacc[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) oacc[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = -INFINITY, l_run = 0.0f;

    // tile loads: 32 keys x 128 floats = 1024 float4 per matrix, 4 per thread
    const int c4 = threadIdx.x & 31;  // float4 column
    const int r8 = threadIdx.x >> 5;  // 8 rows per pass
    const float* kh = a.k + static_cast<size_t>(h) * a.hk + 4 * c4;
    const float* vh = a.v + static_cast<size_t>(h) * a.hv + 4 * c4;
    // Tile loads of keys kb .. kb + kKT - 1 (rows clamped into the prefix; a
    // row past the range end is never used) and their LDS stores.
    v4f pk[kPieces], pv[kPieces];
    auto load_tile = [&](int kb) {
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            int key = kb + r8 + 8 * p;
            key = key < a.c1 ? key : a.c1 - 1;
            pk[p] = *reinterpret_cast<const v4f*>(kh + static_cast<size_t>(key) * a.ldk);
            pv[p] = *reinterpret_cast<const v4f*>(vh + static_cast<size_t>(key) * a.ldv);
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            *reinterpret_cast<v4f*>(lk + (r8 + 8 * p) * kLdsRow + 4 * c4) = pk[p];
            *reinterpret_cast<v4f*>(lv + (r8 + 8 * p) * kLdsRow + 4 * c4) = pv[p];
        }
    };
    load_tile(ks);
    store_tile();
    // every load so far (the Q fragment too) complete on every path into
    // the loop, so the loop's first MFMAs wait for none of the tile loads
    // issued inside it (vmcnt(0): the counter drains in issue order)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    // Each iteration issues the next tile's loads first, consumes the
    // current tile from LDS while they are in flight, then (after every wave
    // has read it) stores the next tile over it. The loads are consumed in
    // the iteration that issues them: a load carried into the next iteration
    // was folded with the one before the loop into a single load at the top
    // of the loop, which waited out a full memory round trip on every tile.
    for (int kb = ks; kb < ke; kb += kKT) {
        const bool more = kb + kKT < ke;
        if (more) load_tile(kb + kKT);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out before the tile's MFMAs

        // S^T for the subtiles of 16 keys; each score dot runs as two
        // 16-step MFMA chains (dims 32g + 16h + [0, 16), h = 0, 1) added at
        // the end, halving the f32 accumulation chain of the 128-term dot.
        // The 2 * kSub chains advance together: each step reads their four
        // dims of K (one 16-byte LDS read per chain) and issues one MFMA per
        // chain and dim, so a chain's dependent MFMAs interleave with the
        // other chains' (each chain's own order is unchanged: u, then dim).
        v4f sc[kSub][2];
#pragma unroll
        for (int n = 0; n < kSub; ++n) sc[n][0] = sc[n][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u2 = 0; u2 < 4; ++u2) {
            v4f kf[kSub][2];
#pragma unroll
            for (int n = 0; n < kSub; ++n)
#pragma unroll
                for (int hh = 0; hh < 2; ++hh)
                    kf[n][hh] = *reinterpret_cast<const v4f*>(lk + (16 * n + j) * kLdsRow + 32 * g + 16 * hh + 4 * u2);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int n = 0; n < kSub; ++n)
#pragma unroll
                    for (int hh = 0; hh < 2; ++hh)
                        sc[n][hh] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[n][hh][c], qf[16 * hh + 4 * u2 + c],
                                                                         sc[n][hh], 0, 0, 0);
        }
        v4f sacc[kSub];
#pragma unroll
        for (int n = 0; n < kSub; ++n) sacc[n] = sc[n][0] + sc[n][1];
        // scale, causal / range mask, online softmax (row j over 4 lanes)
        float pr[kSub][4];
        float tmax = -INFINITY;
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = kb + 16 * n + 4 * g + r;
                const float sv = sacc[n][r] * a.scale;
                const bool ok = key <= t && key < ke;
                pr[n][r] = ok ? sv : -INFINITY;
                tmax = fmaxf(tmax, pr[n][r]);
            }
        tmax = wave16_max(tmax);
        const float m_new = fmaxf(m_run, tmax);
        const float corr = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
        float tsum = 0.0f;
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = pr[n][r] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(pr[n][r] - m_new);
                pr[n][r] = p;
                tsum += p;
            }
        tsum = wave16_sum(tsum);
        l_run = l_run * corr + tsum;
        m_run = m_new;
        // the running output rescaled to the new max, then this tile's
        // V^T . P^T accumulated into it (step (n, r) is key kb + 16n + 4g + r)
#pragma unroll
        for (int m = 0; m < 8; ++m) oacc[m] = oacc[m] * corr;
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float* vr = lv + (16 * n + 4 * g + r) * kLdsRow + 8 * j;
                const v4f v0 = *reinterpret_cast<const v4f*>(vr);
                const v4f v1 = *reinterpret_cast<const v4f*>(vr + 4);
                const float b = pr[n][r];
                oacc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.x, b, oacc[0], 0, 0, 0);
                oacc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.y, b, oacc[1], 0, 0, 0);
                oacc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.z, b, oacc[2], 0, 0, 0);
                oacc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.w, b, oacc[3], 0, 0, 0);
                oacc[4] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.x, b, oacc[4], 0, 0, 0);
                oacc[5] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.y, b, oacc[5], 0, 0, 0);
                oacc[6] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.z, b, oacc[6], 0, 0, 0);
                oacc[7] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.w, b, oacc[7], 0, 0, 0);
            }
        if (more) {  // block-uniform
            __syncthreads();  // every wave is done with this tile
            store_tile();
            __syncthreads();
        }
    }
    if (wrow >= a.cs) return;
    // lane (g, j) holds O[row j][32g + 8r' + m] in oacc[m][r']
    if (a.nsplit == 1) {
        const float inv = 1.0f / l_run;
        float* op = a.out + static_cast<size_t>(wrow) * a.ldo + static_cast<size_t>(h) * a.ho + 32 * g;
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            float4 x0, x1;
            x0.x = oacc[0][rr] * inv;
            x0.y = oacc[1][rr] * inv;
            x0.z = oacc[2][rr] * inv;
            x0.w = oacc[3][rr] * inv;
            x1.x = oacc[4][rr] * inv;
            x1.y = oacc[5][rr] * inv;
            x1.z = oacc[6][rr] * inv;
            x1.w = oacc[7][rr] * inv;
            *reinterpret_cast<float4*>(op + 8 * rr) = x0;
            *reinterpret_cast<float4*>(op + 8 * rr + 4) = x1;
        }
        return;
    }
    const size_t pidx = (static_cast<size_t>(split) * a.heads + h) * a.cs + wrow;
    float* op = a.part_o + pidx * kD + 32 * g;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        *reinterpret_cast<float4*>(op + 8 * rr) = make_float4(oacc[0][rr], oacc[1][rr], oacc[2][rr], oacc[3][rr]);
        *reinterpret_cast<float4*>(op + 8 * rr + 4) = make_float4(oacc[4][rr], oacc[5][rr], oacc[6][rr], oacc[7][rr]);
    }
    if (g == 0) *reinterpret_cast<float2*>(a.part_ml + pidx * 2) = make_float2(m_run, l_run);
}

// Fold the key ranges: out = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s,
// M = max_s m_s, the maxima in base-2 units (a range with no key of the row
// has m = -inf, l = 0, O = 0). Only the ranges below the row tile's last key
// were written. 32 threads share one (row, head), thread c its dims
// 4c .. 4c + 3: lane s of the group reads range s's (max, denominator) and
// forms its weight, once for the group, and each range's output is one
// 16-byte load per thread, four ranges in flight. (The form before had 128
// threads a (row, head), one dim each, every one of which read and weighted
// every range.) Bound by the partials' bytes.
__device__ __forceinline__ float4 merge_row(const AttnArgs& a, int row, int h, int c) {
    const int ns = attn_ranges(a, row);
    const size_t step = static_cast<size_t>(a.heads) * a.cs;  // from one range's (head, row) to the next's
    const size_t p0 = static_cast<size_t>(h) * a.cs + row;
    float M = -INFINITY;
    for (int s0 = 0; s0 < ns; s0 += 32) M = fmaxf(M, s0 + c < ns ? a.part_ml[(p0 + (s0 + c) * step) * 2] : -INFINITY);
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 32));
    float den = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int s0 = 0; s0 < ns; s0 += 32) {
        const int n = min(ns - s0, 32);
        float w = -1.0f;  // a range without a key of the row
        if (c < n) {
            const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + (p0 + (s0 + c) * step) * 2);
            if (ml.x != -INFINITY) w = __builtin_amdgcn_exp2f(ml.x - M);
            den += ml.x == -INFINITY ? 0.0f : w * ml.y;
        }
        for (int s = 0; s < n; s += 4) {
            float4 o[4];
            float ws[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int si = min(s + i, n - 1);  // past the last: its output again, not added
                o[i] = *reinterpret_cast<const float4*>(a.part_o + (p0 + (s0 + si) * step) * kD + 4 * c);
                ws[i] = __shfl(w, si, 32);
                if (s + i >= n) ws[i] = -1.0f;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // (a range without a key of the row adds nothing, whatever the
                // outputs of the other rows of its tile made of V; one whose
                // weight is 0 adds 0 times its output, NaN where V is not finite)
                acc.x += ws[i] < 0.0f ? 0.0f : ws[i] * o[i].x;
                acc.y += ws[i] < 0.0f ? 0.0f : ws[i] * o[i].y;
                acc.z += ws[i] < 0.0f ? 0.0f : ws[i] * o[i].z;
                acc.w += ws[i] < 0.0f ? 0.0f : ws[i] * o[i].w;
            }
        }
    }
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) den += __shfl_xor(den, o, 32);
    return make_float4(acc.x / den, acc.y / den, acc.z / den, acc.w / den);
}

__global__ __launch_bounds__(256) void attn_merge_kernel(const AttnArgs a) {
    const int h = blockIdx.y, c = threadIdx.x & 31;
    const int row = blockIdx.x * 8 + (threadIdx.x >> 5);
    if (row >= a.cs) return;  // whole groups of 32
    *reinterpret_cast<float4*>(a.out + static_cast<size_t>(row) * a.ldo + static_cast<size_t>(h) * a.ho + 4 * c) =
        merge_row(a, row, h, c);
}

// The merge of attn_prefill_small_kernel's ranges (at most kSmRanges): thread =
// one dim of one (row, head), every range's (max, denominator) and output value
// requested at once, one round of latency where the group form above has one
// per four ranges. 64 rows after 448 keys, whole call: 14.7 us with the form
// above, 12.5 with this; many rows pay for the weights that every thread forms
// (1024 rows: 16 against 10 us).
constexpr int kSmRanges = kSmKeys / kKT;

__global__ __launch_bounds__(kD) void attn_merge_small_kernel(const AttnArgs a) {
    const int row = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
    const int ns = attn_ranges(a, row);
    float den = 0.0f, acc = 0.0f;
    float ms[kSmRanges], ls[kSmRanges], os[kSmRanges];
#pragma unroll
    for (int s = 0; s < kSmRanges; ++s) {
        const size_t pidx = (static_cast<size_t>(min(s, ns - 1)) * a.heads + h) * a.cs + row;
        ms[s] = a.part_ml[pidx * 2];
        ls[s] = a.part_ml[pidx * 2 + 1];
        os[s] = a.part_o[pidx * kD + d];
    }
    // every use unconditional (a guarded use lets the compiler sink the load
    // under the guard, one wait per range again): an unused range adds a
    // selected +0
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < kSmRanges; ++s) M = fmaxf(M, ms[s]);
#pragma unroll
    for (int s = 0; s < kSmRanges; ++s) {
        const bool use = s < ns && ms[s] != -INFINITY;
        const float w = __builtin_amdgcn_exp2f((use ? ms[s] : M) - M);
        const float dl = w * ls[s], da = w * os[s];
        den += use ? dl : 0.0f;
        acc += use ? da : 0.0f;
    }
    a.out[static_cast<size_t>(row) * a.ldo + static_cast<size_t>(h) * a.ho + d] = acc / den;
}

// The same merge with the next product's activation quantization fused in
// (o_proj's linear_int8_dynamic: the dynamic rule over the whole output row):
// one block per row over every head, thread t folding the float4 groups
// t + 256 i of the row's heads * 128 values as attn_merge_kernel does, then
// the row's amax, a_scale = amax / 127 (1 for a zero row) and the codes as
// the row quantizers form them, written row-major (TILED false) or in the
// 256 x 128 GEMM's tiled order, four codes to a word. The f32 context rows
// are never stored and the quantize launch goes.
constexpr int kMqGroups = 2;  // float4 groups per thread: rows up to 2048 values

template <bool TILED>
__global__ __launch_bounds__(256) void attn_merge_quant_kernel(const AttnArgs a, int8_t* __restrict__ xq,
                                                               float* __restrict__ xs) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    const int D = a.heads * kD, D4 = D >> 2;
    float4 val[kMqGroups];
    float amax = 0.0f;
#pragma unroll
    for (int gi = 0; gi < kMqGroups; ++gi) {
        const int g4 = tid + 256 * gi;
        float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (g4 < D4) {  // whole groups of 32 threads
            r = merge_row(a, row, g4 >> 5, g4 & 31);
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(r.x), fabsf(r.y)), fmaxf(fabsf(r.z), fabsf(r.w))));
        }
        val[gi] = r;
    }
    amax = wave_max_f_full(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float a_scale = amax > 0.0f ? amax / 127.0f : 1.0f;
    const float inv = 1.0f / a_scale;
    const int nst = D / kI8TiledStage;
#pragma unroll
    for (int gi = 0; gi < kMqGroups; ++gi) {
        const int g4 = tid + 256 * gi;
        if (g4 >= D4) continue;
        const float4 r = val[gi];
        const uint32_t word = static_cast<uint32_t>(static_cast<uint8_t>(quant_rule(r.x, a_scale, inv, kQuantDynamic))) |
                              static_cast<uint32_t>(static_cast<uint8_t>(quant_rule(r.y, a_scale, inv, kQuantDynamic))) << 8 |
                              static_cast<uint32_t>(static_cast<uint8_t>(quant_rule(r.z, a_scale, inv, kQuantDynamic))) << 16 |
                              static_cast<uint32_t>(static_cast<uint8_t>(quant_rule(r.w, a_scale, inv, kQuantDynamic))) << 24;
        const size_t off = TILED ? i8_tiled_act_off(row, g4 >> 2, nst) + 4 * (g4 & 3) : static_cast<size_t>(row) * D + 4 * g4;
        *reinterpret_cast<uint32_t*>(xq + off) = word;
    }
    if (tid == 0) xs[row] = a_scale;
}

// Chunk rows [cs][heads*128] (token-major) into a cache's head-major
// reference block: ref[h][c0 + i][:] = chunk[i][h*128 ..]. Thread = one
// float4 of one (row, head), K and V together.
__global__ __launch_bounds__(256) void attn_scatter_kv_kernel(const float* __restrict__ kc,
                                                              const float* __restrict__ vc, int cs, int heads,
                                                              float* __restrict__ ref_k, float* __restrict__ ref_v,
                                                              int cap, int c0) {
    const int idx = blockIdx.x * 256 + threadIdx.x;  // (row, head, float4)
    const int per_row = heads * (kD / 4);
    if (idx >= cs * per_row) return;
    const int i = idx / per_row;
    const int rem = idx - i * per_row;
    const int h = rem / (kD / 4), c = rem - h * (kD / 4);
    const size_t src = static_cast<size_t>(i) * heads * kD + h * kD + 4 * c;
    const size_t dst = (static_cast<size_t>(h) * cap + c0 + i) * kD + 4 * c;
    *reinterpret_cast<v4f*>(ref_k + dst) = *reinterpret_cast<const v4f*>(kc + src);
    *reinterpret_cast<v4f*>(ref_v + dst) = *reinterpret_cast<const v4f*>(vc + src);
}

}  // namespace

hipError_t launch_attn_scatter_kv(hipStream_t s, const float* k_chunk, const float* v_chunk, int cs, int heads,
                                  float* ref_k, float* ref_v, int cap, int c0) {
    if (cs < 1 || heads < 1 || c0 < 0 || c0 + cs > cap) return hipErrorInvalidValue;
    const int n = cs * heads * (kD / 4);
    FOCR_LAUNCH(attn_scatter_kv_kernel, dim3((n + 255) / 256), dim3(256), 0, s, k_chunk, v_chunk, cs, heads, ref_k,
                ref_v, cap, c0);
    return hipGetLastError();
}

size_t attn_partials_bytes(int cs, int heads, int nsplit) {
    return static_cast<size_t>(nsplit) * heads * cs * (kD + 2) * sizeof(float);
}

// Rows and keys for which attn_prefill_small_kernel is taken (measured beside it)
static bool attn_small(int cs, int c1) { return cs <= 192 && c1 <= kSmKeys && cs * c1 <= 65536; }

// The partials a call may ask scratch for. By time alone the range length grows
// slower than the call: 32768 rows asked for 3.2 GB, 131072 for 25 GB. Past the
// limit ranges get longer, down to one a row tile, which has no partials, and
// cost nothing that shows: 8192 rows (511 MB before) 1.09 to 1.11 ms, 16384
// (1.1 GB) 3.94 to 3.84, 65536 (9.2 GB) 62.1 to 55.0.
constexpr size_t kMaxPartials = size_t(512) << 20;

int attn_pick_splits(int cs, int c1, int heads, int cu_count, int* split_len) {
    if (attn_small(cs, c1)) {
        // the shortest ranges whose blocks are resident at once
        const long long slots = static_cast<long long>(kSmBlocksPerCu) * (cu_count > 0 ? cu_count : 1);
        int per = 1;
        for (;; ++per) {
            long long blocks = 0;
            for (int r = 0; r < cs; r += kSmRT)
                blocks += ((min(c1, c1 - cs + r + kSmRT) + kKT - 1) / kKT + per - 1) / per;
            if (blocks * heads <= slots || per * kKT >= c1) break;
        }
        *split_len = per * kKT;
        return (c1 + *split_len - 1) / *split_len;
    }
    // Row tile i (kRT rows) needs the tiles of keys [0, min(c1, c0 + kRT (i + 1))):
    // ranges of `per` tiles give sum over i of ceil(n_i / per) blocks per
    // head. The length taken is the one with the least estimated time (us),
    // fitted to whole calls of 16 to 1280 rows at 1 to 16 tiles a range: 3.0 a
    // tile where each block has a CU alone, 2 + 4.2 a tile where two share
    // one, more in rounds of that; with more than one range, the partials
    // written and read back at 6.6 TB/s and 11.5 for the merge launch and its
    // tail. Measured calls at the length taken and its neighbours: 1024 rows 3
    // tiles 36.2, 2 43.5, 4 38.2, 7 38.1; 768 rows 4 28.2, 3 32.8, 5 30.7; 256
    // rows after 768 keys 3 23.5, 2 27.5, 4 26.9; 2048 rows 12 83.7, 8 96.5.
    const int c0 = c1 - cs;
    const double cus = cu_count > 0 ? cu_count : 1;
    const int tiles = (c1 + kKT - 1) / kKT;
    double best = 0.0;
    int per = tiles;  // tiles per range
    for (int p = 1; p <= tiles; p += 1 + p / 16) {
        if (p < tiles && attn_partials_bytes(cs, heads, (tiles + p - 1) / p) > kMaxPartials) continue;
        double blocks = 0.0, part_rows = 0.0;
        for (int r = 0; r < cs; r += kRT) {
            const int n = (min(c1, c0 + r + kRT) + kKT - 1) / kKT, ranges = (n + p - 1) / p;
            blocks += static_cast<double>(ranges) * heads;
            part_rows += static_cast<double>(ranges) * heads * min(kRT, cs - r);
        }
        double us = blocks <= cus ? 3.0 * p : ceil(blocks / (kBlocksPerCu * cus)) * (2.0 + 4.2 * p);
        if (p < tiles) us += 11.5 + part_rows * (kD + 2) * sizeof(float) * 2 / 6.6e6;
        if (best == 0.0 || us < best) {
            best = us;
            per = p;
        }
    }
    const int len = per * kKT;
    *split_len = len;
    return (c1 + len - 1) / len;
}

hipError_t launch_attn_prefill(hipStream_t s, const AttnGeom& gm, const float* q, const float* k, const float* v,
                               float* out, int cs, int c0, int c1, int heads, int head_dim, int nsplit,
                               int split_len, float* part, AttnQuantOut* qo) {
    if (head_dim != kD || cs < 1 || c1 < 1 || c0 < 0 || c0 + cs != c1 || heads < 1 || nsplit < 1 ||
        split_len % kKT != 0 || static_cast<long long>(nsplit) * split_len < c1)
        return hipErrorInvalidValue;
    AttnArgs a{q, k, v, out, nullptr, nullptr, gm.ldq, gm.hq, gm.ldk, gm.hk, gm.ldv, gm.hv, gm.ldo, gm.ho,
               cs, c0, c1, heads, split_len, nsplit, kLog2e / sqrtf(static_cast<float>(head_dim))};
    if (nsplit > 1) {
        a.part_o = part;
        a.part_ml = part + static_cast<size_t>(nsplit) * heads * cs * kD;
    }
    if (attn_small(cs, c1)) {
        FOCR_LAUNCH(attn_prefill_small_kernel, dim3((cs + kSmRT - 1) / kSmRT, heads, nsplit), dim3(256),
                    2 * kKT * kLdsRow * sizeof(float), s, a);
    } else {
        int ranges = 0;
        for (int r = 0; r < cs; r += kRT) ranges += (min(c1, c0 + r + kRT) + split_len - 1) / split_len;
        FOCR_LAUNCH(attn_prefill_kernel, dim3(static_cast<unsigned>(heads) * ranges), dim3(256), 0, s, a);
    }
    hipError_t e = hipGetLastError();
    if (qo) qo->done = false;
    if (e != hipSuccess || nsplit == 1) return e;
    const int D = heads * kD;
    if (qo && D % kI8TiledStage == 0 && D <= 4 * 256 * kMqGroups) {
        if (qo->tiled)
            FOCR_LAUNCH(attn_merge_quant_kernel<true>, dim3(cs), dim3(256), 0, s, a, qo->xq, qo->xs);
        else
            FOCR_LAUNCH(attn_merge_quant_kernel<false>, dim3(cs), dim3(256), 0, s, a, qo->xq, qo->xs);
        qo->done = true;
        return hipGetLastError();
    }
    if (attn_small(cs, c1))
        FOCR_LAUNCH(attn_merge_small_kernel, dim3(cs, heads), dim3(kD), 0, s, a);
    else
        FOCR_LAUNCH(attn_merge_kernel, dim3((cs + 7) / 8, heads), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace focr
