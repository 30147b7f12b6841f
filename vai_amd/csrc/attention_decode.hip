// attention_decode.hip -- attention for a few new tokens over a long key range
// (a decode step, a short chunk): the same result as attention.hip's flash
// kernel, cut for the case where each KV head has few query rows.
//
// What bounds it: reading K and V once. The flash kernel gives every query
// head its own 128-row tile, so a decode step under grouped heads reads each
// key Hq / Hkv times and fills 1 of 128 MFMA columns; its partial results are
// 128 rows per unit. Here the Hq / Hkv * Tq query rows that share a KV head
// are the columns of one tile (16 or 32), a workgroup is one chunk of keys of
// one KV head, and its 4 waves take 32-key tiles of the chunk in turn, each
// with its own running softmax, so that no wave waits for another until the
// chunk ends. K fragments go straight to registers (16 keys x 64 bytes per
// load instruction); V goes through the wave's own LDS rows, padded by 32
// bytes so that the transposed reads of 8 rows hit 8 bank groups. The next
// tile's loads are in flight during a tile. fp32 keys and values are rounded
// to fp16 as they arrive (the flash path rounds the whole cache into a copy
// first). Rows of this call's new tokens are read from the call's own K / V,
// and an extra workgroup per KV head appends them to the cache: nothing else
// of the launch depends on the append, which therefore needs no launch of its
// own. The chunks' partial sums (fp32) meet in attention_decode_merge_kernel.
//
// Measured against the three launches this replaces (append, flash, merge),
// back-to-back calls, one fp16 token, 32 query heads over 8 KV heads: D = 64,
// 3000 of 4096 cached rows 19.3 -> 9.0 us (two launches take the host 7.4);
// D = 128, 16000 rows 60 -> 18.4 us (3.6 TB/s); 8 heads, D = 128, 4000 rows
// of an fp32 cache 14.8 us.
#include <algorithm>

#include "device_common.h"
#include "kernels.h"
#include "launch_once.h"

#define LDS_AS __attribute__((address_space(3)))

namespace vai_dev {

typedef float float2v __attribute__((ext_vector_type(2)));

namespace fd {
constexpr int NW = 4, KT = 32;   // waves per workgroup; keys per wave tile
template <int D> struct Lds {
    static constexpr int VROW = D * 2 + 32;             // bytes per V row in LDS
    static constexpr int VWAVE = KT * VROW;             // one wave's V tile
    static constexpr int OROW = D * 4 + 16;             // bytes per fp32 O row in the final exchange
    template <int NQ> static constexpr int bytes()
    {
        const int o = NW * NQ * 16 * OROW;
        return (NW * VWAVE > o ? NW * VWAVE : o) + NW * NQ * 16 * 8;   // (m, l) per wave and row after it
    }
};

// The launch's key range: [tb, te) are the 32-key tiles some row sees. They
// are dealt out in turn, tile tb + i to wave i % NW of unit (i / NW) % units,
// so that which tiles a wave reads first does not wait for the live count
// unless a window moves tb.
struct Range {
    uint32_t cached, live;
    int64_t tb, te;
    uint32_t used;   // units with work (at least 1)
};
__device__ __forceinline__ Range range_of(const AttnDecodeParams& p)
{
    Range r;
    r.cached = p.cache_count ? __builtin_amdgcn_readfirstlane(*p.cache_count) : 0u;
    r.live = p.ring ? r.cached + p.tkv : std::min(r.cached + p.tkv, p.kv_rows);
    const int64_t kend = std::min<int64_t>(p.mask.key_end_cached(p.tq - 1, r.cached), r.live);
    const int64_t kbeg = p.mask.key_start_cached(0, r.cached);
    r.tb = kbeg / KT;
    r.te = kend <= kbeg ? r.tb : (kend + KT - 1) / KT;
    const uint32_t n = __builtin_amdgcn_readfirstlane((uint32_t)(r.te - r.tb));
    r.used = std::min(p.units, std::max<uint32_t>((n + NW - 1) / NW, 1u));
    return r;
}
}

__device__ __forceinline__ half4 fd_read_tr16(const LDS_AS char* a)
{
    typedef short short4 __attribute__((ext_vector_type(4)));
    typedef __fp16 fp16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((LDS_AS fp16x4*)a));
}

// 8 consecutive elements from element index e of an fp16 or fp32 array, as fp16
template <typename T>
__device__ __forceinline__ half8 fd_load8(const T* p)
{
    if constexpr (sizeof(T) == 2) {
        return *(const half8*)p;
    } else {
        const float4v lo = *(const float4v*)p, hi = *(const float4v*)(p + 4);
        return __builtin_shufflevector(__builtin_convertvector(lo, half4), __builtin_convertvector(hi, half4), 0, 1, 2,
                                       3, 4, 5, 6, 7);
    }
}
__device__ __forceinline__ half8 fd_load8(const void* p, int dt, size_t e)
{
    return dt == DT_F16 ? fd_load8((const half_t*)p + e) : fd_load8((const float*)p + e);
}

// D: the padded head dim; NQ: 16-row query blocks per workgroup; T: element of
// K / V (or of the cache). Grid: (units + append, row blocks x hkv, batch).
template <int D, int NQ, typename T>
__global__ __launch_bounds__(256, (D <= 128 && NQ == 1) ? 2 : 1) void attention_decode_kernel(AttnDecodeParams p)
{
    using namespace fd;
    using L = Lds<D>;
    constexpr int KS = D / 32, DB = D / 16;      // 32-wide head-dim steps; 16-wide output blocks
    constexpr int VL = KT * D / 8 / 64;          // V chunks (8 elements) per lane and tile
    constexpr int LPR = D / 8, RPI = 64 / LPR;   // lanes per V row, V rows per load instruction
    extern __shared__ half8 fd_lds[];
    LDS_AS char* lds = (LDS_AS char*)(LDS_AS void*)fd_lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    const uint32_t HD = p.head_dim, unit = blockIdx.x, hk = blockIdx.y % p.hkv, rb = blockIdx.y / p.hkv, b = blockIdx.z;

    if (unit == p.units) {
        // the append: this call's rows into the cache, converted to its dtype
        if (rb != 0) return;
        const uint32_t cached = *p.cache_count;
        T* kc = (T*)p.k + (size_t)hk * p.kv_rows * HD;
        T* vc = (T*)p.v + (size_t)hk * p.kv_rows * HD;
        for (uint32_t e = threadIdx.x; e < p.n_new * HD; e += 256) {
            const uint32_t tok = e / HD, d = e - tok * HD, pos = cached + tok;
            if (!p.ring && pos >= p.kv_rows) continue;
            const size_t src = ((size_t)hk * p.n_new + tok) * HD + d, dst = (size_t)(pos % p.kv_rows) * HD + d;
            kc[dst] = (T)ld(p.k_new, p.new_dtype, src);
            vc[dst] = (T)ld(p.v_new, p.new_dtype, src);
        }
        return;
    }
    const T* kh = uniform_ptr((const T*)p.k + ((size_t)b * p.hkv + hk) * p.kv_rows * HD);
    const T* vh = uniform_ptr((const T*)p.v + ((size_t)b * p.hkv + hk) * p.kv_rows * HD);

    // One tile's loads; rows past the buffer read its first row of the tile.
    struct Tile { half8 k[2][KS], v[VL]; };
    const auto ring_row = [&](int64_t t) __attribute__((always_inline)) {
        const int64_t j0 = t * KT;   // (a ring's size is a multiple of 64: no tile wraps)
        return __builtin_amdgcn_readfirstlane((uint32_t)(p.ring ? j0 % p.kv_rows : j0));
    };
    const auto load = [&](int64_t t, Tile& x) __attribute__((always_inline)) {
        const uint32_t t0 = ring_row(t), n = std::min<uint32_t>(KT, p.kv_rows - t0);
        const T* kt = uniform_ptr(kh + (size_t)t0 * HD);
        const T* vt = uniform_ptr(vh + (size_t)t0 * HD);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t r = 16 * k + c16, rr = r < n ? r : 0u;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const uint32_t d = 32 * s + 8 * g;
                x.k[k][s] = fd_load8(kt + rr * HD + (d < HD ? d : 0u));
            }
        }
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            const uint32_t r = i * RPI + lane / LPR, rr = r < n ? r : 0u, d = 8 * (lane % LPR);
            x.v[i] = fd_load8(vt + rr * HD + (d < HD ? d : 0u));
        }
    };
    // Without a window the first tile's loads need nothing but the arguments:
    // issued before the live count arrives. A tile past it is read in vain: 34 MB
    // for 100 tokens in 16384 rows, 8 KV heads, D = 128, 11.6 us where a cache of
    // 4096 rows takes 9.5 (the flash kernel, which reads what is live, 13.4).
    const uint32_t i0 = unit * NW + wave, step = p.units * NW;
    // (D = 256: a tile is 128 registers, and a second one would spill)
    constexpr bool AHEAD = D <= 128;
    Tile cur;
    const bool early = AHEAD && p.mask.span == 0;
    if (early && (p.ring || i0 * KT < p.kv_rows)) load(i0, cur);

    // query rows: row r of the KV head is query head hk g + r / tq, token r % tq
    const uint32_t rows = p.rows, row0 = rb * p.rpb, rend = std::min(row0 + p.rpb, rows);
    half8 qf[NQ][KS];
    uint32_t tok[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const uint32_t r = std::min(row0 + q * 16 + c16, rend - 1);
        tok[q] = r % p.tq;
        const size_t base = (((size_t)b * p.hkv + hk) * rows + r) * HD;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const uint32_t d = 32 * s + 8 * g;
            const half8 v = fd_load8(p.q, p.q_dtype, base + (d < HD ? d : 0u));
            qf[q][s] = d < HD ? v : (half8)(half_t)0;
        }
    }
    const Range R = range_of(p);
    if (unit >= R.used) return;
    int64_t kbeg[NQ], kend[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        kend[q] = std::min<int64_t>(p.mask.key_end_cached(tok[q], R.cached), R.live);
        kbeg[q] = p.mask.key_start_cached(tok[q], R.cached);
    }

    // After a tile's loads: the call's own rows, read from its K / V; zeros for
    // rows past the live keys and for the padding past the head dim.
    const uint32_t ring0 = p.ring ? R.cached % p.kv_rows : 0u;   // ring row of the first new token
    const auto settle = [&](int64_t t, Tile& x) __attribute__((always_inline)) {
        const uint32_t n = (uint32_t)std::min<int64_t>(KT, R.live - t * KT), t0 = ring_row(t);
        // a row holding one of the new tokens: the token, else >= n_new
        const auto fresh = [&](uint32_t r) __attribute__((always_inline)) {
            uint32_t d = t0 + r - (p.ring ? ring0 : R.cached);
            if (p.ring && (int)d < 0) d += p.kv_rows;
            return d;
        };
        // whether the tile has such a row (uniform)
        const uint32_t f0 = fresh(0);
        if (p.n_new != 0 && (p.ring ? f0 < p.n_new || f0 + KT > p.kv_rows : t0 + KT > R.cached)) {
            const size_t nb = (size_t)hk * p.n_new * HD;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t f = fresh(16 * k + c16);
                if (f < p.n_new) {
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        const uint32_t d = 32 * s + 8 * g;
                        x.k[k][s] = fd_load8(p.k_new, p.new_dtype, nb + (size_t)f * HD + (d < HD ? d : 0u));
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < VL; ++i) {
                const uint32_t f = fresh(i * RPI + lane / LPR), d = 8 * (lane % LPR);
                if (f < p.n_new) x.v[i] = fd_load8(p.v_new, p.new_dtype, nb + (size_t)f * HD + (d < HD ? d : 0u));
            }
        }
        if (n < KT || HD < D) {
#pragma unroll
            for (int s = 0; s < KS; ++s)
                if (32u * s + 8 * g >= HD) x.k[0][s] = x.k[1][s] = (half8)(half_t)0;
#pragma unroll
            for (int i = 0; i < VL; ++i)
                if (i * RPI + lane / LPR >= n || 8u * (lane % LPR) >= HD) x.v[i] = (half8)(half_t)0;
        }
    };

    const float sl2 = p.scale * 1.4426950408889634f;   // scores in log2 units
    float m[NQ], l[NQ];
    float4v o[NQ][DB];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        m[q] = -__builtin_inff();
        l[q] = 0.f;
#pragma unroll
        for (int d = 0; d < DB; ++d) o[q][d] = (float4v)0.f;
    }
    LDS_AS char* vl = lds + wave * L::VWAVE;
    // transposed V read: source lane s of a 16-lane group points at key
    // 4 g + s / 4, columns 4 (s % 4) .. +3 of the output block
    const LDS_AS char* vr = vl + (4 * g + (c16 >> 2)) * L::VROW + (c16 & 3) * 8;

    if (AHEAD && !early && R.tb + i0 < R.te) load(R.tb + i0, cur);
    for (int64_t t = R.tb + i0; t < R.te; t += step) {
        Tile nxt;
        if (!AHEAD) load(t, cur);
        else if (t + step < R.te) load(t + step, nxt);
        settle(t, cur);
#pragma unroll
        for (int i = 0; i < VL; ++i)
            *(LDS_AS half8*)(vl + (i * RPI + lane / LPR) * L::VROW + (lane % LPR) * 16) = cur.v[i];
        // S^T, 16 keys x 16 query rows per fragment: lane (c16, g) holds query
        // row c16 and keys 16 k + 4 g .. +3
        float4v sa[2][NQ];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                sa[k][q] = (float4v)0.f;
#pragma unroll
                for (int s = 0; s < KS; ++s)
                    sa[k][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur.k[k][s], qf[q][s], sa[k][q], 0, 0, 0);
            }
        const int64_t j0 = t * KT;
        half8 pb[NQ];   // P^T operand: MFMA k index 8 g + j is key 16 (j / 4) + 4 g + j % 4
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int lo = (int)std::min<int64_t>(std::max<int64_t>(kbeg[q] - j0, -1), KT + 1);
            const int hi = (int)std::min<int64_t>(std::max<int64_t>(kend[q] - j0, -1), KT + 1);
            float v[8], tmax = -__builtin_inff();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int kl = 16 * (i >> 2) + 4 * g + (i & 3);
                v[i] = (kl >= hi || kl < lo) ? -__builtin_inff() : sa[i >> 2][q][i & 3] * sl2;
                tmax = fmaxf(tmax, v[i]);
            }
            tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
            // the row's reference m moves only when the max exceeds it by
            // more than 8 (P stays below 2^8), for the whole wave at once
            if (__any(tmax > m[q] + 8.f)) {
                const float mnew = fmaxf(m[q], tmax);
                const float alpha = __builtin_amdgcn_exp2f(m[q] - (mnew == -__builtin_inff() ? 0.f : mnew));
                l[q] *= alpha;
                m[q] = mnew;
#pragma unroll
                for (int d = 0; d < DB; ++d) o[q][d] *= alpha;
            }
            const float mref = m[q] == -__builtin_inff() ? 0.f : m[q];
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float e = __builtin_amdgcn_exp2f(v[i] - mref);
                sum += e;
                pb[q][i] = (half_t)e;
            }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            l[q] += sum;
        }
        // O^T += V^T P^T
#pragma unroll
        for (int d = 0; d < DB; ++d) {
            const half4 h0 = fd_read_tr16(vr + d * 32), h1 = fd_read_tr16(vr + 16 * L::VROW + d * 32);
            const half8 va = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                o[q][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[q], o[q][d], 0, 0, 0);
        }
        if (AHEAD) cur = nxt;
    }

    // the waves' sums meet in LDS (the V tiles are done with)
    __syncthreads();
    LDS_AS char* ml = lds + L::template bytes<NQ>() - NW * NQ * 16 * 8;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int r = q * 16 + c16;
        if (g == 0) {
            *(LDS_AS float2v*)(ml + (wave * NQ * 16 + r) * 8) = float2v{m[q], l[q]};
        }
        LDS_AS char* orow = lds + (wave * NQ * 16 + r) * L::OROW;
#pragma unroll
        for (int d = 0; d < DB; ++d) *(LDS_AS float4v*)(orow + (16 * d + 4 * g) * 4) = o[q][d];
    }
    __syncthreads();
    const bool whole = R.used == 1;
    const size_t head = (size_t)b * p.hkv + hk;
    constexpr int C4 = D / 4;
    for (uint32_t e = threadIdx.x; e < (rend - row0) * C4; e += 256) {
        const uint32_t r = e / C4, c = e % C4;
        float mw[NW], lw[NW], M = -__builtin_inff();
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float2v x = *(LDS_AS const float2v*)(ml + (w * NQ * 16 + r) * 8);
            mw[w] = x.x;
            lw[w] = x.y;
            M = fmaxf(M, x.x);
        }
        const float mref = M == -__builtin_inff() ? 0.f : M;
        float4v acc = (float4v)0.f;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float a = __builtin_amdgcn_exp2f(mw[w] - mref);
            acc += a * *(LDS_AS const float4v*)(lds + (w * NQ * 16 + r) * L::OROW + c * 16);
            sum += a * lw[w];
        }
        const uint32_t row = row0 + r;
        if (whole) {
            if (4 * c >= HD) continue;
            acc *= sum > 0.f ? 1.0f / sum : 0.f;
            const uint32_t h = hk * (p.hq / p.hkv) + row / p.tq, t = row % p.tq;
            const size_t out = (((size_t)b * p.tq + t) * p.hq + h) * HD + 4 * c;
            if (p.o_dtype == DT_F16) *(half4*)((half_t*)p.out + out) = __builtin_convertvector(acc, half4);
            else *(float4v*)((float*)p.out + out) = acc;
        } else {
            const size_t part = (head * p.units + unit) * rows + row;
            *(float4v*)(p.ws_o + part * D + 4 * c) = acc;
            if (c == 0) {
                p.ws_ml[2 * part] = M;
                p.ws_ml[2 * part + 1] = sum;
            }
        }
    }
}

// One workgroup per query row: O = sum_u 2^(m_u - M) O_u / sum_u 2^(m_u - M) l_u
// over the units that had keys (none: the row was written whole).
template <int D>
__global__ __launch_bounds__(256) void attention_decode_merge_kernel(AttnDecodeParams p)
{
    constexpr int C4 = D / 4, UG = 256 / C4;   // lanes per unit's row; units read at a time
    constexpr int MAXU = AttnDecodeParams::MAX_UNITS, AHEAD = 4;
    __shared__ float wgt[MAXU];
    __shared__ float4v part[256];
    __shared__ float red[4];
    const uint32_t row = blockIdx.x, hk = blockIdx.y, b = blockIdx.z, t = threadIdx.x, HD = p.head_dim;
    const size_t base = (((size_t)b * p.hkv + hk) * p.units) * p.rows + row;
    // Every load of the first 4 UG units is issued before the live count (and
    // with it the number of units that wrote anything) arrives; what an idle
    // unit's slot holds is dropped.
    const uint32_t c = t % C4, ug = t / C4;
    float2v ml = *(const float2v*)(p.ws_ml + 2 * (base + (size_t)std::min(t, p.units - 1) * p.rows));
    const float* op = p.ws_o + base * D + 4 * c;
    const size_t ustride = (size_t)p.rows * D;
    float4v v[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) v[i] = *(const float4v*)(op + std::min(ug + i * UG, p.units - 1) * ustride);
    const fd::Range R = fd::range_of(p);
    if (R.used == 1) return;
    // thread t weighs unit t (at most 256)
    const float m = t < R.used ? ml.x : -__builtin_inff(), l = t < R.used ? ml.y : 0.f;
    float M = m;
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) M = fmaxf(M, __shfl_xor(M, s));
    if ((t & 63) == 0) red[t >> 6] = M;
    __syncthreads();
    M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float w = M == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m - M);
    wgt[t] = w;
    float sum = w * l;
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) sum += __shfl_xor(sum, s);
    __syncthreads();   // red's readers are done, wgt is written
    if ((t & 63) == 0) red[t >> 6] = sum;
    float4v acc = (float4v)0.f;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
        if (ug + i * UG < R.used) acc += wgt[ug + i * UG] * v[i];
    for (uint32_t u = ug + AHEAD * UG; u < R.used; u += UG) acc += wgt[u] * *(const float4v*)(op + u * ustride);
    part[t] = acc;
    __syncthreads();
    if (t >= C4 || 4 * c >= HD) return;
#pragma unroll
    for (int i = 1; i < UG; ++i) acc += part[i * C4 + c];
    sum = red[0] + red[1] + red[2] + red[3];
    acc *= sum > 0.f ? 1.0f / sum : 0.f;
    const uint32_t h = hk * (p.hq / p.hkv) + row / p.tq, tk = row % p.tq;
    const size_t out = (((size_t)b * p.tq + tk) * p.hq + h) * HD + 4 * c;
    if (p.o_dtype == DT_F16) *(half4*)((half_t*)p.out + out) = __builtin_convertvector(acc, half4);
    else *(float4v*)((float*)p.out + out) = acc;
}

size_t attention_decode_workspace(const AttnParams& p, uint32_t units)
{
    return units <= 1 ? 0 : (size_t)p.batch * p.hkv * units * p.dec_rows * (p.dp + 2) * sizeof(float);
}

// Which calls take this path, and in how many units: called by attention_plan
// once p holds the flash plan (dp != 0). The line at 64 rows and 16 tokens,
// this path against the flash kernel (fp16, us): 64 rows, D = 128, 4000 / 16000
// cached 23 / 43 against 25 / 61; 128 rows 33 / 79 against 25 / 61; 64 rows,
// D = 256 15 / 27 against 24 / 38, 128 rows 23 / 40 against 24 / 38; one head's
// 32 rows (32 tokens), D = 128 24 / 33 against 18 / 27.
void attention_decode_plan(AttnParams& p, uint32_t cus, uint32_t key_rows, size_t flash_workspace)
{
    p.dec_units = 0;
    const uint32_t group = p.hq / p.hkv;
    if (p.tq > 16 || group * p.tq > 64 || (uint64_t)p.hq * p.tq > 65535) return;
    const auto at16 = [](const void* x) { return ((uintptr_t)x % 16) == 0; };
    p.dec_append = p.cache_count && p.tkv > 0 && p.tkv <= 32 && at16(p.k_new) && at16(p.v_new) ? 1u : 0u;
    p.dec_rows = group * p.tq;
    p.dec_rpb = std::min<uint32_t>(p.dec_rows, p.dp == 256 ? 16 : 32);   // (32 rows at D = 256 would spill)
    const uint32_t keys = p.span ? std::min<uint64_t>(key_rows, (uint64_t)p.span + p.tq + 2 * fd::KT) : key_rows;
    const uint32_t tiles = (keys + fd::KT - 1) / fd::KT, most = std::max<uint32_t>((tiles + fd::NW - 1) / fd::NW, 1);
    const uint64_t blocks = (uint64_t)p.batch * p.hkv * ((p.dec_rows + p.dec_rpb - 1) / p.dec_rpb);
    // two workgroups per CU where the kernel's registers allow it (16 rows, D <= 128)
    const uint32_t wgs = p.dec_rpb <= 16 && p.dp <= 128 ? 2 * cus : cus;
    uint32_t units = (uint32_t)std::min<uint64_t>(std::max<uint64_t>((wgs + blocks - 1) / blocks, 1), most);
    units = std::min<uint32_t>(units, AttnDecodeParams::MAX_UNITS);
    // never more workspace than the flash plan asks for
    while (units > 1 && attention_decode_workspace(p, units) > flash_workspace) --units;
    p.dec_units = units;
    // one unit over a long range (no workspace): fewer rows per workgroup, so that the rows fill the CUs
    while (units == 1 && most > 1 && p.dec_rpb > 1 &&
           (uint64_t)p.batch * p.hkv * ((p.dec_rows + p.dec_rpb - 1) / p.dec_rpb) < cus)
        p.dec_rpb = (p.dec_rpb + 1) / 2;
}

template <int D, int NQ, typename T>
static hipError_t decode_launch_t(const AttnDecodeParams& p, dim3 grid, hipStream_t s)
{
    constexpr int bytes = fd::Lds<D>::template bytes<NQ>();
    static PerDevice lds_once;
    if constexpr (bytes > 64 * 1024) {
        hipError_t e = set_max_lds(lds_once, (const void*)attention_decode_kernel<D, NQ, T>, bytes);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((attention_decode_kernel<D, NQ, T>), grid, dim3(256), bytes, s, p);
    return hipGetLastError();
}

template <int D>
static hipError_t decode_launch_d(const AttnDecodeParams& p, int kv_dtype, uint32_t batch, hipStream_t s)
{
    const uint32_t nrb = (p.rows + p.rpb - 1) / p.rpb;
    const dim3 grid(p.units + (p.n_new ? 1u : 0u), nrb * p.hkv, batch);
    hipError_t e;
    if (p.rpb <= 16)
        e = kv_dtype == DT_F16 ? decode_launch_t<D, 1, half_t>(p, grid, s) : decode_launch_t<D, 1, float>(p, grid, s);
    else if constexpr (D == 256)
        e = hipErrorInvalidValue;   // the plan keeps to 16 rows
    else
        e = kv_dtype == DT_F16 ? decode_launch_t<D, 2, half_t>(p, grid, s) : decode_launch_t<D, 2, float>(p, grid, s);
    if (e != hipSuccess || p.units == 1) return e;
    hipLaunchKernelGGL(attention_decode_merge_kernel<D>, dim3(p.rows, p.hkv, batch), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t attention_decode_launch(const AttnParams& a, hipStream_t s)
{
    AttnDecodeParams p{};
    p.out = a.out; p.q = a.q; p.k = a.k; p.v = a.v;
    p.o_dtype = a.o_dtype; p.q_dtype = a.q_dtype;
    p.hq = a.hq; p.hkv = a.hkv; p.tq = a.tq; p.tkv = a.tkv; p.head_dim = a.head_dim;
    p.cache_count = a.cache_count; p.kv_rows = a.kv_rows; p.ring = a.ring;
    if (a.dec_append) { p.k_new = a.k_new; p.v_new = a.v_new; p.n_new = a.tkv; p.new_dtype = a.new_dtype; }
    p.scale = a.scale;
    p.mask = a.mask;
    p.rows = a.dec_rows; p.rpb = a.dec_rpb; p.units = a.dec_units;
    p.ws_o = a.ws_o;
    p.ws_ml = a.ws_o + (size_t)a.batch * a.hkv * a.dec_units * a.dec_rows * a.dp;
    switch (a.dp) {
    case 64: return decode_launch_d<64>(p, a.kv_dtype, a.batch, s);
    case 128: return decode_launch_d<128>(p, a.kv_dtype, a.batch, s);
    default: return decode_launch_d<256>(p, a.kv_dtype, a.batch, s);
    }
}

}   // namespace vai_dev
