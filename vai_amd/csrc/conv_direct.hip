// conv_direct.hip -- implicit-GEMM convolution for fp16 weights as stored, any
// odd kernel, stride, image width and channel count: the rows the packed
// kernels of conv.hip cannot hold (wider than 128 outputs, as in the first
// stages of an image network), and 5x5 and larger kernels.
//
// What bounds these layers is reading the image and writing the output once;
// the matrix work is small. A workgroup of 8 waves takes 4 output rows x 32
// columns and 64 output channels (one row and 32 channels a wave), so that a
// 3x3 reads 1.6 of each input value instead of 3 for one row. Per block of
// input channels it stages the input window transposed, [row][column][channel]
// (8 channels x 8 columns per item: eight 16-byte loads, a register
// transpose, eight 16-byte LDS writes; fp32 rounded to fp16 on the way, the
// staging's contract), and the weights as [output channel][octet][8]. An
// octet is 8 channels of one tap: four of them, whichever they are, make one
// MFMA step (lane group g takes octet 4 s + g through a table of the octets'
// window offsets), so that 3 channels cost 9 octets and not 9 x 32 channels.
// Both strides are odd numbers of 16-byte units: the 16 rows of a fragment
// read hit distinct banks. The weights' taps are spread from their stored
// order, c k k + tap, by two-byte LDS writes, once per workgroup and block.
//
// What is left after that is latency: at 32 -> 64 channels, stride 2, 320x320
// (200 workgroups, one a CU, all channels in one block) load, transpose, barrier
// and MFMAs follow each other; a wave waits for its loads and at the barriers
// 53% of the time and for an issue slot 22%, the VALU (addresses and transpose:
// divisions are multiplications by constants of the launch, the loads share one
// offset where rows are whole aligned pieces) works 13%, LDS 3% and the matrix
// cores 3%. Measured against the generic gather kernel (conv as a GEMM of
// gemm.hip, us): that 33.7 -> 9.7; 64 -> 64, 160x160 55.7 -> 13.0;
// 1x1 17.5 -> 7.6; 16 -> 16, 320x320, fp32 image 52.7 -> 12.6; 32 -> 32,
// 333x333 72 -> 18.6. Reading the window untransposed, 8 two-byte LDS reads a
// lane and fragment, took 21 for the first.
//
// The input is MFMA operand A (16 positions), the weight B, so a lane ends up
// with four consecutive positions of one channel: one 8- or 16-byte store.
#include <algorithm>

#include "device_common.h"
#include "kernels.h"
#include "launch_once.h"

#define LDS_AS __attribute__((address_space(3)))

namespace vai_dev {

namespace cd {
constexpr int PW = 32, NT = 512;      // output columns; threads (8 waves)
constexpr int NF = PW / 16, NB = 2;   // fragments per wave: 32 positions x 32 channels
// output channels per workgroup (32 or 64) -> its output rows, one a wave per 32 channels
__host__ __device__ constexpr int ph_of(int ct) { return 8 * 32 / ct; }

// The staging of one launch: channels per block, the window's rows and (whole
// 8-column pieces of) columns, octets of a block and in whole MFMA steps, the
// 16-byte units per position and weight row, and the LDS sizes.
struct Plan {
    uint32_t cb, c8, rh, rw, oct, oct4, pu, wu;
    uint32_t in_bytes, w_bytes, lds;
};
// n / d as one multiplication, m = magic(d): exact while n d < 2^32
inline uint32_t magic(uint32_t d) { return d == 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d); }
__device__ __forceinline__ uint32_t div_by(uint32_t n, uint32_t m) { return m ? __umulhi(n, m) : n; }
__host__ __device__ inline Plan plan_of(uint32_t cb, uint32_t ks, uint32_t stride, uint32_t ct)
{
    Plan q;
    q.cb = cb;
    q.c8 = (cb + 7) / 8;
    q.rh = (ph_of(ct) - 1) * stride + ks;
    q.rw = ((PW - 1) * stride + ks + 7 + 7) / 8 * 8;   // (the first column lies up to 7 past a multiple of 8)
    q.oct = q.c8 * ks * ks;
    q.oct4 = (q.oct + 3) / 4 * 4;
    q.pu = q.c8 | 1;
    q.wu = q.oct4 | 1;
    q.in_bytes = q.rh * q.rw * q.pu * 16;
    q.w_bytes = ct * q.wu * 16;
    q.lds = q.in_bytes + q.w_bytes + q.oct4 * 4;
    return q;
}
}

// KS: the kernel size 1 or 3, or 0: p.ks.
template <typename TI, int CT, int KS>
__global__ __launch_bounds__(cd::NT, 4) void conv_direct_kernel(ConvDirectParams p)
{
    using namespace cd;
    constexpr int PH = ph_of(CT);
    extern __shared__ half8 cd_lds[];
    LDS_AS char* xin = (LDS_AS char*)(LDS_AS void*)cd_lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const uint32_t ks = KS ? KS : p.ks, kk = ks * ks, sd = p.stride, pad = ks / 2, CI = p.ci, K = CI * kk;
    const Plan q = plan_of(p.cb, ks, sd, CT);
    LDS_AS char* win = xin + q.in_bytes;
    LDS_AS uint32_t* tab = (LDS_AS uint32_t*)(win + q.w_bytes);

    const uint32_t x0 = blockIdx.x * PW, yb = blockIdx.y % p.ytiles, co0 = (blockIdx.y / p.ytiles) * CT, b = blockIdx.z;
    const uint32_t y0 = yb * PH;
    const int cx = (int)(x0 * sd) - (int)pad;                      // the window's first needed column
    const int cx8 = cx >= 0 ? cx / 8 * 8 : -((-cx + 7) / 8 * 8);   // ... and first staged one
    const uint32_t xoff = (uint32_t)(cx - cx8);
    const int ry = (int)(y0 * sd) - (int)pad;
    const TI* X = (const TI*)p.x + (size_t)b * CI * p.hi * p.wi;
    const half_t* W = (const half_t*)p.w;
    const size_t plane = (size_t)p.hi * p.wi;

    // window offset of octet i: channels 8 (i / kk) .., tap i % kk (taps
    // fastest: the weights' two-byte writes then spread over the banks)
    for (uint32_t i = tid; i < q.oct4; i += NT) {
        const uint32_t c = div_by(i, p.m_kk), t = i - c * kk, kh = KS ? t / (KS ? KS : 1) : t / ks, kw = t - kh * ks;
        tab[i] = i < q.oct ? ((kh * q.rw + kw) * q.pu + c) * 16 : 0u;
    }

    // bias and scale of the lane's channels (a missing one reads W and is ignored)
    const uint32_t cw = co0 + (wave / PH) * 32 + fr;   // + 16 j
    float bias[NB], sc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t c = std::min(cw + 16 * j, p.co - 1);
        const float bv = (float)(p.bias ? (const half_t*)p.bias : W)[c], sv = (float)(p.scale ? (const half_t*)p.scale : W)[c];
        bias[j] = p.bias ? bv : 0.f;
        sc[j] = p.scale ? sv : 1.f;
    }

    float4v acc[NF][NB];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[f][j] = (float4v)0.f;

    const uint32_t nv = q.rw / 8, items = q.c8 * q.rh * nv;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    // whole aligned pieces from an image under 2^31 bytes: loads through a
    // resource, one offset for the 8 channels, zero outside the image
    const uint32_t plane_bytes = (uint32_t)plane * sizeof(TI);
    const bool buf = p.wi % 8 == 0 && ((uintptr_t)p.x % 16) == 0 && (size_t)CI * plane * sizeof(TI) < (1ull << 31);
    // the weights in items of one channel's taps (KS 3), else of 8 stored values
    const uint32_t wv = KS == 3 ? q.cb : (q.cb * kk + 7) / 8, witems = CT * wv;
    for (uint32_t c0 = 0; c0 < CI; c0 += q.cb) {
        const uint32_t cn = std::min(q.cb, CI - c0), wn = cn * kk;   // channels and weights per output channel
        if (c0) __syncthreads();   // every wave is done with the last block
        // the first U items of the weights a thread: loaded ahead of the window
        constexpr int U = 4;
        half8 wr[U];
        half_t w9[U];
        const auto load_w = [&](uint32_t base) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t it = std::min(base + u * NT, witems - 1), o = div_by(it, p.m_wv), i = it - o * wv;
                const half_t* row = W + (size_t)std::min(co0 + o, p.co - 1) * K;
                if constexpr (KS == 3) {
                    const half_t* src = row + (c0 + std::min(i, cn - 1)) * 9;
                    wr[u] = load8(src);
                    w9[u] = src[8];
                } else {
                    // (a piece over the end of W's row moves down from its last 8 values)
                    const uint32_t k = c0 * kk + std::min(i * 8, wn - 1), start = std::min(k, K - 8);
                    wr[u] = load8(row + start);
                    if (start != k) wr[u] = shift_down(wr[u], k - start);
                }
            }
        };
        load_w(tid);
        // the weights' padding is zero: octets past the block, channels past Ci,
        // and in a short last block what the block before left (its infinities
        // must not meet the zeros of the window)
        if (q.oct4 != q.oct || cn % 8 || cn != q.cb) {
            for (uint32_t i = tid; i < CT * q.wu; i += NT) *(LDS_AS half8*)(win + i * 16) = (half8)(half_t)0;
            __syncthreads();
        }
        // the window (channel octet fastest: the lanes of a column piece write one run)
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            (void*)uniform_ptr(X + (size_t)c0 * plane), (short)0, (int)((CI - c0) * plane_bytes), 0x00020000);
        for (uint32_t it = tid; it < items; it += NT) {
            const uint32_t rest = div_by(it, p.m_c8), c = it - rest * q.c8, r = div_by(rest, p.m_nv), cv = rest - r * nv;
            const int col = cx8 + (int)cv * 8, y = ry + (int)r;
            const bool in = y >= 0 && y < (int)p.hi && col >= 0 && col < (int)p.wi;
            half8 t[8];
            if (buf) {
                const uint32_t off =
                    in ? ((uint32_t)y * p.wi + (uint32_t)col) * (uint32_t)sizeof(TI) + c * 8 * plane_bytes : 0x80000000u;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if constexpr (sizeof(TI) == 2) {
                        t[e] = __builtin_bit_cast(
                            half8, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(off + e * plane_bytes), 0, 0));
                    } else {
                        const float4v lo = __builtin_bit_cast(
                            float4v, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(off + e * plane_bytes), 0, 0));
                        const float4v hi = __builtin_bit_cast(
                            float4v, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(off + e * plane_bytes), 16, 0));
                        t[e] = __builtin_shufflevector(__builtin_convertvector(lo, half4),
                                                       __builtin_convertvector(hi, half4), 0, 1, 2, 3, 4, 5, 6, 7);
                    }
                }
            } else {
                // (a piece over the row's end moves down from its last 8
                // columns; an octet past the block's last channel reads the first)
                const uint32_t start = in ? std::min((uint32_t)col, p.wi - 8) : 0u;
                const TI* src = X + (size_t)(c0 + (c * 8 < cn ? c * 8 : 0u)) * plane + (in ? (size_t)y * p.wi + start : 0);
#pragma unroll
                for (int e = 0; e < 8; ++e) t[e] = load8(src + (c * 8 + e < cn ? e * plane : 0));
                if (p.wi % 8) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) t[e] = shift_down(t[e], (uint32_t)col - start);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (!in || c * 8 >= cn) t[e] = (half8)(half_t)0;
            }
            if (cn % 8) {   // (other channels' values behind the block's last octet)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (c * 8 + e >= cn) t[e] = (half8)(half_t)0;
            }
            // column j's channel pair (2 k, 2 k + 1) is one dword
            LDS_AS char* dst = xin + ((r * q.rw + cv * 8) * q.pu + c) * 16;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                u32x4 v;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    v[k] = __builtin_amdgcn_perm(__builtin_bit_cast(u32x4, t[2 * k + 1])[j / 2],
                                                 __builtin_bit_cast(u32x4, t[2 * k])[j / 2],
                                                 (j & 1) ? 0x07060302u : 0x05040100u);
                *(LDS_AS u32x4*)(dst + j * q.pu * 16) = v;
            }
        }
        for (uint32_t base = tid;;) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t it = base + u * NT, o = div_by(it, p.m_wv), i = it - o * wv;
                if (it >= witems) continue;
                LDS_AS char* row = win + o * q.wu * 16;
                if constexpr (KS == 3) {
                    if (i >= cn) continue;
                    LDS_AS half_t* d = (LDS_AS half_t*)(row + (i >> 3) * 9 * 16 + (i & 7) * 2);
#pragma unroll
                    for (int e = 0; e < 8; ++e) d[e * 8] = wr[u][e];
                    d[64] = w9[u];
                } else if constexpr (KS == 1) {
                    if (i * 8 < wn) *(LDS_AS half8*)(row + i * 16) = wr[u];
                } else {
                    uint32_t c = i * 8 / kk, t = i * 8 - c * kk;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (i * 8 + e < wn) *(LDS_AS half_t*)(row + ((c >> 3) * kk + t) * 16 + (c & 7) * 2) = wr[u][e];
                        if (++t == kk) { t = 0; ++c; }
                    }
                }
            }
            base += NT * U;
            if (base - tid >= witems) break;
            load_w(base);
        }
        __syncthreads();
        // this wave's output row, positions 16 f + fr, and its 32 channels
        const LDS_AS char* xb = xin + ((wave % PH) * sd * q.rw + xoff + fr * sd) * q.pu * 16;
        const uint32_t fstep = 16 * sd * q.pu * 16;
        const LDS_AS char* wb = win + ((wave / PH) * 32 + fr) * q.wu * 16 + fg * 16;
        for (uint32_t s = 0; s < q.oct4; s += 4) {
            const uint32_t off = tab[s + fg];
            half8 xf[NF], wf[NB];
#pragma unroll
            for (int f = 0; f < NF; ++f) xf[f] = *(const LDS_AS half8*)(xb + off + f * fstep);
            if (s + 4 > q.oct) {   // octets past the block: zero times a zero weight
                if (s + fg >= q.oct)
#pragma unroll
                    for (int f = 0; f < NF; ++f) xf[f] = (half8)(half_t)0;
            }
#pragma unroll
            for (int j = 0; j < NB; ++j) wf[j] = *(const LDS_AS half8*)(wb + j * 16 * q.wu * 16 + s * 16);
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[f][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[f], wf[j], acc[f][j], 0, 0, 0);
        }
    }

    // lane (fr, fg): channel 16 j + fr of the wave's, positions x0 + 16 f + 4 fg .. +3 of its row
    const uint32_t y = y0 + wave % PH;
    if (y >= p.ho) return;
    const bool al = p.wo % 4 == 0 && ((uintptr_t)p.out % 16) == 0 && ((uintptr_t)p.residual % 16) == 0;
    const bool before = p.residual_order == 1;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t co = cw + 16 * j;
        if (co >= p.co) continue;
        const size_t row = (((size_t)b * p.co + co) * p.ho + y) * p.wo;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const uint32_t x = x0 + 16 * f + 4 * fg;
            if (x >= p.wo) continue;
            const size_t o = row + x;
            float4v v = acc[f][j], rr = (float4v)0.f;
            if (p.residual) {
                if (al) {
                    if (p.residual_dtype == DT_F16) rr = __builtin_convertvector(*(const half4*)((const half_t*)p.residual + o), float4v);
                    else rr = *(const float4v*)((const float*)p.residual + o);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) rr[e] = ld(p.residual, p.residual_dtype, row + std::min(x + e, p.wo - 1));
                }
            }
            const auto act = [&](auto EPI) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float t = fmaf(v[e], sc[j], bias[j]) + (before ? rr[e] : 0.f);
                    v[e] = epilogue(t, EPI) + (before ? 0.f : rr[e]);
                }
            };
            switch (p.epilogue) {
            case 0: act(std::integral_constant<uint32_t, 0>{}); break;
            case 1: act(std::integral_constant<uint32_t, 1>{}); break;
            case 2: act(std::integral_constant<uint32_t, 2>{}); break;
            case 3: act(std::integral_constant<uint32_t, 3>{}); break;
            case 4: act(std::integral_constant<uint32_t, 4>{}); break;
            default: act(std::integral_constant<uint32_t, 5>{}); break;
            }
            if (al) {
                if (p.o_dtype == DT_F16) *(half4*)((half_t*)p.out + o) = __builtin_convertvector(v, half4);
                else *(float4v*)((float*)p.out + o) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (x + e < p.wo) st(p.out, p.o_dtype, o + e, v[e]);
            }
        }
    }
}

// Channels per block: all of them, or a multiple of 8 while the stage fits
// `room` bytes; 0: not even 8 do.
static uint32_t block_of(uint32_t ci, uint32_t ks, uint32_t stride, uint32_t ct, uint32_t room)
{
    if (cd::plan_of(ci, ks, stride, ct).lds <= room) return ci;
    uint32_t cb = 0;
    while (cb + 8 < ci && cd::plan_of(cb + 8, ks, stride, ct).lds <= room) cb += 8;
    return cb;
}

// 64 output channels and 4 rows a workgroup, or 32 and 8 (no idle waves) up to 32 channels.
static uint32_t ct_of(uint32_t co) { return co <= 32 ? 32 : 64; }

// Where the gather of gemm.hip takes less time than this kernel (us, gather /
// this). A full chip is more workgroups than CUs can hold idle rows for free.
static bool gather_faster(bool x32, uint32_t ci, uint32_t ho, uint32_t rows, uint32_t ctiles, uint64_t wgs, uint32_t ks,
                          uint32_t stride, uint32_t cus)
{
    // Windows with gaps: the staging reads what no tap uses, once per 64 output
    // channels. 1x1 stride 4, 256 -> 64, 40x132 22 / 65. 1x1 stride 2 pays off for
    // one tile of channels (64 -> 64, 160x160 17.9 / 10.4) and where several leave
    // CUs idle (64 -> 256, 40x132 13.2 / 10.6, 300x300 61 / 83; 512 -> 512, 8x136
    // fp16 36.5 / 41, fp32 71 / 54), stride 3 with few fp16 channels (64 -> 64,
    // 160x160 17.9 / 13.0, fp32 40x132 12.7 / 15.3); 3x3 stride 4 likewise (64 -> 64,
    // 160x160 54 / 28; 64 -> 256, 85 / 98, 40x132 49 / 30).
    if (stride > ks) {
        if (ks == 1 && stride == 2) return ctiles > 1 && (x32 ? wgs > 2 * cus : ci >= 512 || wgs > cus);
        if (ks == 1) return stride > 3 || x32 || ci > 64 || (ctiles > 1 && wgs > cus);
        return ctiles > 1 && wgs > cus;
    }
    // Images of one row (of the 4 or 8 that a workgroup takes) that fill the chip:
    // 3x3 stride 2, 512 -> 512, 8000 columns 352 / 562, stride 1 353 / 371 (4000
    // columns 1 / 0.63; 64 -> 64, 64000, fp16 77 / 69); 5x5 stride 2, 64 -> 64, 64000
    // columns 185 / 219. 1x1, whose gather is cheap, and strides as wide as the
    // kernel, with up to a quarter of the rows (1x1 16 -> 32, 2x64000 23 / 27; 3x3
    // stride 3, 4x64000 57 / 75); 1x1 with many channels beyond that (fp16 512 ->
    // 512, 5x8000 174 / 212; fp32 2x8000 98 / 127, 3x8000 168 / 157).
    const bool thin = 4 * (uint64_t)ho <= rows;
    if (ks > 1 && stride == ks && thin && wgs > 2 * cus) return true;
    if (wgs <= 4 * cus) return false;
    if (ks == 1) return thin || (ci >= 256 && (x32 ? 2 * (uint64_t)ho <= rows : 8 * (uint64_t)ho <= 7 * (uint64_t)rows));
    return ho == 1 && (ks == 3 ? stride > 1 || x32 || ci >= 256 : ks == 5 && stride > 1);
}

// Rows of at least one 8-column piece, weights of at least one 8-value piece,
// and a grid of at most 65535 in y and z.
bool conv_direct_ok(uint32_t batch, uint32_t ci, uint32_t wi, uint32_t co, uint32_t ho, uint32_t ks, uint32_t stride,
                    int x_dt, uint32_t cus)
{
    const uint32_t ct = ct_of(co), ph = cd::ph_of(ct), wo = (wi - 1) / stride + 1;
    const uint64_t ytiles = (ho + ph - 1) / ph, ctiles = (co + ct - 1) / ct;
    return wi >= 8 && ks <= 31 && stride <= 64 && (uint64_t)ci * ks * ks >= 8 && (uint64_t)ci * ks * ks < (1u << 24) &&
           batch <= 65535 && ytiles * ctiles <= 65535 && block_of(ci, ks, stride, ct, 160 * 1024) > 0 &&
           !gather_faster(x_dt == DT_F32, ci, ho, (uint32_t)ytiles * ph, (uint32_t)ctiles,
                          batch * ytiles * ctiles * ((wo + cd::PW - 1) / cd::PW), ks, stride, cus);
}

template <typename TI, int CT, int KS>
static hipError_t launch_ks(const ConvDirectParams& p, dim3 grid, uint32_t lds, hipStream_t s)
{
    static PerDevice lds_once;
    const hipError_t e = set_max_lds(lds_once, (const void*)conv_direct_kernel<TI, CT, KS>, 160 * 1024);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((conv_direct_kernel<TI, CT, KS>), grid, dim3(cd::NT), lds, s, p);
    return hipGetLastError();
}

template <typename TI, int CT>
static hipError_t launch_ct(const ConvDirectParams& p, dim3 grid, uint32_t lds, hipStream_t s)
{
    return p.ks == 1 ? launch_ks<TI, CT, 1>(p, grid, lds, s)
         : p.ks == 3 ? launch_ks<TI, CT, 3>(p, grid, lds, s) : launch_ks<TI, CT, 0>(p, grid, lds, s);
}

hipError_t conv_direct_launch(ConvDirectParams p, int x_dt, hipStream_t s)
{
    int cus = 0;
    const hipError_t e = device_cus(&cus);
    if (e != hipSuccess) return e;
    const uint32_t ct = ct_of(p.co), ctiles = (p.co + ct - 1) / ct;
    p.ytiles = (p.ho + cd::ph_of(ct) - 1) / cd::ph_of(ct);
    const dim3 grid((p.wo + cd::PW - 1) / cd::PW, p.ytiles * ctiles, p.batch);
    // two workgroups on a CU where there are that many and 8 channels fit, else as many channels as one can hold
    const uint64_t wgs = (uint64_t)grid.x * grid.y * grid.z;
    p.cb = wgs > (uint64_t)cus ? block_of(p.ci, p.ks, p.stride, ct, 80 * 1024) : 0;
    if (!p.cb) p.cb = block_of(p.ci, p.ks, p.stride, ct, 160 * 1024);
    const cd::Plan q = cd::plan_of(p.cb, p.ks, p.stride, ct);
    const uint32_t lds = q.lds, kk = p.ks * p.ks;
    p.m_kk = cd::magic(kk);
    p.m_c8 = cd::magic(q.c8);
    p.m_nv = cd::magic(q.rw / 8);
    p.m_wv = cd::magic(p.ks == 3 ? p.cb : (p.cb * kk + 7) / 8);
    if (x_dt == DT_F16)
        return ct == 32 ? launch_ct<half_t, 32>(p, grid, lds, s) : launch_ct<half_t, 64>(p, grid, lds, s);
    return ct == 32 ? launch_ct<float, 32>(p, grid, lds, s) : launch_ct<float, 64>(p, grid, lds, s);
}

}   // namespace vai_dev
