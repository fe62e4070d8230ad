// lut_rvq.hip -- multi-stage residual-VQ LUT GEMM (the math engine's
// subspace_lut_rvq_gemm) and the codec's bit packing, on gfx950.
//
//   Y[b, m] = row_scales[m] * sum_{s, g} <X[b, g, :], C_s[code_s[m, g]]> + bias[m]
// with X zero-padded from `columns` to G * block columns, code_s the stage-s
// codes of vector v = m * G + g read from a little-endian bit stream of
// `bits` bits per code (bits in {1, 2, 4, 8}: code v sits at bit v * bits and
// never straddles a 32-bit word), and C_s the stage-s codebook [2^bits][block].
// This is ojasx_24x96/math_engine.py:136-208 with the packing of
// ojasx_24x96/codec.py:176-214; the reference's row_block_size only bounds
// its gather's working memory and has no counterpart here.
//
// lut_rvq_kernel (one or two fp32 tokens, and the shapes lut_rvq_mm_kernel below
// does not take): workgroup = 32 rows x 8 group sets; thread (q, r) owns row
// r and groups q, q+8, ...  Round trip 1 stages, with branch-free batched
// loads, the 32 rows' code words of every stage (one contiguous bit range per
// stage), all stage codebooks (when they fit) and x for up to 4 tokens in
// LDS.  Each thread then unpacks its codes from LDS, computes the dots
// <x_g, C_s[code]> from LDS and the 8 group-set partials are summed in LDS in
// a fixed order.  The epilogue is (scale * sum) + bias, stored in the input
// dtype.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "common.h"

namespace ojx {

namespace {
constexpr int kNT = 256;
constexpr int kR = 32;                   // rows per workgroup
constexpr int kQG = kNT / kR;            // group sets per row
constexpr int kMaxBT = 4;                // tokens per workgroup (at most)
constexpr size_t kMaxLds = 160 * 1024;
}  // namespace

struct RvqParams {
    const void *x;            // [B][columns]
    const uint8_t *packed;    // stage s at packed + s * stage_stride
    const float *cb;          // [S][Q][D]
    const float *scales;      // [rows]
    const float *bias;        // [rows] or null
    void *y;                  // [B][rows]
    size_t stage_stride;      // bytes between stages
    size_t stage_bytes;       // packed bytes per stage = ceil(rows * G * bits / 8)
    int B, columns, rows, S, bits, D, Q, G;
    int cb_lds;               // codebooks staged in LDS
    int words;                // LDS words per stage for one workgroup's rows
    uint32_t magic;           // e / D = umulhi(e, magic)
};

// 32-bit word w of a stage's bit stream, where the stream starts `off` bytes
// into the 4-byte-aligned pointer `base`; bytes at or past `end` (offset from
// base) read as zero.  Loads stay inside [base, base + end).
__device__ __forceinline__ uint32_t stream_word(const uint8_t *base, size_t end, long w) {
    const long b0 = w * 4;
    if (b0 + 4 <= (long)end && b0 >= 0) return *reinterpret_cast<const uint32_t *>(base + b0);
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const long b = b0 + i;
        if (b >= 0 && b < (long)end) v |= (uint32_t)base[b] << (8 * i);
    }
    return v;
}

// First bit of a workgroup's rows in stage s, counted from the stage's 4-byte
// aligned start.
__device__ __forceinline__ size_t stage_bit(const RvqParams &p, int s, int m0) {
    const uintptr_t sp = reinterpret_cast<uintptr_t>(p.packed) + (size_t)s * p.stage_stride;
    return (sp & 3) * 8 + (size_t)m0 * p.G * p.bits;
}

// The code words of rows m0 .. m0 + 31 into cw [S][words] (NT threads): of stage
// s the bits of vectors m0*G .. (m0+32)*G - 1; word 0 is the stream's word
// containing the first bit.
template <int NT>
__device__ __forceinline__ void stage_words(const RvqParams &p, int m0, uint32_t *cw, int tid) {
    const int n = p.S * p.words;
    for (int b = tid; b < n; b += 4 * NT) {
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = min(b + u * NT, n - 1), s = i / p.words;
            const uintptr_t sp = reinterpret_cast<uintptr_t>(p.packed) + (size_t)s * p.stage_stride;
            const long w0 = (long)(stage_bit(p, s, m0) >> 5);
            v[u] = stream_word(reinterpret_cast<const uint8_t *>(sp & ~uintptr_t(3)), (sp & 3) + p.stage_bytes,
                               w0 + (i - s * p.words));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) cw[min(b + u * NT, n - 1)] = v[u];
    }
}

template <typename T, int DT, int kBT>
__global__ __launch_bounds__(kNT) void lut_rvq_kernel(RvqParams p) {
    extern __shared__ float sm[];
    const int D = DT > 0 ? DT : p.D;
    const int GD = p.G * D;
    float *xs = sm;                                        // [kBT][G*D]
    float *cbs = xs + kBT * GD;                            // [S][Q][D] when cb_lds
    uint32_t *cw = reinterpret_cast<uint32_t *>(cbs + (p.cb_lds ? p.S * p.Q * D : 0));  // [S][words]
    __shared__ float red[kQG][kBT][kR];
    const int tid = threadIdx.x;
    const int r = tid % kR, q = tid / kR;
    const int m0 = blockIdx.x * kR;
    const int m = m0 + r;
    const int t0 = blockIdx.y * kBT;
    const int nt = min(kBT, p.B - t0);
    const T *__restrict__ x = static_cast<const T *>(p.x);

    // ---- round trip 1: x (zero past columns), codebooks, code words
    {
        const int n = kBT * GD;
        for (int b = tid; b < n; b += 4 * kNT) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = min(b + u * kNT, n - 1);
                const int t = min(i / GD, nt - 1), c = i - (i / GD) * GD;
                v[u] = c < p.columns ? load_act(x, (size_t)(t0 + t) * p.columns + c) : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) xs[min(b + u * kNT, n - 1)] = v[u];
        }
    }
    if (p.cb_lds) {
        const int n = p.S * p.Q * D;
        for (int b = tid; b < n; b += 4 * kNT) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = p.cb[min(b + u * kNT, n - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) cbs[min(b + u * kNT, n - 1)] = v[u];
        }
    }
    stage_words<kNT>(p, m0, cw, tid);
    __syncthreads();

    // ---- dots over this thread's groups and all stages
    float acc[kBT];
#pragma unroll
    for (int t = 0; t < kBT; ++t) acc[t] = 0.f;
    const uint32_t mask = (1u << p.bits) - 1u;
    for (int s = 0; s < p.S; ++s) {
        const uint8_t *sp = p.packed + (size_t)s * p.stage_stride;
        const size_t off = reinterpret_cast<uintptr_t>(sp) & 3;
        const size_t bit0 = off * 8 + (size_t)m0 * p.G * p.bits;   // stream bit of vector m0*G
        const size_t wbase = bit0 >> 5;
        const float *C = p.cb_lds ? cbs + (size_t)s * p.Q * D : p.cb + (size_t)s * p.Q * D;
        for (int g = q; g < p.G; g += kQG) {
            const size_t bit = bit0 + ((size_t)r * p.G + g) * p.bits;
            const uint32_t code = (cw[s * p.words + (int)((bit >> 5) - wbase)] >> (bit & 31)) & mask;
            const float *c = C + (size_t)code * D;
            const float *xg = xs + g * D;
            if (DT > 0) {
                float cr[DT > 0 ? DT : 1];
#pragma unroll
                for (int d = 0; d < D; ++d) cr[d] = c[d];
#pragma unroll
                for (int t = 0; t < kBT; ++t) {
                    float dot = 0.f;
#pragma unroll
                    for (int d = 0; d < D; ++d) dot = fmaf(xg[t * GD + d], cr[d], dot);
                    acc[t] += dot;
                }
            } else {
#pragma unroll
                for (int t = 0; t < kBT; ++t) {
                    float dot = 0.f;
                    for (int d = 0; d < D; ++d) dot = fmaf(xg[t * GD + d], c[d], dot);
                    acc[t] += dot;
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < kBT; ++t) red[q][t][r] = acc[t];
    __syncthreads();
    if (q != 0 || m >= p.rows) return;
    const float sc = p.scales[m];
    const float bs = p.bias ? p.bias[m] : 0.f;
    T *y = static_cast<T *>(p.y);
#pragma unroll
    for (int t = 0; t < kBT; ++t) {
        if (t >= nt) break;
        float a = red[0][t][r];
#pragma unroll
        for (int k = 1; k < kQG; ++k) a += red[k][t][r];
        float v = a * sc;
        if (p.bias) v += bs;
        store_act(y, (size_t)(t0 + t) * p.rows + m, v);
    }
}

// lut_rvq_mm_kernel: the same product on v_mfma_f32_32x32x16_bf16, for block
// sizes 4 and multiples of 8 whose split codebooks fit the LDS: workgroup = 32
// rows x 32 TT tokens, the input split over its 8 waves 16 dims at a time.  A
// wave's A operand is x itself (each lane 8 dims of one token straight from
// memory, kRvqAhead chunks ahead: no other wave of the workgroup reads them, so
// nothing is staged and the loop has no barrier), its B operand 8 values of a
// row, one LDS read per piece at the row's code, for every stage.  Both sides as
// exact bf16 pieces (x of type bf16: one): the six (three) products with
// i + j <= 4, accumulated in fp32 smallest first, two chunks of a stage to a fresh
// tile that is then added to the wave's sums; the 8 partial tiles meet in LDS in wave
// order.
// What bounds it: LDS reads of random codebook rows and the MFMAs of a padded
// token tile, behind one staging round trip.  The kernel above reads a codebook
// row for 4 tokens and runs the dots on the VALU: 6912 x 2560, two 8-bit stages
// of block 16, 32 tokens 383 us against 23 here (bf16 x 410 against 19), 128
// tokens 1474 against 82; error against 64 bits 1.34e-7 (1.63e-7 above).
namespace {
constexpr int kRvqNT = 512, kRvqWaves = kRvqNT / 64;
constexpr int kRvqAhead = 2;             // chunk pairs of x in flight per wave
}  // namespace

template <typename T, int TT, bool B4>
__global__ __launch_bounds__(kRvqNT) void lut_rvq_mm_kernel(RvqParams p) {
    constexpr bool BF = !std::is_same<T, float>::value;
    constexpr int PX = BF ? 1 : 3;
    extern __shared__ __align__(16) unsigned char smb[];
    // [stage][piece][code][D] bf16, then the stages' code words; the partial
    // tiles at the end
    const int cbn = p.Q * p.D;                       // values of a stage's codebook
    __bf16 *cbs = reinterpret_cast<__bf16 *>(smb);
    uint32_t *cw = reinterpret_cast<uint32_t *>(smb + (size_t)p.S * 3 * cbn * 2);
    const int tid = threadIdx.x, lane = tid & 63, q = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, n = lane & 31;
    const int m0 = blockIdx.x * kR, t0 = blockIdx.y * 32 * TT;
    const int chunks = (p.G * p.D + 15) / 16;
    const T *x = static_cast<const T *>(p.x);

    // ---- x: chunk c of token tile t (dims past columns are zero).  Rows may
    // start at any element, so these are unaligned 16-byte loads; the chunk
    // that ends past the row is read element by element
    typedef unsigned int v4u __attribute__((ext_vector_type(4), aligned(2)));
    struct Raw { v4u v[BF ? 1 : 2]; };
    const T *xrow[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) xrow[t] = x + (size_t)min(t0 + 32 * t + n, p.B - 1) * p.columns;
    auto load_x = [&](int c, int t) __attribute__((always_inline)) {
        Raw r;
        const int e = 16 * c + 8 * h;
        if (16 * c + 16 <= p.columns) {
            typedef __attribute__((address_space(1))) const v4u global_t;
            const uintptr_t src = reinterpret_cast<uintptr_t>(xrow[t] + e);
#pragma unroll
            for (int i = 0; i < (BF ? 1 : 2); ++i) r.v[i] = *reinterpret_cast<global_t *>(src + 16 * i);
        } else {
            T v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = xrow[t][min(e + i, p.columns - 1)];
            __builtin_memcpy(&r, v, sizeof(v));
        }
        return r;
    };
    auto pieces = [&](int c, const Raw &r, bf16x8_t (&a)[PX]) __attribute__((always_inline)) {
        const int e = 16 * c + 8 * h;
        T v[8];
        __builtin_memcpy(v, &r, sizeof(v));
        if constexpr (BF) {
            uint16_t w[8];
            __builtin_memcpy(w, v, sizeof(w));
#pragma unroll
            for (int i = 0; i < 8; ++i) w[i] = e + i < p.columns ? w[i] : (uint16_t)0;
            __builtin_memcpy(&a[0], w, sizeof(w));
        } else {
            float f[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = e + i < p.columns ? v[i] : 0.f;
            split3_trunc(f, a);
        }
    };
    Raw xr[kRvqAhead][2][TT];
#pragma unroll
    for (int u = 0; u < kRvqAhead; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < TT; ++t)
                xr[u][i][t] = load_x(min(2 * (q + u * kRvqWaves) + i, chunks - 1), t);

    // ---- codebooks split into LDS, 4 values per thread and round; code words
    {
        const int n4 = p.S * cbn / 4, per = cbn / 4;
        for (int b = tid; b < n4; b += 4 * kRvqNT) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float *src = p.cb + 4 * (size_t)min(b + u * kRvqNT, n4 - 1);
                v[u] = make_float4(src[0], src[1], src[2], src[3]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = min(b + u * kRvqNT, n4 - 1), st = i / per;
                const float f[8] = {v[u].x, v[u].y, v[u].z, v[u].w, 0.f, 0.f, 0.f, 0.f};
                bf16x8_t pc[3];
                split3_bf16(f, pc);
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    __builtin_memcpy(cbs + ((size_t)(st * 3 + k) * cbn + 4 * (i - st * per)), &pc[k], 8);
            }
        }
    }
    stage_words<kRvqNT>(p, m0, cw, tid);
    __syncthreads();

    // ---- the wave's chunk pairs q, q + 8, ...
    f32x16_t acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = f32x16_t{};
    const uint32_t mask = (1u << p.bits) - 1u;
    auto pair = [&](const int pr, const int u) __attribute__((always_inline)) {
        bf16x8_t a[2][TT][PX];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < TT; ++t) pieces(2 * pr + i, xr[u][i][t], a[i][t]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < TT; ++t)
                xr[u][i][t] = load_x(min(2 * (pr + kRvqAhead * kRvqWaves) + i, chunks - 1), t);
        for (int s = 0; s < p.S; ++s) {
            const uint32_t *w = cw + s * p.words;
            const uint32_t b0 = stage_bit(p, s, m0) & 31u;
            auto code = [&](int g) __attribute__((always_inline)) {
                const uint32_t bit = b0 + (uint32_t)(n * p.G + min(g, p.G - 1)) * p.bits;
                return (w[bit >> 5] >> (bit & 31u)) & mask;
            };
            bf16x8_t b[2][3];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int e = 16 * (2 * pr + i) + 8 * h;
                if constexpr (B4) {
                    const uint32_t c0 = code(e >> 2), c1 = code((e >> 2) + 1);
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const __bf16 *src = cbs + (size_t)(s * 3 + k) * cbn;
                        uint2 lo, hi;
                        __builtin_memcpy(&lo, __builtin_assume_aligned(src + c0 * 4, 8), 8);
                        __builtin_memcpy(&hi, __builtin_assume_aligned(src + c1 * 4, 8), 8);
                        const uint4 v = make_uint4(lo.x, lo.y, hi.x, hi.y);
                        __builtin_memcpy(&b[i][k], &v, 16);
                    }
                } else {
                    const int g = __umulhi((uint32_t)e, p.magic);   // e / D
                    const uint32_t at = code(g) * p.D + (e - g * p.D);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        b[i][k] = *reinterpret_cast<const bf16x8_t *>(cbs + (size_t)(s * 3 + k) * cbn + at);
                }
            }
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                f32x16_t d = {};
                // the products x piece j of codebook piece k, smallest first
                auto both = [&](int j, int k) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][t][j], b[i][k], d, 0, 0, 0);
                };
                both(0, 2);
                if constexpr (!BF) {
                    both(1, 1);
                    both(2, 0);
                }
                both(0, 1);
                if constexpr (!BF) both(1, 0);
                both(0, 0);
                acc[t] += d;
            }
        }
    };
    // pairs past the last chunk read clamped x and codes and add nothing: the
    // first dim of a chunk >= chunks is past columns, so its pieces are zero
    const int pairs = (chunks + 1) / 2;
    int pr = q;
    for (; pr + (kRvqAhead - 1) * kRvqWaves < pairs; pr += kRvqAhead * kRvqWaves)
#pragma unroll
        for (int u = 0; u < kRvqAhead; ++u) pair(pr + u * kRvqWaves, u);
#pragma unroll
    for (int u = 0; u < kRvqAhead - 1; ++u)
        if (pr + u * kRvqWaves < pairs) pair(pr + u * kRvqWaves, u);

    // ---- partial tiles through LDS; thread: (value v, lane) of the tile
    __syncthreads();
    float *red = reinterpret_cast<float *>(smb);     // [TT][wave][16][64]
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) red[((t * kRvqWaves + q) * 16 + v) * 64 + lane] = acc[t][v];
    __syncthreads();
    const int m = m0 + n;
    if (m >= p.rows) return;
    const float sc = p.scales[m];
    const float bs = p.bias ? p.bias[m] : 0.f;
    T *y = static_cast<T *>(p.y);
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16 / kRvqWaves; ++i) {
            const int v = q * (16 / kRvqWaves) + i;
            const int b = t0 + 32 * t + 8 * (v >> 2) + 4 * h + (v & 3);
            if (b >= p.B) continue;
            const float *src = red + (t * kRvqWaves * 16 + v) * 64 + lane;
            float a = src[0];
#pragma unroll
            for (int k = 1; k < kRvqWaves; ++k) a += src[k * 16 * 64];
            // an infinite or NaN x or codebook value has no pieces
            if (!(fabsf(a) < INFINITY)) {
                a = 0.f;
                for (int s = 0; s < p.S; ++s) {
                    const uint8_t *sp = p.packed + (size_t)s * p.stage_stride;
                    for (int e = 0; e < p.columns; ++e) {
                        const int g = __umulhi((uint32_t)e, p.magic);
                        const size_t bit = ((size_t)m * p.G + g) * p.bits;
                        const uint32_t code = (sp[bit >> 3] >> (bit & 7)) & mask;
                        a = fmaf(load_act(x, (size_t)b * p.columns + e),
                                 p.cb[((size_t)s * p.Q + code) * p.D + (e - g * p.D)], a);
                    }
                }
            }
            float r = a * sc;
            if (p.bias) r += bs;
            store_act(y, (size_t)b * p.rows + m, r);
        }
}

// codes[i] (uint8, < 2^bits) -> little-endian bit stream, one output byte per thread.
__global__ __launch_bounds__(kNT) void pack_codes_kernel(const uint8_t *codes, long count, int bits,
                                                         uint8_t *packed, long nbytes) {
    const long i = (long)blockIdx.x * kNT + threadIdx.x;
    if (i >= nbytes) return;
    const int per = 8 / bits;
    uint32_t v = 0;
    for (int k = 0; k < per; ++k) {
        const long c = i * per + k;
        if (c < count) v |= ((uint32_t)codes[c] & ((1u << bits) - 1u)) << (k * bits);
    }
    packed[i] = (uint8_t)v;
}

__global__ __launch_bounds__(kNT) void unpack_codes_kernel(const uint8_t *packed, long count, int bits,
                                                           uint8_t *codes) {
    const long i = (long)blockIdx.x * kNT + threadIdx.x;
    if (i >= count) return;
    const long bit = i * bits;
    codes[i] = (uint8_t)((packed[bit >> 3] >> (bit & 7)) & ((1u << bits) - 1u));
}

namespace {

bool valid_bits(int bits) { return bits == 1 || bits == 2 || bits == 4 || bits == 8; }

template <typename T, int TT, bool B4>
int launch_rvq_mm_k(const RvqParams &p, size_t lds, hipStream_t st) {
    static size_t granted = 0;
    const void *fn = reinterpret_cast<const void *>(&lut_rvq_mm_kernel<T, TT, B4>);
    int rc = ensure_dyn_lds(fn, lds, &granted);
    if (rc) return rc;
    dim3 grid((p.rows + kR - 1) / kR, (p.B + 32 * TT - 1) / (32 * TT));
    OJX_LAUNCH((lut_rvq_mm_kernel<T, TT, B4>), grid, dim3(kRvqNT), lds, st, p);
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

// The MFMA kernel where it takes the call and is the faster one; 1 otherwise.
// fp32 x of one or two tokens with block 8 or 16 stays on the VALU kernel (us,
// that one against this: 6912 x 2560, two stages of 8 bits, block 16: 1 token
// 19.2 / 24.0, 2 tokens 22.2 / 24.3, 4 tokens 56.8 / 24.1; one stage 11.2 / 16.3,
// 13.7 / 16.4, 31.9 / 16.8; 512 x 1003, block 8, 4 bits, two stages 7.7 / 9.9,
// 9.5 / 9.9, 13.2 / 10.1), which holds the staged codebook rows conflict-free
// there; bf16 x stays for one token and one stage (12.0 / 12.4; two stages 20.1
// / 17.8).  Two token
// tiles per workgroup once single ones fill the CUs (432 workgroups at 64 tokens
// and 6912 rows: bf16 26.5 against 30.7 us, fp32 42.1 against 43.3; 32 at 512
// rows: 23.8 against 13.0).
template <typename T>
int try_rvq_mm(RvqParams &p, bool cb_lds, hipStream_t st) {
    if (p.D != 4 && p.D % 8) return 1;
    const int few = std::is_same<T, float>::value ? 2 : p.S == 1 ? 1 : 0;
    if (p.B <= few && (p.D == 8 || p.D == 16) && cb_lds) return 1;
    const size_t staged = (size_t)p.S * 3 * p.Q * p.D * 2 + (size_t)p.S * p.words * sizeof(uint32_t);
    const long tiles = (long)((p.rows + kR - 1) / kR) * ((p.B + 31) / 32);
    const int tt = p.B > 32 && tiles > 256 ? 2 : 1;
    const size_t lds = std::max(staged, (size_t)tt * kRvqWaves * 16 * 64 * sizeof(float));
    if (lds > kMaxLds) return 1;
    p.magic = (uint32_t)(((1ull << 32) + p.D - 1) / p.D);
    if (p.D == 4) return tt == 1 ? launch_rvq_mm_k<T, 1, true>(p, lds, st) : launch_rvq_mm_k<T, 2, true>(p, lds, st);
    return tt == 1 ? launch_rvq_mm_k<T, 1, false>(p, lds, st) : launch_rvq_mm_k<T, 2, false>(p, lds, st);
}

template <typename T, int DT, int BT>
int launch_rvq_bt(RvqParams &p, size_t lds, hipStream_t st) {
    static size_t granted = 0;
    const void *fn = reinterpret_cast<const void *>(&lut_rvq_kernel<T, DT, BT>);
    int rc = ensure_dyn_lds(fn, lds, &granted);
    if (rc) return rc;
    dim3 grid((p.rows + kR - 1) / kR, (p.B + BT - 1) / BT);
    OJX_LAUNCH((lut_rvq_kernel<T, DT, BT>), grid, dim3(kNT), lds, st, p);
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

template <typename T, int DT>
int launch_rvq_d(RvqParams &p, int bt, size_t lds, hipStream_t st) {
    if (bt == 4) return launch_rvq_bt<T, DT, 4>(p, lds, st);
    if (bt == 2) return launch_rvq_bt<T, DT, 2>(p, lds, st);
    return launch_rvq_bt<T, DT, 1>(p, lds, st);
}

template <typename T>
int launch_rvq(RvqParams &p, int bt, size_t lds, hipStream_t st) {
    switch (p.D) {
        case 4: return launch_rvq_d<T, 4>(p, bt, lds, st);
        case 8: return launch_rvq_d<T, 8>(p, bt, lds, st);
        case 16: return launch_rvq_d<T, 16>(p, bt, lds, st);
        default: return launch_rvq_d<T, 0>(p, bt, lds, st);
    }
}

}  // namespace
}  // namespace ojx

extern "C" {

OJASX_API int ojasx_subspace_lut_gemm_device(const void *x, int batch, int columns, int rows,
                                             const uint8_t *packed_codes, size_t stage_stride_bytes,
                                             int stages, int bits, int block_size,
                                             const float *codebooks, const float *row_scales,
                                             const float *bias, void *y, int dtype, void *stream) {
    using namespace ojx;
    if (!x || !packed_codes || !codebooks || !row_scales || !y) return OJASX_ERR_NULL;
    if (batch <= 0 || rows <= 0) return OJASX_OK;
    if (columns <= 0 || stages <= 0 || !valid_bits(bits) || block_size <= 0 || block_size > 64) {
        set_error("invalid LUT GEMM shape: columns=%d stages=%d bits=%d block=%d", columns, stages,
                  bits, block_size);
        return OJASX_ERR_INVALID;
    }
    if (dtype != OJASX_DTYPE_F32 && dtype != OJASX_DTYPE_BF16) {
        set_error("unsupported dtype %d", dtype);
        return OJASX_ERR_INVALID;
    }
    if ((long)batch > 65535L) {
        set_error("batch %d too large for one call", batch);
        return OJASX_ERR_INVALID;
    }
    RvqParams p{};
    p.x = x;
    p.packed = packed_codes;
    p.cb = codebooks;
    p.scales = row_scales;
    p.bias = bias;
    p.y = y;
    p.B = batch;
    p.columns = columns;
    p.rows = rows;
    p.S = stages;
    p.bits = bits;
    p.D = block_size;
    p.Q = 1 << bits;
    p.G = (columns + block_size - 1) / block_size;
    p.stage_stride = stage_stride_bytes;
    p.stage_bytes = ((size_t)rows * p.G * bits + 7) / 8;
    if (stages > 1 && stage_stride_bytes < p.stage_bytes) {
        set_error("stage stride %zu below the %zu packed bytes of a stage", stage_stride_bytes,
                  p.stage_bytes);
        return OJASX_ERR_INVALID;
    }
    // code words of kR rows per stage, plus one for the unaligned start
    p.words = (int)(((size_t)kR * p.G * bits + 31) / 32 + 2);
    hipStream_t st = static_cast<hipStream_t>(stream);
    // tokens per workgroup: 4, or fewer when x of 4 tokens and the code words
    // do not fit the LDS; codebooks are staged when they still fit
    const size_t xrow = (size_t)p.G * block_size * sizeof(float);
    const size_t cwb = (size_t)stages * p.words * sizeof(uint32_t);
    const size_t cbb = (size_t)stages * p.Q * block_size * sizeof(float);
    int bt = std::min(batch, kMaxBT) >= 3 ? 4 : std::min(batch, kMaxBT);
    while (bt > 1 && bt * xrow + cwb > kMaxLds) bt /= 2;
    if (bt * xrow + cwb > kMaxLds) {
        set_error("LUT GEMM of %d columns x %d stages does not fit the 160 KB LDS", columns, stages);
        return OJASX_ERR_INVALID;
    }
    p.cb_lds = bt * xrow + cwb + cbb <= kMaxLds;
    const int rc = dtype == OJASX_DTYPE_F32 ? try_rvq_mm<float>(p, p.cb_lds, st)
                                            : try_rvq_mm<__hip_bfloat16>(p, p.cb_lds, st);
    if (rc != 1) return rc;
    const size_t lds = bt * xrow + cwb + (p.cb_lds ? cbb : 0);
    return dtype == OJASX_DTYPE_F32 ? launch_rvq<float>(p, bt, lds, st)
                                    : launch_rvq<__hip_bfloat16>(p, bt, lds, st);
}

OJASX_API int ojasx_pack_codes_device(const uint8_t *codes, long count, int bits, uint8_t *packed,
                                      void *stream) {
    using namespace ojx;
    if (!codes || !packed) return OJASX_ERR_NULL;
    if (!valid_bits(bits) || count < 0) {
        set_error("bits must be 1, 2, 4 or 8");
        return OJASX_ERR_INVALID;
    }
    const long nbytes = (count * bits + 7) / 8;
    if (nbytes == 0) return OJASX_OK;
    OJX_LAUNCH(pack_codes_kernel, dim3((nbytes + kNT - 1) / kNT), dim3(kNT), 0,
               static_cast<hipStream_t>(stream), codes, count, bits, packed, nbytes);
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

OJASX_API int ojasx_unpack_codes_device(const uint8_t *packed, long count, int bits, uint8_t *codes,
                                        void *stream) {
    using namespace ojx;
    if (!codes || !packed) return OJASX_ERR_NULL;
    if (!valid_bits(bits) || count < 0) {
        set_error("bits must be 1, 2, 4 or 8");
        return OJASX_ERR_INVALID;
    }
    if (count == 0) return OJASX_OK;
    OJX_LAUNCH(unpack_codes_kernel, dim3((count + kNT - 1) / kNT), dim3(kNT), 0,
               static_cast<hipStream_t>(stream), packed, count, bits, codes);
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

}  // extern "C"
