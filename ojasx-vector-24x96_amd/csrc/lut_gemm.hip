// lut_gemm.hip -- the LUT linear (block_dim 16, 256 centroids) for prefill
// batches: y = x . W^T as a tiled matrix product whose weight operand is
// decoded from the codes in LDS.
//
// y[b][m] = (s_m * sum_g <x_b[16g ..], C[codes[m, g]]> + bias_m) + sum_j val_j x_b[col_j]
// (ojasx_lut_cpu.cpp:132-206), the sum over groups as v_mfma_f32_32x32x16: one
// group per MFMA, A = 32 tokens of x, B = 32 weight rows.  A lane's B operand
// (8 values of its row) is one 16-byte LDS read of the codebook at the row's
// code, so the weights never exist in memory.
//
// What bounds it: the matrix cores, and close behind them the LDS (the codebook
// reads are random rows: about three times the cycles of an ordered read).  A
// wave holds WT token tiles x WR row tiles, so a codebook read feeds WT MFMAs
// and a read of x WR; lut_mm32_kernel (32 rows x 64 tokens per workgroup, every
// operand feeding at most two MFMAs, x split in every workgroup) is bound by
// the LDS and the VALU from about 100 tokens on.
//
// Products per multiply-add, both sides as exact bf16 pieces (bf16 keeps fp32's
// exponent, so a value of any size beside any other is held whole):
//  * kBf1: bf16 x and a codebook whose values are bf16: one, exact.
//  * kBf3: bf16 x, fp32 codebook C = c1 + c2 + c3: three, exact.
//  * kBf6: fp32 x = x1 + x2 + x3: the six products x_i c_j with i + j <= 4, as
//    lut_mm32_kernel's; the three left out are below 2^-22 of the term.
// The sums are fp32 in the accumulators.
//
// The pieces of fp32 x (K padded to 64 with zeros) and, where the layer has
// outliers, x transposed are written by gemm_prep_kernel into scratch of the
// calling thread and stream.  Outliers: after the K loop the waves take the
// tile's rows in turn, a lane holding BT / 64 neighbouring tokens: an entry is
// one coalesced read of x^T and BT / 64 FMAs, sixteen entries' reads in flight;
// the sums cross to the accumulators' layout through LDS.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "lut_gemm_x.h"

namespace ojx {

namespace {
enum { kBf1 = 1, kBf3 = 3, kBf6 = 6 };
constexpr int kGK = kGemmStep;      // input dims per step: four groups
constexpr long kGemmCUs = 256;
constexpr size_t kGemmScratch = size_t(256) << 20;   // scratch bytes per pass over tokens

typedef int i32x4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16), aligned(4)));
// A wave-uniform load of data no kernel writes: a scalar load wherever it stands.
template <typename V>
__device__ __forceinline__ V uld(const V *p) {
    typedef __attribute__((address_space(4))) const V const_t;
    return *reinterpret_cast<const_t *>(reinterpret_cast<uintptr_t>(p));
}

struct GemmParams {
    const uint8_t *codes;           // [S][Mp][16]
    const void *cb;                 // kBf1: bf16 [half][256][8]; else the pieces (split_codebook_bf16x3)
    const float *scales, *bias;
    const int *gptr, *orow, *ocol;  // outlier groups (LinearGemm) or null
    const float *oval;
    const void *x;                  // bf16 x: [B][K]; fp32 x: its pieces [3][Bp][Kp] in bf16
    const void *xt;                 // [K + 1][Bp] x transposed (outliers), row K zero
    void *y;                        // [B][M]
    int K, Kp, M, Mp, B, Bp;
    int nr, nt, n_tiles;            // row tiles, token tiles, their product
};
}  // namespace

// Tokens per tile BT = 32 WT NWT, rows per tile BR = 32 WR NWR; NWT x NWR waves.
template <typename T, int PROD, int WT, int WR, int NWT, int NWR, int PXD>
__global__ __launch_bounds__(64 * NWT * NWR) __attribute__((amdgpu_waves_per_eu(2))) void lut_gemm_kernel(GemmParams p) {
    constexpr int NW = NWT * NWR, NT = 64 * NW;
    constexpr int BT = 32 * WT * NWT, BR = 32 * WR * NWR;
    constexpr int PX = PROD == kBf6 ? 3 : 1, PC = PROD == kBf1 ? 1 : 3;
    constexpr int XU = BT * 8 / NT;                  // 16-byte units of a step's plane per thread
    constexpr int PB = BT * 128;                     // bytes of a step's plane
    constexpr int CB = 256 * 32;                     // bytes of a codebook piece
    constexpr int OT = BT >= 128 ? BT / 64 : 2;      // tokens per lane of an outlier read
    static_assert(BT % 64 == 0 && (BT * 8) % NT == 0 && NT % 8 == 0, "tile shapes");
    extern __shared__ __align__(16) unsigned char sm[];
    unsigned char *cbs = sm;                         // [piece][half][256][16 bytes]
    unsigned char *xs = sm + PC * CB;                // [2 buffers][PX][BT][128 bytes]
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, n = lane & 31;
    const int wt = w % NWT, wr = w / NWT;
    // Tiles in row-fastest order, each XCD (workgroup id mod 8) a contiguous
    // run of them: an XCD's workgroups share few token tiles of x in its L2.
    const int per = (p.n_tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= p.n_tiles || (int)(blockIdx.x >> 3) >= per) return;
    const int b0 = (tile / p.nr) * BT, m0 = (tile % p.nr) * BR;

    // ---- codebook into LDS, [centroid][half][piece] to piece planes
    {
        constexpr int NU = PC * CB / 16;
        const uint4 *src = static_cast<const uint4 *>(p.cb);
#pragma unroll
        for (int i = 0; i < (NU + NT - 1) / NT; ++i) {
            const int u = min(tid + i * NT, NU - 1);
            const int to = PC == 1 ? u : u % PC * 512 + u / PC % 2 * 256 + u / (2 * PC);
            reinterpret_cast<uint4 *>(cbs)[to] = gld(src + u);
        }
    }
    // ---- x staging: unit i of a plane = (token i / 8, dims 8 (i % 8) ..) of
    // the step; a token's 8 units are swizzled by (token / 2) % 8, so the 16
    // tokens a fragment read covers per phase fall in all 16 four-bank groups
    constexpr int ROWB = PROD == kBf6 ? 1 : 0;       // planes are padded, bf16 x is not
    const unsigned char *xb = static_cast<const unsigned char *>(p.x);
    size_t xoff[XU];
    int xst[XU];
    const size_t pitch = (size_t)(ROWB ? p.Kp : p.K) * 2;
    const int xc = tid & 7;                          // NT % 8 == 0: the same for each of its units
#pragma unroll
    for (int i = 0; i < XU; ++i) {
        const int t = (tid + i * NT) >> 3;
        xoff[i] = (size_t)min(b0 + t, p.B - 1) * pitch;
        xst[i] = t * 128 + ((xc ^ ((t >> 1) & 7)) << 4);
    }
    const size_t plane = (size_t)p.Bp * p.Kp * 2;
    uint4 xr[PXD][PX][XU];
    auto load_x = [&](int s, uint4 (&xr)[PX][XU]) __attribute__((always_inline)) {
        const size_t o = gemm_x_unit(s, xc, ROWB ? p.Kp : p.K);
#pragma unroll
        for (int q = 0; q < PX; ++q)
#pragma unroll
            for (int i = 0; i < XU; ++i)
                xr[q][i] = gld(reinterpret_cast<const uint4 *>(xb + q * plane + xoff[i] + o));
    };
    auto store_x = [&](int s, uint4 (&xr)[PX][XU]) __attribute__((always_inline)) {
        unsigned char *dst = xs + (s & 1) * (PX * PB);
#pragma unroll
        for (int q = 0; q < PX; ++q)
#pragma unroll
            for (int i = 0; i < XU; ++i) {
                uint4 v = xr[q][i];
                if (!ROWB && s * kGK + 8 * xc >= p.K) v = make_uint4(0, 0, 0, 0);
                *reinterpret_cast<uint4 *>(dst + q * PB + xst[i]) = v;
            }
    };
    // ---- codes of the wave's rows: 4 bytes per row and step
    const uint8_t *cp[WR];
#pragma unroll
    for (int r = 0; r < WR; ++r)
        cp[r] = p.codes + (size_t)min(m0 + 32 * (wr * WR + r) + n, p.Mp - 1) * 16;
    auto load_codes = [&](int s, int r) __attribute__((always_inline)) {
        return gld(reinterpret_cast<const uint32_t *>(cp[r] + (size_t)(s >> 2) * p.Mp * 16 + (s & 3) * 4));
    };
    const int steps = (p.K + kGK - 1) / kGK;
    uint32_t cc[PXD + 1][WR];                        // codes of steps s .. s + PXD
    load_x(0, xr[0]);
#pragma unroll
    for (int u = 0; u <= PXD; ++u)
#pragma unroll
        for (int r = 0; r < WR; ++r) cc[u][r] = load_codes(min(u, steps - 1), r);
    store_x(0, xr[0]);
#pragma unroll
    for (int u = 0; u < PXD; ++u) load_x(min(u + 1, steps - 1), xr[u]);
    __syncthreads();

    f32x16_t acc[WT][WR];
#pragma unroll
    for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int r = 0; r < WR; ++r) acc[t][r] = f32x16_t{};
    // the lane's unit offsets of the step's four groups in a token's row
    int go[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) go[g] = ((2 * g + h) ^ ((n >> 1) & 7)) << 4;
    const unsigned char *ar = xs + (32 * wt * WT + n) * 128;
    const unsigned char *br = cbs + h * (CB / 2);
    // step s: x of step s + 1 from register set u = s % PXD to LDS, the set
    // refilled with step s + 1 + PXD (clamped: past the last step never stored)
    auto step = [&](const int s, const int u) __attribute__((always_inline)) {
        if (s + 1 < steps) store_x(s + 1, xr[u]);
        load_x(min(s + 1 + PXD, steps - 1), xr[u]);
        const unsigned char *xa = ar + (s & 1) * (PX * PB);
        // kBf6: a step's products into fresh tiles, then added to the sums:
        // one rounding of the running sum per step instead of 24
        f32x16_t d[WT][WR];
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
            for (int r = 0; r < WR; ++r) {
                if constexpr (PROD == kBf6) d[t][r] = f32x16_t{};
                else d[t][r] = acc[t][r];
            }
        // group g's products x piece i of codebook piece j with i + j = k for k
        // from HI down to LO, smallest first; every tile before the next product,
        // so that neighbouring MFMAs do not wait for each other
        auto group = [&](const int g, auto hi, auto lo) __attribute__((always_inline)) {
            constexpr int HI = decltype(hi)::value, LO = decltype(lo)::value, NX = PX > 1 ? HI + 1 : 1;
            bf16x8_t a[NX][WT], b[HI + 1][WR];
#pragma unroll
            for (int r = 0; r < WR; ++r)
#pragma unroll
                for (int q = 0; q <= HI; ++q)
                    b[q][r] = *reinterpret_cast<const bf16x8_t *>(
                        br + q * CB + ((cc[0][r] >> (8 * g)) & 0xffu) * 16);
#pragma unroll
            for (int t = 0; t < WT; ++t)
#pragma unroll
                for (int q = 0; q < NX; ++q)
                    a[q][t] = *reinterpret_cast<const bf16x8_t *>(xa + q * PB + t * (32 * 128) + go[g]);
#pragma unroll
            for (int k = HI; k >= LO; --k)
#pragma unroll
                for (int i = 0; i <= (PX > 1 ? k : 0); ++i)
#pragma unroll
                    for (int t = 0; t < WT; ++t)
#pragma unroll
                        for (int r = 0; r < WR; ++r)
                            d[t][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][t], b[k - i][r], d[t][r],
                                                                              0, 0, 0);
        };
        constexpr std::integral_constant<int, PC - 1> top{};
        constexpr std::integral_constant<int, 0> first{};
        if constexpr (PROD == kBf6) {
            // the step's small products before its large ones (the compiler
            // holds these operands in registers over the step): the large
            // partial sums are rounded four times instead of twenty.  Error against 64 bits 1.09e-7 -> 9.3e-8 at 2560
            // inputs, 1.74e-7 -> 1.61e-7 at 9728, 8.0e-8 -> 5.9e-8 at 512, for
            // 0 to 1 % of the time (4 % at 9728 -> 2560 and 256 tokens)
#pragma unroll
            for (int g = 0; g < 4; ++g) group(g, top, std::integral_constant<int, 1>{});
#pragma unroll
            for (int g = 0; g < 4; ++g) group(g, first, first);
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) group(g, top, first);
        }
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
            for (int r = 0; r < WR; ++r) {
                if constexpr (PROD == kBf6) acc[t][r] += d[t][r];
                else acc[t][r] = d[t][r];
            }
#pragma unroll
        for (int r = 0; r < WR; ++r) {
#pragma unroll
            for (int k = 0; k < PXD; ++k) cc[k][r] = cc[k + 1][r];
            cc[PXD][r] = load_codes(min(s + 1 + PXD, steps - 1), r);
        }
        __syncthreads();   // step s + 1 staged; step s's reads done before its buffer is rewritten
    };
    int s0 = 0;
    for (; s0 + PXD <= steps; s0 += PXD)
#pragma unroll
        for (int u = 0; u < PXD; ++u) step(s0 + u, u);
#pragma unroll
    for (int u = 0; u < PXD - 1; ++u)
        if (s0 + u < steps) step(s0 + u, u);

    // ---- epilogue: (s_m * sum + bias) + outliers, OR rows of each row
    // group's tiles per round
    constexpr int OP = BT + 4;                       // floats per row of outlier sums
    float *os = reinterpret_cast<float *>(sm);       // [NWR][32][OP]
    const T *xt = static_cast<const T *>(p.xt);
    T *y = static_cast<T *>(p.y);
#pragma unroll
    for (int r = 0; r < WR; ++r) {
        if (p.gptr) {
            // rows 32 (q WR + r) + i of the tile, q < NWR, i < 32: NWR * 32 rows
            // over NW waves, 32 / NWT consecutive rows each
            if (r) __syncthreads();                  // the last round's sums are read
            constexpr int RW = 32 / NWT;
            const int q = w / NWT, i0 = (w % NWT) * RW;
            const int mr = m0 + 32 * (q * WR + r) + i0;
            const int rlim = min(RW, p.M - mr);
            if (rlim > 0) {
                // The rows' outlier groups (four entries of one row each) in
                // order, four groups per batch, without a branch per entry: a
                // batch's columns, values and group rows are scalar loads, the
                // reads of x^T of two batches are in flight, and after each
                // group the row's running sum goes to LDS (the last one stays).
                constexpr int OU = 16;
                typedef unsigned int vu_t __attribute__((ext_vector_type(OT * sizeof(T) / 4)));
                const unsigned char *xl = reinterpret_cast<const unsigned char *>(xt + b0);
                const int ol = lane & (BT / OT - 1);     // 64 tokens: both half-waves read them
                const uint32_t lo = OT * sizeof(T) * ol, cpitch = p.Bp * sizeof(T);
                const int g0 = uld(p.gptr + mr), g1 = uld(p.gptr + mr + rlim);
                float *od = os + (size_t)(q * 32 + i0) * OP + OT * ol;
                float o[OT];
#pragma unroll
                for (int j = 0; j < OT; ++j) o[j] = 0.f;
                vu_t xq[2][OU];
                f32x16_t vq[2];
                i32x4_t iq[2];
                auto load_out = [&](int g, int k) __attribute__((always_inline)) {
                    const int gs = min(g, g1);       // past the end: the slack's groups, not added
                    const i32x16_t c = uld(reinterpret_cast<const i32x16_t *>(p.ocol + 4 * gs));
                    vq[k] = uld(reinterpret_cast<const f32x16_t *>(p.oval + 4 * gs));
                    iq[k] = uld(reinterpret_cast<const i32x4_t *>(p.orow + gs));
#pragma unroll
                    for (int u = 0; u < OU; ++u)
                        xq[k][u] = gld(reinterpret_cast<const vu_t *>(xl + (size_t)((uint32_t)c[u] * cpitch) + lo));
                };
                auto add_out = [&](int g, int k) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        // a group's row, with bit 31 set in the row's first group
                        const bool first = iq[k][i] < 0;
                        const int at = ((iq[k][i] & 0x7fffffff) - mr) * OP;
#pragma unroll
                        for (int j = 0; j < OT; ++j) o[j] = first ? 0.f : o[j];
#pragma unroll
                        for (int u = 4 * i; u < 4 * i + 4; ++u)
#pragma unroll
                            for (int j = 0; j < OT; ++j) {
                                uint32_t bits;
                                if constexpr (std::is_same<T, float>::value) bits = xq[k][u][j];
                                else bits = j % 2 ? xq[k][u][j / 2] & 0xffff0000u : xq[k][u][j / 2] << 16;
                                o[j] = fmaf(vq[k][u], __uint_as_float(bits), o[j]);
                            }
                        if (g + i < g1)
#pragma unroll
                            for (int j = 0; j < OT; ++j) od[at + j] = o[j];
                    }
                };
                load_out(g0, 0);
                for (int g = g0; g < g1; g += 8) {
                    load_out(g + 4, 1);
                    add_out(g, 0);
                    load_out(g + 8, 0);
                    add_out(g + 4, 1);
                }
            }
            __syncthreads();
        }
        const int m = m0 + 32 * (wr * WR + r) + n;
        const bool ok = m < p.M;
        const float sc = ok ? gld(p.scales + m) : 0.f;
        const float bs = ok && p.bias ? gld(p.bias + m) : 0.f;
        const float *orow = os + (size_t)(wr * 32 + n) * OP + 32 * wt * WT;
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
                const int tk = 32 * t + 8 * v4 + 4 * h;  // token within the wave's tiles, + j
                const int b = b0 + 32 * wt * WT + tk;
                float o4[4] = {0.f, 0.f, 0.f, 0.f};
                if (p.gptr) {
                    const float4 f = *reinterpret_cast<const float4 *>(orow + tk);
                    o4[0] = f.x; o4[1] = f.y; o4[2] = f.z; o4[3] = f.w;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (!ok || b + j >= p.B) continue;
                    float yv = acc[t][r][4 * v4 + j] * sc;
                    if (p.bias) yv += bs;
                    store_act(y, (size_t)(b + j) * p.M + m, yv + o4[j]);
                }
            }
    }
}

// 64 tokens x 64 dims: the pieces of fp32 x (PX 3; zero from K to Kp) and x
// transposed.
template <typename T, int PX, bool XT>
__global__ __launch_bounds__(256) void gemm_prep_kernel(const T *x, int B, int K, int Kp, int Bp,
                                                       uint16_t *planes, T *xt) {
    __shared__ T ts[64][72];                         // [dim][token], XT only
    const int k0 = blockIdx.x * 64, b0 = blockIdx.y * 64, tid = threadIdx.x;
    // thread: tokens tid / 8 + 32 i, dims 8 (tid % 8) ..
    const int k = k0 + 8 * (tid & 7);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int tl = (tid >> 3) + 32 * i, b = b0 + tl;
        const bool in = k < K && b < B;              // K % 16 == 0: 8 dims are in or out
        float v[8];
        const float4 lo = load4_act(x, (size_t)min(b, B - 1) * K + min(k, K - 8));
        const float4 hi = load4_act(x, (size_t)min(b, B - 1) * K + min(k, K - 8) + 4);
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
        v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = in ? v[j] : 0.f;
        if constexpr (PX > 0) {
            if (b < B && k < Kp) {
                bf16x8_t pc[3];
                split3_trunc(v, pc);
#pragma unroll
                for (int q = 0; q < PX; ++q)
                    *reinterpret_cast<bf16x8_t *>(planes + ((size_t)q * Bp + b) * Kp + k) = pc[q];
            }
        }
        if constexpr (XT)
#pragma unroll
            for (int j = 0; j < 8; ++j) store_act(&ts[8 * (tid & 7) + j][tl], 0, v[j]);
    }
    if constexpr (XT) {
        __syncthreads();
        // rows of 64 tokens, 16 bytes per thread and pass
        constexpr int E = 16 / (int)sizeof(T), PER = 64 / E;
#pragma unroll
        for (int i = tid; i < 64 * PER; i += 256) {
            const int d = i / PER, c = i % PER;
            if (k0 + d <= K)                         // row K: zeros
                *reinterpret_cast<uint4 *>(xt + (size_t)(k0 + d) * Bp + b0 + c * E) =
                    *reinterpret_cast<const uint4 *>(&ts[d][c * E]);
        }
    }
}

// gptr: the running sum of the rows' group counts, one workgroup.
__global__ __launch_bounds__(1024) void group_scan_kernel(const int *rowp, int M, int *gptr) {
    __shared__ int sums[1024];
    const int tid = threadIdx.x, per = (M + 1023) / 1024;
    const int m0 = min(tid * per, M), m1 = min(m0 + per, M);
    int n = 0;
    for (int m = m0; m < m1; ++m) n += max(1, (rowp[m + 1] - rowp[m] + 3) / 4);
    sums[tid] = n;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int v = tid >= o ? sums[tid - o] : 0;
        __syncthreads();
        sums[tid] += v;
        __syncthreads();
    }
    int at = sums[tid] - n;
    for (int m = m0; m < m1; ++m) {
        gptr[m] = at;
        at += max(1, (rowp[m + 1] - rowp[m] + 3) / 4);
    }
    if (tid == 1023) gptr[M] = sums[tid];
}

// Thread m: row m's groups; threads M .. M + 3 the four groups past the last.
__global__ __launch_bounds__(256) void group_fill_kernel(const int *rowp, const int *col, const float *val,
                                                        int M, int K, const int *gptr, int *ocol,
                                                        float *oval, int *orow) {
    const int m = blockIdx.x * 256 + threadIdx.x;
    if (m >= M + 4) return;
    const int g0 = m < M ? gptr[m] : gptr[M] + m - M, g1 = m < M ? gptr[m + 1] : g0 + 1;
    const int j0 = m < M ? rowp[m] : 0, n = m < M ? rowp[m + 1] - j0 : 0;
    for (int g = g0; g < g1; ++g) {
        orow[g] = g == g0 ? (int)(m | 0x80000000u) : m;
        for (int i = 0; i < 4; ++i) {
            const int j = 4 * (g - g0) + i;
            ocol[4 * g + i] = j < n ? col[j0 + j] : K;
            oval[4 * g + i] = j < n ? val[j0 + j] : 0.f;
        }
    }
}

int launch_outlier_groups(const int *rowp, const int *col, const float *val, int M, int K, int *gptr,
                          int *ocol, float *oval, int *orow, hipStream_t st) {
    OJX_LAUNCH(group_scan_kernel, dim3(1), dim3(1024), 0, st, rowp, M, gptr);
    OJX_LAUNCH(group_fill_kernel, dim3((M + 4 + 255) / 256), dim3(256), 0, st, rowp, col, val, M, K,
               (const int *)gptr, ocol, oval, orow);
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

namespace {

template <typename T, int PROD, int WT, int WR, int NWT, int NWR, int PXD>
int launch_gemm_tile(GemmParams p, hipStream_t st) {
    constexpr int NT = 64 * NWT * NWR, BT = 32 * WT * NWT, BR = 32 * WR * NWR;
    constexpr int PX = PROD == kBf6 ? 3 : 1, PC = PROD == kBf1 ? 1 : 3;
    constexpr size_t stage = (size_t)PC * 8192 + 2 * PX * BT * 128;
    constexpr size_t sums = (size_t)NWR * 32 * (BT + 4) * sizeof(float);
    const size_t lds = p.gptr ? std::max(stage, sums) : stage;
    static_assert(stage <= 160 * 1024 && sums <= 160 * 1024, "LDS");
    static size_t granted = 0;
    int rc = ensure_dyn_lds(reinterpret_cast<const void *>(&lut_gemm_kernel<T, PROD, WT, WR, NWT, NWR, PXD>), lds, &granted);
    if (rc) return rc;
    p.nr = (p.M + BR - 1) / BR;
    p.nt = (p.B + BT - 1) / BT;
    p.n_tiles = p.nr * p.nt;
    OJX_LAUNCH((lut_gemm_kernel<T, PROD, WT, WR, NWT, NWR, PXD>), dim3(8 * ((p.n_tiles + 7) / 8)), dim3(NT), lds, st, p);
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

// Tile by how full it leaves the 256 CUs (one workgroup's K loop is a fixed
// time, whatever the batch).  Measured, us per call, tokens x rows of a tile:
//   one product, 2560 -> 6912, tokens     512   1024   2048
//     64 x 128                           47.6   81.8  137.8
//     128 x 128                          50.3   72.9  132.9
//     256 x 256                         103.7  107.7  119.4
// 128 x 128 from 384 tiles (9728 -> 2560 at 1024 tokens, 160 tiles: 176 against
// 143 us); 256 x 256 where its last round of workgroups is at least four fifths
// full (2560 -> 19456 at 1024 tokens, 304 tiles: 209 against 160 us).
//   six products (three), tokens          256        512        1024       2048
//     64 x 128                          73 (46)   130 (72)   240 (132)  429 (229)
//     128 x 128                        101 (60)   115 (63)   225 (110)  448 (215)
//     128 x 256                        168 (91)   171 (96)   197 (106)  393 (193)
// Their times go by whole rounds of workgroups over the CUs: six products 61 us
// a round and 9, 112 and 195; three 31 and 13, 51 and 10, 93.  The least of the
// three sums is also the fastest at 9728 -> 2560, 2560 -> 19456, 2560 -> 2560 and
// 512 -> 4096.
template <typename T, int PROD>
int launch_gemm_prod(const GemmParams &p, hipStream_t st) {
    auto tiles = [&](int rows, int tokens) {
        return (long)((p.M + rows - 1) / rows) * ((p.B + tokens - 1) / tokens);
    };
    auto rounds = [&](int rows, int tokens) { return (tiles(rows, tokens) + kGemmCUs - 1) / kGemmCUs; };
    if constexpr (PROD == kBf1) {
        if (5 * tiles(256, 256) >= 4 * kGemmCUs * rounds(256, 256))
            return launch_gemm_tile<T, PROD, 4, 2, 2, 4, 1>(p, st);
        if (2 * tiles(128, 128) >= 3 * kGemmCUs) return launch_gemm_tile<T, PROD, 2, 2, 2, 2, 2>(p, st);
        return launch_gemm_tile<T, PROD, 1, 1, 2, 4, 2>(p, st);
    } else {
        constexpr bool six = PROD == kBf6;
        const long small = (six ? 61 : 31) * rounds(128, 64) + (six ? 9 : 13);
        const long mid = (six ? 112 : 51) * rounds(128, 128) + (six ? 0 : 10);
        const long big = (six ? 195 : 93) * rounds(256, 128);
        if (big <= mid && big <= small) {
            if constexpr (six) return launch_gemm_tile<T, PROD, 4, 1, 1, 8, 1>(p, st);
            else return launch_gemm_tile<T, PROD, 2, 2, 2, 4, 1>(p, st);
        }
        if (mid <= small) return launch_gemm_tile<T, PROD, 2, 1, 2, 4, 1>(p, st);
        return launch_gemm_tile<T, PROD, 1, 1, 2, 4, 1>(p, st);
    }
}

// The pieces of fp32 x (planes) and x transposed (xt), where they are wanted.
int launch_prep(const GemmParams &p, const void *x, bool f32, void *planes, void *xt, hipStream_t st) {
    const dim3 grid(xt ? p.K / 64 + 1 : p.Kp / 64, (p.B + 63) / 64);   // x^T: rows 0 .. K
    uint16_t *pl = static_cast<uint16_t *>(planes);
    if (!f32)
        OJX_LAUNCH((gemm_prep_kernel<__hip_bfloat16, 0, true>), grid, dim3(256), 0, st,
                   static_cast<const __hip_bfloat16 *>(x), p.B, p.K, p.Kp, p.Bp, pl,
                   static_cast<__hip_bfloat16 *>(xt));
    else if (xt)
        OJX_LAUNCH((gemm_prep_kernel<float, 3, true>), grid, dim3(256), 0, st, static_cast<const float *>(x),
                   p.B, p.K, p.Kp, p.Bp, pl, static_cast<float *>(xt));
    else
        OJX_LAUNCH((gemm_prep_kernel<float, 3, false>), grid, dim3(256), 0, st, static_cast<const float *>(x),
                   p.B, p.K, p.Kp, p.Bp, pl, static_cast<float *>(xt));
    OJX_HIP(hipGetLastError());
    return OJASX_OK;
}

}  // namespace

// Where the batched kernel's workgroups (32 rows x 64 tokens for bf16 x, 64 x 32
// for fp32) no longer fit one per CU, each further round of them costs about
// 21 us at 2560 inputs, and the tiles above start at 30 us (one product), 43
// (three) or 70 (six, the x planes' launch included): 2560 -> 6912 at 128 tokens
// 30.9 against 43.2 us in bf16; fp32 70 against 50 at 128 (two rounds), 73
// against 96 at 256 (four).  At 9728 inputs two rounds lose already (210 against
// 246 us for 2560 rows at 256 fp32 tokens).
bool gemm_pays(const LinearGemm &g, int B, int dtype) {
    const bool f32 = dtype == OJASX_DTYPE_F32;
    const long wgs = f32 ? (long)((g.M + 63) / 64) * ((B + 31) / 32) : (long)((g.M + 31) / 32) * ((B + 63) / 64);
    const bool one = !f32 && g.cb_bf16;
    return B > 64 && wgs > (one || g.K >= 4096 ? kGemmCUs : 2 * kGemmCUs);
}

int launch_gemm(const LinearGemm &g, const void *x, void *y, int B, int dtype, hipStream_t st) {
    const bool f32 = dtype == OJASX_DTYPE_F32;
    const int prod = f32 ? kBf6 : g.cb_bf16 ? kBf1 : kBf3;
    const int px = f32 ? 3 : 0;                      // planes of x
    const size_t es = f32 ? 4 : 2;
    GemmParams p{};
    p.codes = g.codes;
    p.cb = prod == kBf1 ? g.cb_bf16 : g.cb3;
    p.scales = g.scales;
    p.bias = g.bias;
    p.gptr = g.gptr;
    p.orow = g.orow;
    p.ocol = g.ocol;
    p.oval = g.oval;
    p.K = g.K;
    p.Kp = (int)round_up(g.K, kGK);
    p.M = g.M;
    p.Mp = g.Mp;
    // tokens per pass: the scratch stays below kGemmScratch
    const size_t per_token = (size_t)px * p.Kp * 2 + (g.gptr ? (size_t)(p.K + 1) * es : 0) + 1;
    const int most = (int)std::max<size_t>(256, kGemmScratch / per_token / 256 * 256);
    for (int b = 0; b < B; b += most) {
        const int nb = std::min(most, B - b);
        p.B = nb;
        p.Bp = (int)round_up(nb, 256);
        const size_t planes = (size_t)px * p.Bp * p.Kp * 2, xt = g.gptr ? (size_t)p.Bp * (p.K + 1) * es : 0;
        unsigned char *ws = nullptr;
        if (planes + xt) {
            int rc = stream_scratch(st, planes + xt, reinterpret_cast<void **>(&ws));
            if (rc) return rc;
        }
        const unsigned char *xb = static_cast<const unsigned char *>(x) + (size_t)b * g.K * es;
        void *pl = px ? ws : nullptr, *tt = g.gptr ? ws + planes : nullptr;
        int rc = px || tt ? launch_prep(p, xb, f32, pl, tt, st) : OJASX_OK;
        if (rc) return rc;
        p.x = px ? pl : xb;
        p.xt = tt;
        p.y = static_cast<unsigned char *>(y) + (size_t)b * g.M * es;
        rc = prod == kBf6 ? launch_gemm_prod<float, kBf6>(p, st)
             : prod == kBf3 ? launch_gemm_prod<__hip_bfloat16, kBf3>(p, st)
                            : launch_gemm_prod<__hip_bfloat16, kBf1>(p, st);
        if (rc) return rc;
    }
    return OJASX_OK;
}

}  // namespace ojx
