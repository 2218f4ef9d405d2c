// rows.hip -- a Q8_0 matrix times several fp32 rows (matmulQ80xF32 for the
// rows of a batch or a prompt) on the matrix cores, at fp32 accuracy.
//
// Reference: matmulQ80xF32, src/tensor.js:26-53, once per row.
//
// Accuracy: an fp32 activation is the exact sum of three bf16 values (8 + 8 +
// 8 significand bits, cut off rather than rounded), and an int8 weight is a
// bf16 value, so per 32-value block three MFMAs per k step give
// sum(x_lo q) + sum(x_mid q) + sum(x_hi q) from exact products with fp32
// accumulation; the block's fp16 scale is applied to that fp32 sum.  bf16 has
// the exponents of fp32 but not its 24 bits below 2^-110, and 32 unscaled
// products of values from 2^115 on can leave fp32: a wave (GEMM: workgroup)
// that met activations all below 2^-63, or whose sums are not finite, forms
// its sums again from rows scaled by a power of two (scale_of).  So a finite
// row of any magnitude, subnormals too, is taken as exactly as any other.
// Long sums are kept in two levels (RG_FLUSH blocks, then the total).
// Relative L2 against binary64 at 2048 -> 7168, 200 rows: 8.6e-8 (the fp32
// vector-unit kernel this replaces: 2.2e-7).
//
// Before, every workgroup of 32 outputs took 4 rows: the weights were read
// and converted rows / 4 times and the products ran on the vector units.
// us, before / now:
//   rows       2048 -> 7168   7168 -> 2048   1024 -> 3072   2048 -> 65536   256 -> 256
//      2        9.6 / 5.7     28.5 / 10.4     5.9 / 3.6     39.5 / 24.1     3.7 / 3.5
//     16       21.4 / 7.0     48.5 / 16.3     8.9 / 4.3      170 / 28.1     4.1 / 3.5
//     64       62.1 / 13.6    65.4 / 18.9    17.9 / 6.1      629 / 58.5     4.2 / 3.6
//    200        192 / 31.7     248 / 34.3    44.5 / 16.7      -             4.3 / 3.6
//   1000        952 / 107     1057 / 108      232 / 35.4      -             8.9 / 4.2
#include <type_traits>

#include "qq_device.h"

namespace qq {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef float f16v_t __attribute__((ext_vector_type(16)));

// Top halves of two words: (lo >> 16) | (hi & 0xffff0000).
__device__ __forceinline__ uint32_t top16(uint32_t hi, uint32_t lo)
{
    return __builtin_amdgcn_perm(hi, lo, 0x07060302u);
}

// 8 fp32 values -> three bf16 planes with v = h + m + l: exactly from 2^-110
// on; of smaller values the bits below 2^-133 are cut off.  A NaN stays one;
// an infinity turns into one unless INF, where it goes to h alone (on a path no
// finite row takes).
template <bool INF>
__device__ __forceinline__ void split3(const float (&v)[8], uint4 &h, uint4 &m, uint4 &l)
{
    uint32_t u[8], rb[8], lb[8];
    float t[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        u[i] = __float_as_uint(v[i]);
        const float r = v[i] - __uint_as_float(u[i] & 0xffff0000u);
        rb[i] = __float_as_uint(r);
        t[i] = r - __uint_as_float(rb[i] & 0xffff0000u);
        lb[i] = __float_as_uint(t[i]);
    }
    if constexpr (INF) {
        float chk = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i += 2) chk = fmaf(t[i], t[i + 1], chk);
        if (chk != chk) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if ((u[i] & 0x7f800000u) == 0x7f800000u) {
                    if (u[i] & 0x007fffffu) u[i] = 0x7fc00000u;
                    rb[i] = lb[i] = 0;
                }
        }
    }
    h = make_uint4(top16(u[1], u[0]), top16(u[3], u[2]), top16(u[5], u[4]), top16(u[7], u[6]));
    m = make_uint4(top16(rb[1], rb[0]), top16(rb[3], rb[2]), top16(rb[5], rb[4]), top16(rb[7], rb[6]));
    l = make_uint4(top16(lb[1], lb[0]), top16(lb[3], lb[2]), top16(lb[5], lb[4]), top16(lb[7], lb[6]));
}

// or8 collects the bits of all activations met; tiny_bits: all below 2^-63
// (both top exponent bits clear) and not all 0.
__device__ __forceinline__ uint32_t or8(const float (&v)[8], uint32_t o)
{
#pragma unroll
    for (int i = 0; i < 8; i += 2) o = o | __float_as_uint(v[i]) | __float_as_uint(v[i + 1]);
    return o;
}

__device__ __forceinline__ bool tiny_bits(uint32_t o) { return (o & 0x7fffffffu) != 0 && (o & 0x60000000u) == 0; }

// Whether 8 values are all below 2^-63, from their h plane.
__device__ __forceinline__ bool small8(const uint4 h) { return (((h.x | h.y | h.z) | h.w) & 0x60006000u) == 0; }

__device__ __forceinline__ float max8(const float (&v)[8], float m)
{
#pragma unroll
    for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(v[i]));
    return m;
}

__device__ __forceinline__ bool tiny(float m) { return m > 0.0f && m < 0x1p-63f; }

// The power of two that a row enters with whose largest value (NaN apart) is m.
__device__ __forceinline__ float scale_of(float m) { return tiny(m) ? 0x1p64f : m > 0x1p115f ? 0x1p-32f : 1.0f; }

// Of products of pairs of sums: finite only if all of these are (the other way
// round only up to 2^63, past which a look at the rows does no harm).
__device__ __forceinline__ bool finite_sum(float c) { return fabsf(c) <= 0x1.fffffep127f; }

__device__ __forceinline__ b8_t as_b8(const uint4 v) { return __builtin_bit_cast(b8_t, v); }

// 8 int8 weights -> 8 bf16 holding the same integers exactly (|q| <= 128 has
// at most 8 significant bits, so the top half of the fp32 value is exact).
__device__ __forceinline__ b8_t int8_to_bf16x8(const uint32_t w0, const uint32_t w1)
{
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t w = i < 2 ? w0 : w1;
        const int s = 16 * (i & 1);
        const float a = (float)(int8_t)(w >> s), b = (float)(int8_t)(w >> (s + 8));
        o[i] = top16(__float_as_uint(b), __float_as_uint(a));
    }
    return __builtin_bit_cast(b8_t, make_uint4(o[0], o[1], o[2], o[3]));
}

// 8 consecutive activations.  RAG: at any 4-byte alignment.
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

template <bool RAG>
__device__ __forceinline__ void load8(const float *x, float (&v)[8])
{
    if constexpr (RAG) {
        const f4u_t a = *reinterpret_cast<const f4u_t *>(x);
        const f4u_t b = *reinterpret_cast<const f4u_t *>(x + 4);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = a[i];
            v[4 + i] = b[i];
        }
    } else {
        const float4 a = *reinterpret_cast<const float4 *>(x);
        const float4 b = *reinterpret_cast<const float4 *>(x + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
}

// Activations k .. k + 7 of a row of n values, zero from n on.
__device__ __forceinline__ void load8_end(const float *xr, int k, int n, float (&v)[8])
{
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float t = xr[min(k + i, n - 1)];
        v[i] = k + i < n ? t : 0.0f;
    }
}

struct RowsArgs {
    const int8_t *qs;        // the matrix's first block
    const uint16_t *d;       // its scales (fp16 bits)
    const float *x;
    float *y;
    int rows, nb, in_dim;    // weight rows (outputs), blocks, inputs
    int ldx, ldy, nvec;      // row strides, input rows
    int ncg;                 // column groups
};

// ---------------------------------------------------------------------------
// A few rows (a decode batch): bound by reading the weights (2 rows of 2048 ->
// 65536: 24 us, 5.9 TB/s; at 16 rows, 28 us, the vector units are busy half the
// time).  A workgroup owns
// 16 NF outputs and 16 MF input rows; its NW waves split the blocks of the
// reduction and stream their weights (8 bytes of a column per lane and
// fragment) straight into registers RS_PF blocks ahead, with no barrier until
// their sums are added, as a tree (relative error 7.3e-8 at 32 to 64 blocks; one
// wave after the other 7.9e-8 to 9.0e-8, the GEMM 7.5e-8 to 8.7e-8).
// ---------------------------------------------------------------------------
constexpr int RS_NW = 8;
constexpr int RS_PF = 2;

template <int MF, int NF, bool RAG>
struct RsBlock {
    float a[MF][8];
    uint2 q[NF];
    uint16_t d[NF];
};

template <int MF, int NF, bool RAG>
__global__ __launch_bounds__(RS_NW *WAVE, 2) void q8_0_rows_kernel(RowsArgs a)
{
    constexpr int NC = 16 * NF;
    __shared__ float red[RS_NW][16][NC + 1];
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int rt = blockIdx.x / a.ncg, cg = blockIdx.x - rt * a.ncg;
    const int v0 = rt * 16 * MF, c0 = cg * NC;
    const int l16 = lane & 15, kq = 8 * (lane >> 4);

    const float *xr[MF];
#pragma unroll
    for (int m = 0; m < MF; m++) xr[m] = a.x + (size_t)min(v0 + 16 * m + l16, a.nvec - 1) * a.ldx;
    int col[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) col[f] = min(c0 + 16 * f + l16, a.rows - 1);

    f4_t acc[MF][NF];
#pragma unroll
    for (int m = 0; m < MF; m++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[m][f] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    using Blk = RsBlock<MF, NF, RAG>;
    auto load_w = [&](Blk &b, int kb) {
        const size_t o = (size_t)kb * a.rows;
#pragma unroll
        for (int f = 0; f < NF; f++) {
            b.q[f] = *reinterpret_cast<const uint2 *>(a.qs + (o + col[f]) * QK + kq);
            b.d[f] = a.d[o + col[f]];
        }
    };
    auto load = [&](Blk &b, int kb) {
        load_w(b, kb);
#pragma unroll
        for (int m = 0; m < MF; m++) load8<RAG>(xr[m] + kb * QK + kq, b.a[m]);
    };
    // ... of the block that crosses the end of the row (RAG)
    auto load_end = [&](Blk &b, int kb) {
        load_w(b, kb);
#pragma unroll
        for (int m = 0; m < MF; m++) load8_end(xr[m], kb * QK + kq, a.in_dim, b.a[m]);
    };
    uint32_t bits[MF];
#pragma unroll
    for (int m = 0; m < MF; m++) bits[m] = 0;
    auto mul_any = [&](const Blk &b, auto any) {
        b8_t ah[MF], am[MF], al[MF];
#pragma unroll
        for (int m = 0; m < MF; m++) {
            uint4 h, mm, l;
            split3<decltype(any)::value>(b.a[m], h, mm, l);
            ah[m] = as_b8(h);
            am[m] = as_b8(mm);
            al[m] = as_b8(l);
        }
#pragma unroll
        for (int f = 0; f < NF; f++) {
            const b8_t q = int8_to_bf16x8(b.q[f].x, b.q[f].y);
            const float d = (float)__builtin_bit_cast(_Float16, b.d[f]);
#pragma unroll
            for (int m = 0; m < MF; m++) {
                f4_t p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[m], q, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am[m], q, p, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[m], q, p, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[m][f][r] = fmaf(p[r], d, acc[m][f][r]);
            }
        }
    };
    auto mul = [&](const Blk &b) {
#pragma unroll
        for (int m = 0; m < MF; m++) bits[m] = or8(b.a[m], bits[m]);
        mul_any(b, std::false_type());
    };

    // The blocks whose 32 activations all exist, then (RAG) the one that
    // crosses the end of the row: no load of the loop is under a condition.
    const int nfull = RAG ? a.in_dim / QK : a.nb;
    if (!RAG || nfull > 0) {
        const int n = (nfull - wave + RS_NW - 1) / RS_NW;   // this wave's blocks
        Blk blk[RS_PF];
        // Every load of the steady loop is unconditional: a wait for one block
        // can then leave the blocks behind it in flight (past a branch that may
        // or may not have issued loads the compiler has to wait for all of them).
#pragma unroll
        for (int u = 0; u < RS_PF; u++) load(blk[u], min(wave + RS_NW * u, nfull - 1));
        int i = 0;
        for (; i + 2 * RS_PF <= n; i += RS_PF) {
#pragma unroll
            for (int u = 0; u < RS_PF; u++) {
                mul(blk[u]);
                // the refill behind the products
                __builtin_amdgcn_sched_barrier(0);
                load(blk[u], wave + RS_NW * (i + u + RS_PF));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int u = 0; u < RS_PF; u++)
            if (i + u < n) {
                mul(blk[u]);
                if (i + u + RS_PF < n) load(blk[u], wave + RS_NW * (i + u + RS_PF));
            }
#pragma unroll
        for (int u = 0; u < RS_PF; u++)
            if (i + u + RS_PF < n) mul(blk[u]);
    }
    if (RAG && nfull < a.nb && nfull % RS_NW == wave) {
        Blk b;
        load_end(b, nfull);
        mul(b);
    }

    // rows outside the range of the split, or sums outside that of fp32?
    float chk = 0.0f;
    bool look = false, again = false;
    float sc[MF];
#pragma unroll
    for (int m = 0; m < MF; m++) {
        look = look || tiny_bits(bits[m]);
        sc[m] = 0.0f;
#pragma unroll
        for (int f = 0; f < NF; f++)
#pragma unroll
            for (int r = 0; r < 4; r += 2) chk = fmaf(acc[m][f][r], acc[m][f][r + 1], chk);
    }
    if (__any(look || !finite_sum(chk))) {
#pragma unroll 1
        for (int kb = wave; kb < a.nb; kb += RS_NW) {
            Blk b;
            if (RAG && kb == nfull)
                load_end(b, kb);
            else
                load(b, kb);
#pragma unroll
            for (int m = 0; m < MF; m++) sc[m] = max8(b.a[m], sc[m]);
        }
#pragma unroll
        for (int m = 0; m < MF; m++) {   // lanes l, l + 16, l + 32, l + 48 hold a row
            sc[m] = fmaxf(sc[m], __shfl_xor(sc[m], 16, WAVE));
            sc[m] = scale_of(fmaxf(sc[m], __shfl_xor(sc[m], 32, WAVE)));
            again = again || sc[m] != 1.0f;
        }
    }
    if (__any(again)) {
#pragma unroll
        for (int m = 0; m < MF; m++)
#pragma unroll
            for (int f = 0; f < NF; f++) acc[m][f] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int kb = wave; kb < a.nb; kb += RS_NW) {
            Blk b;
            if (RAG && kb == nfull)
                load_end(b, kb);
            else
                load(b, kb);
#pragma unroll
            for (int m = 0; m < MF; m++)
#pragma unroll
                for (int j = 0; j < 8; j++) b.a[m][j] *= sc[m];
            mul_any(b, std::true_type());
        }
#pragma unroll
        for (int m = 0; m < MF; m++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float inv = 1.0f / __shfl(sc[m], 4 * (lane >> 4) + r, WAVE);
#pragma unroll
                for (int f = 0; f < NF; f++) acc[m][f][r] *= inv;
            }
    }
#pragma unroll
    for (int m = 0; m < MF; m++) {
        __syncthreads();
#pragma unroll
        for (int f = 0; f < NF; f++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[wave][4 * (lane >> 4) + r][16 * f + l16] = acc[m][f][r];
        __syncthreads();
        const int nr = min(16, a.nvec - v0 - 16 * m);
        for (int i = threadIdx.x; i < nr * NC; i += RS_NW * WAVE) {
            const int row = i / NC, c = i % NC;
            float s[RS_NW];
#pragma unroll
            for (int w = 0; w < RS_NW; w++) s[w] = red[w][row][c];
#pragma unroll
            for (int w = 1; w < RS_NW; w *= 2)
#pragma unroll
                for (int i = 0; i < RS_NW; i += 2 * w) s[i] += s[i + w];
            if (c0 + c < a.rows) a.y[(size_t)(v0 + 16 * m + row) * a.ldy + c0 + c] = s[0];
        }
    }
}

// ---------------------------------------------------------------------------
// Many rows (a prompt): a GEMM on v_mfma_f32_32x32x16_bf16 (1000 rows of 2048 ->
// 7168: 280 TFLOP/s of results, 840 on the matrix pipe; 200 rows: 187 and 560, one
// round of 224 workgroups).  No pipe is full at 200 rows: the vector units are
// busy 32 % of the time with the conversions, the matrix pipes 22 % with three
// products per weight, and the two waves of a SIMD wait a third of theirs, at a
// barrier every step.  Splitting the rows ahead,
// in a launch of its own, was slower (38.6 us at 200 rows against 32.7): the
// planes are 6 bytes a value to read instead of 4.  A workgroup of 8
// waves owns 64 input rows, 32 NWN outputs and a range of steps, a step being
// two Q8_0 blocks: with NWN = 4, waves 0-3 take the first block of each step
// and waves 4-7 the second (two waves per SIMD where the tiles alone would
// give one, so one wave's conversions run under the other's MFMAs); with
// NWN = 8 every wave takes both.  Each wave computes all 64 rows of its 32
// outputs.  The step's 64 x 64 activations are split into their planes on the
// way into one of two LDS buffers, one barrier per step; a wave's weights (16
// bytes of a column per lane and block) go straight to registers, RG_BD steps
// ahead.  The reduction index is permuted identically in A and B: lane half h
// carries k = 16h + 8s + j in MFMA step s.  Where the tiles leave CUs idle the
// steps are split over S workgroups, whose partial sums a last small launch
// adds in order.
// ---------------------------------------------------------------------------
constexpr int RG_BM = 64;
constexpr int RG_NT = 8 * WAVE;
constexpr int RG_PL = RG_BM * 64;            // one plane of one block: 64 rows x 32 bf16
constexpr int RG_BUF = 2 * 3 * RG_PL;        // a step: 2 blocks x 3 planes
constexpr int RG_BD = 4;                     // weight register sets
constexpr int RG_FLUSH = 8;                  // steps summed in one level
constexpr int RG_SMAX = 8;                   // workgroups a tile's steps are split over
static_assert(RG_NT == RG_BM * 2 * 4, "one 8-value chunk per thread and step");

// 16-byte slot of (row r, chunk c): chunks XORed so that the rows a 16-lane
// group reads touch 16 different bank groups.
__device__ __forceinline__ int rg_slot(int r, int c) { return 4 * r + (c ^ (((r >> 1) ^ (r >> 2)) & 3)); }

template <int NWN, bool RAG>
__global__ __launch_bounds__(RG_NT, 2) void q8_0_gemm_kernel(RowsArgs a, int nrt, int S)
{
    constexpr int NJ = NWN / 4;     // blocks of a step per wave
    static_assert(NWN == 4 || NWN == 8, "8 waves");
    __shared__ __align__(16) char lds[2 * RG_BUF];
    __shared__ uint32_t rowmax[RG_BM];
    __shared__ int sh_look;
    // blocks x, x+8, ... run on one XCD: each takes a contiguous run of the
    // items (row tiles of a column group and segment next to each other), so
    // the weights of a column group are read through one L2
    const int R = nrt * a.ncg * S, per = (R + 7) >> 3;
    const int bi = (int)(blockIdx.x >> 3), it = (int)(blockIdx.x & 7) * per + bi;
    if (bi >= per || it >= R) return;
    const int q = it / nrt, v0 = (it - q * nrt) * RG_BM;
    const int cg = q / S, seg = q - cg * S;
    const int steps_all = (a.nb + 1) >> 1;
    const int s0 = (int)((long)seg * steps_all / S), steps = (int)((long)(seg + 1) * steps_all / S) - s0;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wn = wave % NWN, kg = wave / NWN;
    const int l32 = lane & 31, hf = lane >> 5;
    const int c0 = cg * 32 * NWN + 32 * wn;
    const int col = min(c0 + l32, a.rows - 1);

    // staging: thread t takes (block t / 256, row t / 4 % 64, chunk t % 4) of
    // a step.  Blocks past the end (the last step of an odd count) are read at
    // the last block and enter with zero activations and scale.
    const int ab = wave >> 2, ar = (threadIdx.x >> 2) & 63, ac = threadIdx.x & 3;
    const float *xs = a.x + (size_t)min(v0 + ar, a.nvec - 1) * a.ldx;
    char *const xd = lds + ab * 3 * RG_PL + 16 * rg_slot(ar, ac);
    float av[2][8];
    auto load_a = [&](float (&v)[8], int s) {   // s: step from s0 on
        const int kb = min(2 * (s0 + s) + ab, a.nb - 1);
        if (RAG && kb * QK + QK > a.in_dim)   // the block that crosses the end of the row (kb is wave-uniform)
            load8_end(xs, kb * QK + 8 * ac, a.in_dim, v);
        else
            load8<RAG>(xs + kb * QK + 8 * ac, v);
    };
    uint32_t met = 0;   // chunks of small values, not all 0
    auto store_a = [&](const float (&v)[8], int s, int buf, auto inf) {
        uint4 h, m, l;
        // (in the loop, infinities may turn into NaN: such sums are formed again.
        // What NWN = 8 needs there is the branch: without it the compiler spills
        // 400 bytes a lane.)
        split3<NWN == 8 || decltype(inf)::value>(v, h, m, l);
        if (small8(h) && (or8(v, 0) & 0x7fffffffu)) {
            met = 1;
            asm volatile("" : "+v"(met));   // keeps this a branch, for the same reason
        }
        if (2 * (s0 + s) + ab >= a.nb) h = m = l = make_uint4(0, 0, 0, 0);
        char *p = xd + buf * RG_BUF;
        *reinterpret_cast<uint4 *>(p) = h;
        *reinterpret_cast<uint4 *>(p + RG_PL) = m;
        *reinterpret_cast<uint4 *>(p + 2 * RG_PL) = l;
    };
    struct BSet {
        uint4 q[NJ];
        uint16_t d[NJ];
    };
    BSet bs[RG_BD];
    auto load_b = [&](BSet &b, int s) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int blk = 2 * (s0 + s) + (NJ == 2 ? j : kg);
            const size_t o = (size_t)min(blk, a.nb - 1) * a.rows + col;
            b.q[j] = *reinterpret_cast<const uint4 *>(a.qs + o * QK + 16 * hf);
            b.d[j] = a.d[o];
        }
    };
    f16v_t acc[2], tot[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = tot[i][r] = 0.0f;
    const int ao0 = 16 * rg_slot(l32, 2 * hf), ao1 = 16 * rg_slot(l32, 2 * hf + 1);
    auto mul = [&](const BSet &b, int s, int buf) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const bool in = 2 * (s0 + s) + (NJ == 2 ? j : kg) < a.nb;
            const char *st = lds + buf * RG_BUF + (NJ == 2 ? j : kg) * 3 * RG_PL;
            const b8_t q0 = int8_to_bf16x8(b.q[j].x, b.q[j].y), q1 = int8_to_bf16x8(b.q[j].z, b.q[j].w);
            const float d = in ? (float)__builtin_bit_cast(_Float16, b.d[j]) : 0.0f;
            f16v_t p[2];
#pragma unroll
            for (int pl = 2; pl >= 0; pl--)
#pragma unroll
                for (int i = 0; i < 2; i++) {   // row 32i + x has the swizzle of row x
                    const b8_t a0 = *reinterpret_cast<const b8_t *>(st + pl * RG_PL + ao0 + 2048 * i);
                    const b8_t a1 = *reinterpret_cast<const b8_t *>(st + pl * RG_PL + ao1 + 2048 * i);
                    p[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, q0, pl == 2 ? f16v_t{} : p[i], 0, 0, 0);
                    p[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, q1, p[i], 0, 0, 0);
                }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][r] = fmaf(p[i][r], d, acc[i][r]);
        }
    };

    auto flush = [&]() {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                tot[i][r] += acc[i][r];
                acc[i][r] = 0.0f;
            }
    };
    // As in the row kernel, the steady loop's loads are unconditional.
    const int last = steps - 1;
    if (threadIdx.x < RG_BM) rowmax[threadIdx.x] = 0;
    if (threadIdx.x == 0) sh_look = 0;
    load_a(av[0], 0);
#pragma unroll
    for (int u = 0; u < RG_BD; u++) load_b(bs[u], min(u, last));
    load_a(av[1], min(1, last));
    store_a(av[0], 0, 0, std::false_type());
    load_a(av[0], min(2, last));
    __syncthreads();
    int sb = 0;
    for (; sb + RG_BD + 2 < steps; sb += RG_BD) {   // every sub-step has a step + 3
#pragma unroll
        for (int u = 0; u < RG_BD; u++) {
            const int s = sb + u;
            store_a(av[(u + 1) & 1], s + 1, (u + 1) & 1, std::false_type());
            load_a(av[(u + 1) & 1], s + 3);
            __builtin_amdgcn_sched_barrier(0);
            mul(bs[u], s, u & 1);
            __builtin_amdgcn_sched_barrier(0);
            load_b(bs[u], min(s + RG_BD, last));
            __syncthreads();
        }
        if ((sb & (RG_FLUSH - 1)) == RG_FLUSH - RG_BD) flush();
    }
    for (; sb < steps; sb += RG_BD) {   // the last one or two groups
#pragma unroll
        for (int u = 0; u < RG_BD; u++) {
            const int s = sb + u;
            if (s < steps) {
                if (s < last) store_a(av[(u + 1) & 1], s + 1, (u + 1) & 1, std::false_type());
                if (s + 3 < steps) load_a(av[(u + 1) & 1], s + 3);
                mul(bs[u], s, u & 1);
                if (s + RG_BD < steps) load_b(bs[u], s + RG_BD);
                __syncthreads();
            }
        }
        if ((sb & (RG_FLUSH - 1)) == RG_FLUSH - RG_BD) flush();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) tot[i][r] += acc[i][r];
    // rows outside the range of the split, or sums outside that of fp32?
    float chk = 0.0f;
    bool again = false;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r += 2) chk = fmaf(tot[i][r], tot[i][r + 1], chk);
    if (met || !finite_sum(chk)) sh_look = 1;
    __syncthreads();
    if (sh_look) {
        float mx = 0.0f;
#pragma unroll 8
        for (int s = 0; s < steps; s++) {
            load_a(av[0], s);
            mx = max8(av[0], mx);
        }
        atomicMax(&rowmax[ar], __float_as_uint(mx));
        __syncthreads();
        // (the same in every wave: lane l looks at row l)
        again = __any(scale_of(__uint_as_float(rowmax[lane])) != 1.0f);
    }
    if (again) {
        const float sc = scale_of(__uint_as_float(rowmax[ar]));
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][r] = tot[i][r] = 0.0f;
#pragma unroll 1
        for (int s = 0; s < steps; s++) {
            load_a(av[0], s);
            load_b(bs[0], s);
#pragma unroll
            for (int j = 0; j < 8; j++) av[0][j] *= sc;
            store_a(av[0], s, 0, std::true_type());
            __syncthreads();
            mul(bs[0], s, 0);
            if ((s & (RG_FLUSH - 1)) == RG_FLUSH - 1) flush();
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = 32 * i + 8 * (r >> 2) + 4 * hf + (r & 3);
                tot[i][r] = (tot[i][r] + acc[i][r]) * (1.0f / scale_of(__uint_as_float(rowmax[row])));
            }
    }
    if (NJ == 1) {   // the second blocks' sums pass through LDS to the waves of the first
        float *red = reinterpret_cast<float *>(lds) + wn * 2 * 16 * WAVE + lane;
        if (kg == 1) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) red[(i * 16 + r) * WAVE] = tot[i][r];
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) tot[i][r] += red[(i * 16 + r) * WAVE];
    }
    // lane holds output c0 + lane % 32 and rows 8*(r/4) + 4*(lane/32) + r%4 of each fragment
    if (c0 + l32 >= a.rows) return;
    float *y = a.y + (size_t)seg * a.nvec * a.ldy;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = v0 + 32 * i + 8 * (r >> 2) + 4 * hf + (r & 3);
            if (row < a.nvec) y[(size_t)row * a.ldy + c0 + l32] = tot[i][r];
        }
}

// y = sum of the S partial sums in order (n outputs each, contiguous).
__global__ __launch_bounds__(256) void q8_0_seg_sum_kernel(const float *__restrict__ part, int S, size_t n, int rows,
                                                           int ldy, float *__restrict__ y)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float v[RG_SMAX];
#pragma unroll
    for (int s = 0; s < RG_SMAX; s++) v[s] = part[(size_t)min(s, S - 1) * n + i];
    float t = v[0];
#pragma unroll
    for (int s = 1; s < RG_SMAX; s++)
        if (s < S) t += v[s];
    const size_t row = i / rows;
    y[row * ldy + (i - row * rows)] = t;
}

template <int MF, int NF>
static void launch_rows(qq_ctx *ctx, const RowsArgs &a0, bool rag)
{
    RowsArgs a = a0;
    a.ncg = (a.rows + 16 * NF - 1) / (16 * NF);
    const dim3 grid((unsigned)a.ncg * (unsigned)((a.nvec + 16 * MF - 1) / (16 * MF)));
    if (rag)
        QQ_LAUNCH(ctx, (q8_0_rows_kernel<MF, NF, true>), grid, dim3(RS_NW * WAVE), 0, a);
    else
        QQ_LAUNCH(ctx, (q8_0_rows_kernel<MF, NF, false>), grid, dim3(RS_NW * WAVE), 0, a);
}

template <int NWN>
static void launch_gemm(qq_ctx *ctx, const RowsArgs &a0, int S, bool rag)
{
    RowsArgs a = a0;
    a.ncg = (a.rows + 32 * NWN - 1) / (32 * NWN);
    const int nrt = (a.nvec + RG_BM - 1) / RG_BM;
    if (S > 1) {   // partial sums [S][nvec][rows]
        a.y = ctx->rows_part;
        a.ldy = a.rows;
    }
    const dim3 grid(8u * (unsigned)((a.ncg * nrt * S + 7) / 8));
    if (rag)
        QQ_LAUNCH(ctx, (q8_0_gemm_kernel<NWN, true>), grid, dim3(RG_NT), 0, a, nrt, S);
    else
        QQ_LAUNCH(ctx, (q8_0_gemm_kernel<NWN, false>), grid, dim3(RG_NT), 0, a, nrt, S);
    if (S > 1) {
        const size_t n = (size_t)a.nvec * a.rows;
        QQ_LAUNCH(ctx, q8_0_seg_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->rows_part, S, n, a.rows,
                  a0.ldy, a0.y);
    }
}

int launch_q8_0_rows(qq_ctx *ctx, const qq_tensor *t, int mat, const float *x, int ldx, float *y, int ldy,
                     int rows)
{
    RowsArgs a;
    const size_t o = (size_t)mat * t->nb * t->out_dim;   // the matrix's first block
    a.qs = t->qs + o * QK;
    a.d = reinterpret_cast<const uint16_t *>(t->d) + o;
    a.rows = t->out_dim;
    a.nb = t->nb;
    a.in_dim = t->in_dim;
    a.ldx = ldx;
    a.ldy = ldy;
    a.ncg = 0;
    const bool rag = t->in_dim % QK != 0 || ldx % 4 != 0 || ((uintptr_t)x & 15) != 0;
    // a launch takes at most 2^15 rows, so its grid stays within 2^32 threads
    // for any matrix of up to 2^20 outputs
    constexpr int CHUNK = 1 << 15;
    const int cu = ctx->num_cus;
    prof_begin(ctx, K_MATVEC);
    for (int v = 0; v < rows; v += CHUNK) {
        a.x = x + (size_t)v * ldx;
        a.y = y + (size_t)v * ldy;
        a.nvec = std::min(CHUNK, rows - v);
        const int nrt = (a.nvec + RG_BM - 1) / RG_BM;
        const int tiles = nrt * ((a.rows + 127) / 128);
        if (a.nvec <= 16) {
            if ((a.rows + 63) / 64 >= 2 * cu)
                launch_rows<1, 4>(ctx, a, rag);
            else if ((a.rows + 31) / 32 >= cu / 2)
                launch_rows<1, 2>(ctx, a, rag);
            else
                launch_rows<1, 1>(ctx, a, rag);
            continue;
        }
        // The row kernel in one round of the CUs, in the smallest of its tiles
        // that makes one (2 x 2 fragments take as many workgroups as 1 x 4): its time is that of one tile, and grows with the blocks
        // where the GEMM splits them over workgroups (us, row kernel's tiles
        // from 16 x 16 to 32 x 64 / GEMM on a quarter of the workgroups: 8 blocks
        // 3.9 to 5.9 / 8, 32 blocks 4.4 to 9.1 / 15, 64 blocks 6.5 to 14 / 16, 128
        // blocks 7 to 16 / 12 to 16).
        if (a.nb <= 64) {
            const auto round = [&](int mf, int nf) {
                return (long)((a.rows + 16 * nf - 1) / (16 * nf)) * ((a.nvec + 16 * mf - 1) / (16 * mf)) <= cu;
            };
            bool done = true;
            if (round(1, 1))
                launch_rows<1, 1>(ctx, a, rag);
            else if (round(1, 2))
                launch_rows<1, 2>(ctx, a, rag);
            else if (round(1, 4))
                launch_rows<1, 4>(ctx, a, rag);
            else if (round(2, 4))
                launch_rows<2, 4>(ctx, a, rag);
            else
                done = false;
            if (done) continue;
        }
        // In several rounds the row kernel reads every row once per column group:
        // cheaper than the GEMM's steps and partial sums for one row tile, or few
        // rows x blocks (us, row kernel / GEMM: 32 rows of 7168 -> 2048 32 / 20; 24
        // of 2048 -> 65536 47 / 55; 100 of 512 -> 8192 11.5 / 15.1, of 256 -> 8192
        // 10.4 / 8.2, of 64 -> 8192 9.6 / 5.6)
        if ((long)a.nvec * a.nb > 2048 || (a.nvec > 32 && a.nb < 16)) {
            // 256 outputs per workgroup where that still fills the CUs
            if (nrt * ((a.rows + 255) / 256) >= cu)
                launch_gemm<8>(ctx, a, 1, rag);
            else   // segments of at least 4 steps; S x tiles x 32 KiB <= rows_part
                launch_gemm<4>(ctx, a, std::max(1, std::min({cu / tiles, (a.nb + 1) / 2 / 4, RG_SMAX})), rag);
        } else if ((a.rows + 63) / 64 >= cu / 2) {   // the widest group that leaves a quarter to half of the CUs a workgroup
            launch_rows<2, 4>(ctx, a, rag);
        } else if ((a.rows + 31) / 32 >= cu / 4) {
            launch_rows<2, 2>(ctx, a, rag);
        } else {
            launch_rows<2, 1>(ctx, a, rag);
        }
    }
    prof_end(ctx);
    QQ_HIP(ctx, hipGetLastError());
    return QQ_OK;
}

}  // namespace qq
