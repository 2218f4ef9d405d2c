// q8_0.hip -- one-time Q8_0 repack and the Q8_0 x fp32 matvec (matmulQ80xF32).
//
// Reference: matmulQ80xF32, src/tensor.js:26-53.  Block = {fp16 d, int8 qs[32]}
// (src/tensor.js:1-2); a GGUF [in_dim, out_dim] tensor stores column c as
// ceil(in_dim/32) consecutive blocks (src/tensor.js:4-5, 36).
//
// Device layout (block-major panels): for matrix m and block column b, the 32
// quants of every row r are contiguous, rows in order:
//   qs[((m*nb + b)*rows + r)*32 + i],   d[(m*nb + b)*rows + r]
// A wavefront load of 64 lanes x 16 bytes is then 32 rows x one block: 1 KiB
// contiguous, whichever rows a kernel owns.  The scales are also kept row by
// row, dcm[(m*rows + r)*nbp + b] (nbp = nb rounded up to 8, zero padded).
#include "qq_device.h"

namespace qq {

// ---------------------------------------------------------------------------
// Repack.  One thread per GGUF block; reads are consecutive 34-byte blocks.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void repack_q8_0_kernel(const uint8_t *__restrict__ src,
                                                          int8_t *__restrict__ qs,
                                                          __half *__restrict__ d,
                                                          __half *__restrict__ dcm, size_t nblocks,
                                                          int rows, int nb, int nbp)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nblocks) return;
    const uint16_t *s16 = reinterpret_cast<const uint16_t *>(src + i * QBLK);  // 2-byte aligned
    const size_t col = i / nb;                  // m*rows + r (GGUF column)
    const int b = (int)(i - col * nb);
    const int m = (int)(col / rows);
    const int r = (int)(col - (size_t)m * rows);
    const size_t o = bm_index(m, nb, b, rows, r);
    uint32_t w[8];
#pragma unroll
    for (int j = 0; j < 8; j++) w[j] = (uint32_t)s16[1 + 2 * j] | ((uint32_t)s16[2 + 2 * j] << 16);
    int4 *dst = reinterpret_cast<int4 *>(qs + o * QK);
    dst[0] = make_int4((int)w[0], (int)w[1], (int)w[2], (int)w[3]);
    dst[1] = make_int4((int)w[4], (int)w[5], (int)w[6], (int)w[7]);
    d[o] = __ushort_as_half(s16[0]);
    dcm[col * nbp + b] = __ushort_as_half(s16[0]);
}

int launch_repack_q8_0(qq_ctx *ctx, const uint8_t *gguf_dev, qq_tensor *t)
{
    const size_t nblocks = (size_t)t->n_mats * t->out_dim * t->nb;
    const unsigned grid = (unsigned)((nblocks + 255) / 256);
    prof_begin(ctx, K_REPACK);
    QQ_LAUNCH(ctx, repack_q8_0_kernel, dim3(grid), dim3(256), 0, gguf_dev,
                       t->qs, t->d, t->dcm, nblocks, t->out_dim, t->nb, t->nbp);
    prof_end(ctx);
    QQ_HIP(ctx, hipGetLastError());
    return QQ_OK;
}

// ---------------------------------------------------------------------------
// Single input vector.  A workgroup owns RPW output rows and all of their
// block columns; lane l of a wave takes half h = l & 1 of a block, row
// (l >> 1) % RPW and block slot l / (2 RPW), so one 16-byte load per lane
// covers RPW rows x 64 / (2 RPW) block columns (each a contiguous run of
// 32 RPW bytes); scales come from the row-major copy, so the RPW rows' scales
// are whole lines no other workgroup reads.  Every lane issues the weight and scale loads of its first
// NBW blocks before the input row is staged in LDS, so at 1024 -> 3072 the
// whole matrix is requested at once by 384 workgroups; a kernel that only
// loads the same weights takes as long.  Each lane forms its own half-block
// sums; rows are summed over the lanes of a wave and then over the waves in
// wave order.  RAG: in_dim is not a multiple of 32 (the missing activations
// of the last block read as zero).
constexpr int MV1_MAX_NB = 384;   // 48 KiB of activations in LDS

template <int RPW, int NWV, int NBW, bool RAG>
__global__ __launch_bounds__(NWV * WAVE) void q8_0_matvec1_kernel(const int8_t *__restrict__ qs,
                                                                  const __half *__restrict__ dcm, int mat,
                                                                  int rows, int nb, int nbp, int in_dim,
                                                                  const float *__restrict__ x,
                                                                  float *__restrict__ y)
{
    constexpr int SPW = WAVE / (2 * RPW);   // block slots per wave
    constexpr int BPR = NWV * SPW;          // block columns per round of the workgroup
    constexpr int NT = NWV * WAVE;
    extern __shared__ __align__(16) float mv_x[];   // nb * 32 activations
    __shared__ float red[NWV][RPW];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int h = lane & 1, r = (lane >> 1) & (RPW - 1), s = lane / (2 * RPW);
    const int row = blockIdx.x * RPW + r;
    const bool row_ok = row < rows;
    const int rc = min(row, rows - 1);
    const int first = wave * SPW + s;
    int4 q[NBW];
    float dd[NBW];
    // branch-free: clamped block, zero scale past the last one
    auto load = [&](int c0) {
#pragma unroll
        for (int u = 0; u < NBW; u++) {
            const int bc = min(c0 + first + BPR * u, nb - 1);
            const size_t o = bm_index(mat, nb, bc, rows, rc);
            q[u] = *reinterpret_cast<const int4 *>(qs + o * QK + 16 * h);
            dd[u] = __half2float(dcm[((size_t)mat * rows + rc) * nbp + bc]);
        }
#pragma unroll
        for (int u = 0; u < NBW; u++) dd[u] = (row_ok && c0 + first + BPR * u < nb) ? dd[u] : 0.0f;
    };
    load(0);
    const int kp = nb * QK;
    for (int k = 4 * threadIdx.x; k < kp; k += 4 * NT) {
        float4 v;
        if (!RAG || k + 4 <= in_dim) {
            v = *reinterpret_cast<const float4 *>(x + k);
        } else {
            v.x = k < in_dim ? x[k] : 0.0f;
            v.y = k + 1 < in_dim ? x[k + 1] : 0.0f;
            v.z = k + 2 < in_dim ? x[k + 2] : 0.0f;
            v.w = k + 3 < in_dim ? x[k + 3] : 0.0f;
        }
        *reinterpret_cast<float4 *>(&mv_x[k]) = v;
    }
    __syncthreads();
    float acc = 0.0f;
    for (int c0 = 0;;) {
#pragma unroll
        for (int u = 0; u < NBW; u++) {
            const int bc = min(c0 + first + BPR * u, nb - 1);
            float xr[16];
            const float4 *p = reinterpret_cast<const float4 *>(&mv_x[bc * QK + 16 * h]);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 v = p[i];
                xr[4 * i] = v.x;
                xr[4 * i + 1] = v.y;
                xr[4 * i + 2] = v.z;
                xr[4 * i + 3] = v.w;
            }
            float xs = 0.0f;
#pragma unroll
            for (int j = 0; j < 16; j++) xs += xr[j];
            acc = fmaf(dot16_q8(q[u], xr, xs), dd[u], acc);
        }
        c0 += NBW * BPR;
        if (c0 >= nb) break;
        load(c0);
    }
    acc += __shfl_xor(acc, 1, WAVE);
#pragma unroll
    for (int o = 2 * RPW; o < WAVE; o <<= 1) acc += __shfl_xor(acc, o, WAVE);
    if (lane < 2 * RPW && h == 0) red[wave][r] = acc;
    __syncthreads();
    if (threadIdx.x < RPW) {
        const int orow = blockIdx.x * RPW + threadIdx.x;
        if (orow < rows) {
            float v = red[0][threadIdx.x];
#pragma unroll
            for (int w = 1; w < NWV; w++) v += red[w][threadIdx.x];
            y[orow] = v;
        }
    }
}

template <bool RAG>
static void launch_matvec1(qq_ctx *ctx, const qq_tensor *t, int mat, const float *x, float *y)
{
    // launch shapes measured at 1024 -> 3072, 2048 -> 2048, 7168 -> 2048 and
    // 2048 -> 7168: 8 rows per workgroup, 4 waves up to 32 block columns,
    // else 8; up to 2 blocks in flight per lane for 64 block columns, else 4
    constexpr int RPW = 8;
    const dim3 grid((t->out_dim + RPW - 1) / RPW);
    const size_t shm = (size_t)t->nb * QK * sizeof(float);
    if (t->nb <= 16)
        QQ_LAUNCH(ctx, (q8_0_matvec1_kernel<RPW, 4, 1, RAG>), grid, dim3(4 * WAVE), shm, t->qs, t->dcm, mat,
                  t->out_dim, t->nb, t->nbp, t->in_dim, x, y);
    else if (t->nb <= 32)
        QQ_LAUNCH(ctx, (q8_0_matvec1_kernel<RPW, 4, 2, RAG>), grid, dim3(4 * WAVE), shm, t->qs, t->dcm, mat,
                  t->out_dim, t->nb, t->nbp, t->in_dim, x, y);
    else if (t->nb <= 64)
        QQ_LAUNCH(ctx, (q8_0_matvec1_kernel<RPW, 8, 2, RAG>), grid, dim3(8 * WAVE), shm, t->qs, t->dcm, mat,
                  t->out_dim, t->nb, t->nbp, t->in_dim, x, y);
    else
        QQ_LAUNCH(ctx, (q8_0_matvec1_kernel<RPW, 8, 4, RAG>), grid, dim3(8 * WAVE), shm, t->qs, t->dcm, mat,
                  t->out_dim, t->nb, t->nbp, t->in_dim, x, y);
}

// Matrices whose one-row product the row kernel forms sooner: this kernel
// stages the row once per 8 outputs, which takes long for many blocks; for very
// few a workgroup has next to nothing else to do.  us, this kernel / the row
// kernel: 2048 inputs, 7168 outputs 5.9 / 6.1, 16384 11.2 / 8.9, 65536 34 / 24;
// 896 inputs, 16384 outputs 5.7 / 5.0; 768 inputs 4.3 / 4.7, 131072 outputs 23.5 /
// 25.8; 512 inputs, 32768 outputs 4.5 / 5.1; 128 inputs 4.2 / 3.8, 50000 outputs
// 5.6 / 5.8, 65536 6.7 / 5.9.
static bool matvec1_large(int out_dim, int nb)
{
    return (nb >= 28 && out_dim >= 16384) || (nb <= 4 && out_dim >= 65536);
}

int launch_q8_0_matvec(qq_ctx *ctx, const qq_tensor *t, int mat, const float *x, int ldx,
                       float *y, int ldy, int rows)
{
    if (rows <= 0) return QQ_OK;
    // one vector whose activations fit in LDS (in_dim <= 12288), of a matrix that
    // is not large; everything else takes the row kernels
    if (rows > 1 || ((uintptr_t)x & 15) != 0 || t->nb > MV1_MAX_NB || matvec1_large(t->out_dim, t->nb))
        return launch_q8_0_rows(ctx, t, mat, x, ldx, y, ldy, rows);
    prof_begin(ctx, K_MATVEC);
    if (t->in_dim % QK)
        launch_matvec1<true>(ctx, t, mat, x, y);
    else
        launch_matvec1<false>(ctx, t, mat, x, y);
    prof_end(ctx);
    QQ_HIP(ctx, hipGetLastError());
    return QQ_OK;
}

}  // namespace qq
