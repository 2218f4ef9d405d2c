// stream.hip -- decode batches (a few to a few dozen tokens per expert) on
// the matrix cores at fp32 accuracy.
//
// With ~8 rows per expert (64 tokens, 32 experts, top-4) every weight is used
// by very few rows, so the layer is bound by streaming the experts' Q8_0
// weights from HBM once.  A workgroup owns one expert, one tile of 16*MF
// slots and a group of weight columns (two halves of 16 NFH: 32 to 112 gate
// and the same up features, 64 to 128 down columns); its 4 waves split the reduction
// dimension block by block (each streaming its blocks straight into
// registers, a few blocks ahead, below) and their partial sums are added in
// wave order through LDS.
//
// Accuracy (the fp32 path's 1e-4 relative L2): activations are split into
// two fp16 halves, a = a_hi + a_lo (22 significant bits); the int8 weights
// are exact in fp16.  Per 32-value block two MFMAs give the block's partial
// sum a_hi*q + a_lo*q with exact products and fp32 accumulation, and the
// block's fp16 scale is applied to that fp32 partial (one FMA per output),
// as the reference applies d per block.  Error ~1e-7 relative, like the fp32
// kernels.
//   gate/up  A = x rows of the tile's tokens (gathered by perm), B = 16 NFH gate
//            columns and the same up columns; epilogue silu(g) * u -> act[slot][F]
//            (fp32)
//   down     A = act rows, B = 32 NFH down columns -> y[slot][H] (fp32)
// followed by the gather combine.
//
// us per call before / now, LFM2 shape (H 2048, F 1792, 32 experts, top-4):
// 2 tokens 47 / 38, 6 tokens 71 / 56, 12 tokens 77 / 71, 64 tokens 86 / 83,
// 128 tokens 120 / 113; Qwen3 shape (F 768, 128 experts, top-8): 16 tokens
// 105 / 96, 64 tokens 139 / 130.  From the steady loop's unconditional loads
// (st_mainloop) and, up to ~12 tokens, the width of the items (st_width).  The
// conversion outside inline assembly (int8_to_f16x8) takes five instructions per
// four weights instead of four, which a launch of two row fragments on few experts
// feels: 8 experts of H 1024, F 3584, top-2, 100 tokens 62.8 / 65.5.
#include "qq_device.h"

namespace qq {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr int ST_THREADS = 256;   // 4 waves split the reduction dimension

struct StreamArgs {
    const float *x;          // [T][H] activations
    float *act;              // [slots][F] SwiGLU products
    float *y;                // [slots][H] expert outputs
    const int32_t *perm, *counts, *offsets;
    const int32_t *tile_e, *tile_m0, *n_tiles;
    const int8_t *gq, *uq, *dq;
    const uint16_t *gd, *ud, *dd;   // fp16 scale bits
    uint64_t *part;          // partial sums of split items (st_work), tagged words
    uint32_t *seg_ctr;       // per split item: segments done (zero between launches)
    uint32_t *seg_gen;       // [0] generation: a launch's partials carry gen + 1;
                             // [1] split items done in the launch (zero between launches)
    uint32_t *err;           // device error word (a bounded wait expired)
    uint64_t wait_ticks;
    int H, F, K, nbH, nbF;
    int G;                   // resident workgroups (2 per CU)
    int tile_cap;            // row tiles the grid is sized for
};

// 8 consecutive fp32 values -> high and low fp16 halves.  hi is rounded
// toward zero (v_cvt_pkrtz_f16_f32); v - hi is exact in fp32 and its fp16
// rounding is the split's only loss.
__device__ __forceinline__ void split8(const float4 a, const float4 b, h8_t &hi, h8_t &lo)
{
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const h2_t h = __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_pkrtz(v[2 * i], v[2 * i + 1]));
        hw[i] = __builtin_bit_cast(uint32_t, h);
        lw[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(v[2 * i] - (float)h[0],
                                                                          v[2 * i + 1] - (float)h[1]));
    }
    hi = __builtin_bit_cast(h8_t, make_uint4(hw[0], hw[1], hw[2], hw[3]));
    lo = __builtin_bit_cast(h8_t, make_uint4(lw[0], lw[1], lw[2], lw[3]));
}

// 8 int8 weights (one lane's share of a 16x32 fragment) -> 8 fp16 holding
// the same integers exactly: bytes in offset binary (q + 128) paired with the
// exponent byte 0x64 give 1152 + q, and the subtraction is exact.  No inline
// assembly here: the outputs may take the registers of a partial sum that an
// MFMA in flight still reads, and the compiler keeps the wait states that
// needs only between instructions it knows.
__device__ __forceinline__ h8_t int8_to_f16x8(const uint2 q)
{
    const h2_t off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t u = (i ? q.y : q.x) ^ 0x80808080u;
        o[2 * i] = __builtin_bit_cast(
            uint32_t, __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + off);
        o[2 * i + 1] = __builtin_bit_cast(
            uint32_t, __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + off);
    }
    return __builtin_bit_cast(h8_t, make_uint4(o[0], o[1], o[2], o[3]));
}

// ---------------------------------------------------------------------------
// Operand stream.  Wave w reduces blocks w, w+4, w+8, ... of the reduction
// dimension.  Every operand of a block goes straight to registers: the
// lane's 8 activations of each of its MF rows (two float4), its 8 weight
// bytes of each of the 2 NFH fragment columns (uint2) and one fp16 scale per
// 64 columns of a half: load u of lane l reads column c0[h] + 64u + l's, and
// a fragment's scale is taken from the lane that loaded it (fragment f of a
// half: load f/4, lanes 16(f%4) .. 16(f%4)+15).  Each wave keeps ST_PF
// blocks in flight: block i + ST_PF is requested as soon as block i's
// products are done.  (Staged through LDS the stream is held to ~100 KB in
// flight per CU by the LDS size.)
// Fragment j: column 16*(j%NFH) + lane%16 of half j/NFH; lane l holds row
// l%16 of A and column l%16 of B at k = 8*(l/16) .. 8*(l/16) + 7 of the block.
// ---------------------------------------------------------------------------
template <int MF, int NFH>
struct StBlock {
    static constexpr int NF = 2 * NFH;      // fragments
    static constexpr int NS = (NFH + 3) / 4;   // scale loads per column half
    float4 a[MF][2];     // rows 16m + lane%16, k = 8*(lane/16) .. +7
    uint2 q[NF];         // fragment j's 8 weight bytes
    uint32_t ds[2][NS];  // scale bits of column c0[h] + 64 s + lane of half h
};

// Blocks in flight per wave.  Two, at every width: 3 of the narrower ones took
// longer (down at 64 tokens 26.3 us against 23.9, gate/up at 6 tokens 25.5
// against 24.8).
constexpr int ST_PF = 2;

template <int MF, int NFH>
struct StSrc {
    static constexpr int NS = (NFH + 3) / 4;
    const char *abase;          // activation rows (bytes)
    uint32_t arow[MF];          // lane's row 16m + lane%16: byte offset + its k chunk
    const int8_t *qb[2];        // weights of column halves 0 / 1 at the expert's block 0
    const uint16_t *db[2];      // their scales
    int cb[2];                  // column half h: the lane's column c0[h] + lane%16 (fragment f of the half adds 16 f)
    int cmax;                   // last column (loads clamp to it)
    uint32_t sc[2][NS];         // column of this lane's scale load s in half h (clamped)
    uint32_t qk;                // the lane's byte offset within a column's 32 bytes
    uint32_t qstep, dstep;      // one block: rows * 32 bytes, rows scales
    uint32_t okm;               // bit j: fragment j's column in range (else its scale is zero)
};

// 32-bit offsets from workgroup-uniform bases (one VGPR per address).
template <int MF, int NFH>
__device__ __forceinline__ void st_load(StBlock<MF, NFH> &b, const StSrc<MF, NFH> &s, int kb)
{
    const uint32_t ak = (uint32_t)kb * (QK * 4), qk = (uint32_t)kb * s.qstep, dk = (uint32_t)kb * s.dstep;
#pragma unroll
    for (int m = 0; m < MF; m++) {
        b.a[m][0] = *reinterpret_cast<const float4 *>(s.abase + (size_t)(s.arow[m] + ak));
        b.a[m][1] = *reinterpret_cast<const float4 *>(s.abase + (size_t)(s.arow[m] + ak + 16));
    }
    // one row tile per expert (MF == 1: at most 16 rows on average) reads
    // every weight byte once, so those loads are non-temporal; with more
    // rows the expert's other row tiles read the same bytes through the L2
#pragma unroll
    for (int j = 0; j < 2 * NFH; j++) {
        const uint32_t c = (uint32_t)min(s.cb[j / NFH] + 16 * (j % NFH), s.cmax);
        const uint2 *src = reinterpret_cast<const uint2 *>(s.qb[j / NFH] + (size_t)(qk + c * QK + s.qk));
        if constexpr (MF == 1) {
            typedef unsigned int v2u __attribute__((ext_vector_type(2)));
            const v2u v = __builtin_nontemporal_load(reinterpret_cast<const v2u *>(src));
            b.q[j] = make_uint2(v.x, v.y);
        } else {
            b.q[j] = *src;
        }
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int u = 0; u < StSrc<MF, NFH>::NS; u++)
            b.ds[h][u] = *reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(s.db[h]) +
                                                             (size_t)(2u * (dk + s.sc[h][u])));
}

// The block's int8 weights enter the MFMA exactly (as fp16 integers); the
// block's scale is applied to the block's fp32 partial sum:
//   acc += d * (a_hi * q + a_lo * q).
// A lane's four outputs of a fragment share one column, hence one scale.
template <int MF, int NFH>
__device__ __forceinline__ void st_block(const StBlock<MF, NFH> &b, const StSrc<MF, NFH> &s,
                                         f4_t (&acc)[MF][2 * NFH])
{
    h8_t ah[MF], al[MF];
#pragma unroll
    for (int m = 0; m < MF; m++) split8(b.a[m][0], b.a[m][1], ah[m], al[m]);
    const int l16 = threadIdx.x & 15;
#pragma unroll
    for (int j = 0; j < 2 * NFH; j++) {
        const int f = j % NFH;
        const uint32_t bits = (uint32_t)__shfl((int)b.ds[j / NFH][f / 4], 16 * (f & 3) + l16, WAVE);
        const float d = ((s.okm >> j) & 1u) ? (float)__builtin_bit_cast(_Float16, (uint16_t)bits) : 0.0f;
        const h8_t qh = int8_to_f16x8(b.q[j]);
#pragma unroll
        for (int m = 0; m < MF; m++) {
            f4_t p = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[m], qh, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            p = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[m], qh, p, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) acc[m][j][r] = fmaf(p[r], d, acc[m][j][r]);
        }
    }
}

// Wave w reduces blocks kb0 + w, kb0 + w + 4, ... of the nb blocks from kb0
// on, with ST_PF blocks in flight.
template <int MF, int NFH>
__device__ __forceinline__ void st_mainloop(const StSrc<MF, NFH> &s, int kb0, int nb, int wave,
                                            f4_t (&acc)[MF][2 * NFH])
{
    constexpr int PF = ST_PF;
    const int nblk = (nb - wave + 3) / 4;
    const int kw = kb0 + wave;
    StBlock<MF, NFH> r[PF];
    // Every load of the steady loop is unconditional: a wait for one block
    // then leaves the blocks behind it in flight.  (Past a branch that may or
    // may not have issued loads the compiler has to wait for all of them: so
    // it drained every block in flight once per PF blocks.)
#pragma unroll
    for (int u = 0; u < PF; u++) st_load<MF, NFH>(r[u], s, min(kw + 4 * u, kb0 + nb - 1));
    int i = 0;
    for (; i + 2 * PF <= nblk; i += PF) {
#pragma unroll
        for (int u = 0; u < PF; u++) {
            st_block<MF, NFH>(r[u], s, acc);
            // the refill goes out only after the products
            __builtin_amdgcn_sched_barrier(0);
            st_load<MF, NFH>(r[u], s, kw + 4 * (i + u + PF));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
        if (i + u < nblk) {
            st_block<MF, NFH>(r[u], s, acc);
            if (i + u + PF < nblk) st_load<MF, NFH>(r[u], s, kw + 4 * (i + u + PF));
        }
#pragma unroll
    for (int u = 0; u < PF; u++)
        if (i + u + PF < nblk) st_block<MF, NFH>(r[u], s, acc);
}

// Load offsets: activation row r of the tile has byte offset rowoff(r);
// weight halves start at columns c0[0], c0[1] of a matrix with `rows`
// columns per block (clamped into range).
template <int MF, int NFH, typename RowOff>
__device__ __forceinline__ void st_offsets(StSrc<MF, NFH> &s, RowOff rowoff, const int (&c0)[2],
                                           int rows, int lane)
{
#pragma unroll
    for (int m = 0; m < MF; m++) s.arow[m] = rowoff(16 * m + (lane & 15)) + 32 * (lane >> 4);
    s.qk = 8 * (lane >> 4);
    s.cb[0] = c0[0] + (lane & 15);
    s.cb[1] = c0[1] + (lane & 15);
    s.cmax = rows - 1;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int u = 0; u < StSrc<MF, NFH>::NS; u++) s.sc[h][u] = (uint32_t)min(c0[h] + 64 * u + lane, rows - 1);
    s.okm = 0;
#pragma unroll
    for (int j = 0; j < 2 * NFH; j++)
        s.okm |= (c0[j / NFH] + 16 * (j % NFH) + (lane & 15) < rows ? 1u : 0u) << j;
}

// Cross-wave sums of fragment row block m: each wave writes its fragments of
// half 0 to red0 and of half 1 to red1 ([wave][16 rows][16 NFH + 1 columns]).
template <int MF, int NFH>
__device__ __forceinline__ void st_spill(float (*red0)[16][16 * NFH + 1], float (*red1)[16][16 * NFH + 1],
                                         const f4_t (&acc)[MF][2 * NFH], int m, int wave, int lane)
{
    const int cl = lane & 15, rq = 4 * (lane >> 4);
#pragma unroll
    for (int j = 0; j < 2 * NFH; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            (j < NFH ? red0 : red1)[wave][rq + r][16 * (j % NFH) + cl] = acc[m][j][r];
}

template <int NFH>
__device__ __forceinline__ float wave_order_sum(const float (*red)[16][16 * NFH + 1], int row, int c)
{
    return ((red[0][row][c] + red[1][row][c]) + red[2][row][c]) + red[3][row][c];
}

// LDS: the cross-wave reduction tiles only
template <int NFH>
constexpr int st_lds() { return 2 * 4 * 16 * (16 * NFH + 1) * 4; }

// The work of one workgroup among R items (row tile x column group, row-tile
// major).  Items that fill whole rounds of the G resident workgroups run
// whole.  A remainder of L < G items would run as a round of its own on L
// workgroups, each streaming only as fast as its own blocks in flight allow:
// a tail as long as a full round for a few percent of the work.  Instead each
// remainder item is split into S segments of the reduction dimension (S L <=
// G / 2, at least 8 blocks each, and S L within the grid's room past the
// whole items, which is sized for the most row tiles there can be; the
// remainder is widened back to the first tile of its first expert, so all
// rows of an expert are summed the same way whatever their order within the
// expert) run by S L more workgroups, which store
// their fp32 partial sums as tagged words (tag = the kernel's generation + 1,
// new in every launch); the last segment to finish adds them in segment order
// and applies the epilogue (st_last, st_seg_sum).  The tags stand in for a
// release / acquire pair, whose device-scope fences would write back the
// whole L2.
constexpr int ST_SEG_MAX = 8;   // segments of a split item

// Width (NFH: fragments of 16 columns a half) of a launch that few tokens make:
// the narrowest from LO to HI at which n row tiles are one round of the G
// resident workgroups.  Each workgroup streams at a rate set by its own blocks
// in flight, so with few tiles the time is that of one item, and an item's
// time is its width (gate/up, one round: 15 us at 2, 24.8 at 4, 43.7 at 7).
// The count of row tiles is known on the device only (the experts a few tokens
// touch), so every workgroup works the width out.  An item's own sums do not depend
// on it; which items are left for a last round, and split (st_work), does.
constexpr int ST_GU_MIN = 2, ST_GU_MAX = 7, ST_DN_MIN = 2, ST_DN_MAX = 4;

template <int LO, int HI>
__host__ __device__ inline int st_width(int n, int cols, int G)
{
    int best = HI;
#pragma unroll
    for (int w = HI - 1; w >= LO; w--)
        if (n * ((cols + 16 * w - 1) / (16 * w)) <= G) best = w;
    return best;
}

struct StWork {
    int item;         // tile * ncg + column group
    int seg, nseg;    // segment of the reduction dimension; nseg == 1: whole
    int li;           // remainder item: counter li, partial slot li * nseg + seg
    int L;            // remainder items (split when nseg > 1)
};

__device__ __forceinline__ bool st_work(int R, int G, int nb, int ncg, int bm, const int32_t *tile_m0,
                                        StWork &w)
{
    int W = R;                               // items run whole
    int L = 0, S = 1;
    // R mod G by subtraction (R / G is a few rounds at most): the divisions
    // below sit on every workgroup's way to its first load, so they are
    // taken only where a split can follow (S >= 2: G >= 4 L, blocks >= 16;
    // widening the remainder only narrows S)
    int rem = R;
    while (rem >= G) rem -= G;
    if (rem && 4 * rem <= G && nb >= 16) {
        const int t = (R - rem) / ncg;      // tile of the first remainder item
        W = (t - tile_m0[t] / bm) * ncg;
        L = R - W;
        const int room = (int)gridDim.x - 8 * ((W + 7) >> 3);
        S = max(1, min(min(min(G / (2 * L), nb / 8), ST_SEG_MAX), room / L));
        if (S == 1) {
            W = R;
            L = 0;
        }
    }
    const int per = (W + 7) >> 3;
    const int b = blockIdx.x;
    w.L = L;
    if (b < 8 * per) {
        // the dispatcher deals workgroups to the 8 XCDs round robin (one XCD
        // runs blocks x, x+8, ...); each XCD takes a contiguous run of the
        // items, so the column groups of a row tile read its activation rows
        // through one L2
        const int x = b & 7, i = b >> 3, it = x * per + i;
        if (it >= W) return false;
        w.item = it;
        w.seg = 0;
        w.nseg = 1;
        w.li = 0;
        return true;
    }
    const int q = b - 8 * per;
    if (S == 1 || q >= L * S) return false;
    w.li = q / S;
    w.seg = q - w.li * S;
    w.nseg = S;
    w.item = W + w.li;
    return true;
}

// Counts this workgroup's segment of a split item in once its partial sums
// are stored; true in the workgroup of the last segment to arrive.  That
// workgroup returns the counter to zero for the next launch.  sh: one int of
// LDS.
__device__ __forceinline__ bool st_last(uint32_t *ctr, int nseg, int *sh)
{
    wait_vm<0>();   // this wave's tagged stores are out
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t old = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = old == (uint32_t)nseg - 1u;
        if (last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *sh = last;
    }
    __syncthreads();
    return *sh != 0;
}

// The last segment's workgroup, after its reduction: counts the item done;
// the last of the launch's L split items moves the generation on (every
// segment of the launch read it before its item's counter reached the end).
__device__ __forceinline__ void st_item_done(uint32_t *gen, int L, uint32_t tag)
{
    if (threadIdx.x == 0) {
        const uint32_t d = __hip_atomic_fetch_add(gen + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == (uint32_t)L - 1u) {
            __hip_atomic_store(gen + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(gen, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Sums of a split item's partial sums: the 4 words from offset o[i] of each
// segment (segments PSZ words apart) into r[i], added in segment order.  All
// loads go out before the first add; words not yet carrying `tag` are read
// again (bounded by wait_ticks: false when the wait expired).
template <int PSZ, int NO>
__device__ __forceinline__ bool st_seg_sum(const uint64_t *p0, const int (&o)[NO], int nseg, uint32_t tag,
                                           uint64_t wait_ticks, float (&r)[NO][4])
{
    uint64_t v[ST_SEG_MAX][NO][4];
    uint64_t t0 = 0;
    for (bool first = true;; first = false) {
        bool ok = true;
#pragma unroll
        for (int sg = 0; sg < ST_SEG_MAX; sg++)
#pragma unroll
            for (int i = 0; i < NO; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (sg < nseg)
                        v[sg][i][j] = __hip_atomic_load(p0 + (size_t)sg * PSZ + o[i] + j, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int sg = 0; sg < ST_SEG_MAX; sg++)
#pragma unroll
            for (int i = 0; i < NO; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (sg < nseg) ok = ok && (uint32_t)(v[sg][i][j] >> 32) == tag;
        if (ok) break;
        if (first) {
            t0 = wall_clock64();
        } else if (wall_clock64() - t0 >= wait_ticks) {
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
#pragma unroll
    for (int i = 0; i < NO; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float x = __uint_as_float((uint32_t)v[0][i][j]);
#pragma unroll
            for (int sg = 1; sg < ST_SEG_MAX; sg++)
                if (sg < nseg) x += __uint_as_float((uint32_t)v[sg][i][j]);
            r[i][j] = x;
        }
    return true;
}

__device__ __forceinline__ float silu_mul(float g, float u)
{
    const double g64 = (double)g;
    return (float)(g64 * (1.0 / (1.0 + exp(-g64)))) * u;
}

// ---------------------------------------------------------------------------
// gate/up: column half 0 = gate features f0 .. f0 + 16 NFH - 1, half 1 = the
// same up features.
// ---------------------------------------------------------------------------
template <int MF, int NFH>
__device__ __forceinline__ void st_gateup(const StreamArgs &a, int n_tiles, char *lds, int *sh_last)
{
    constexpr int NC = 16 * NFH;   // features per workgroup
    const int ncg = (a.F + NC - 1) / NC;
    StWork wk;
    if (!st_work(n_tiles * ncg, a.G, a.nbH, ncg, 16 * MF, a.tile_m0, wk)) return;
    const int tile = wk.item / ncg, cg = wk.item - tile * ncg;
    const int e = a.tile_e[tile], m0 = a.tile_m0[tile];
    const int n = min(16 * MF, a.counts[e] - m0);
    const int slot0 = a.offsets[e] + m0;
    const int f0 = cg * NC;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);

    StSrc<MF, NFH> src;
    src.abase = reinterpret_cast<const char *>(a.x);
    const size_t eb = (size_t)e * a.nbH * a.F;     // expert's first block-row
    src.qb[0] = a.gq + eb * QK;
    src.qb[1] = a.uq + eb * QK;
    src.db[0] = a.gd + eb;
    src.db[1] = a.ud + eb;
    src.qstep = (uint32_t)a.F * QK;
    src.dstep = (uint32_t)a.F;
    const int c0[2] = {f0, f0};
    st_offsets<MF, NFH>(src, [&](int r) {
        return (uint32_t)(a.perm[slot0 + min(r, n - 1)] / a.K) * a.H * 4;
    }, c0, a.F, lane);

    f4_t acc[MF][2 * NFH];
#pragma unroll
    for (int m = 0; m < MF; m++)
#pragma unroll
        for (int j = 0; j < 2 * NFH; j++) acc[m][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int kb0 = wk.nseg > 1 ? wk.seg * a.nbH / wk.nseg : 0;
    const int kb1 = wk.nseg > 1 ? (wk.seg + 1) * a.nbH / wk.nseg : a.nbH;
    const uint32_t tag =
        wk.nseg > 1 ? __hip_atomic_load(a.seg_gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u : 0u;
    st_mainloop<MF, NFH>(src, kb0, kb1 - kb0, wave, acc);
    float (*red0)[16][NC + 1] = reinterpret_cast<float (*)[16][NC + 1]>(lds);
    float (*red1)[16][NC + 1] = red0 + 4;
    // split item: partial [16 MF rows][NC gate | NC up] of each segment
    constexpr int PSZ = 16 * MF * 2 * NC;
    uint64_t *pp = a.part + (size_t)(wk.li * wk.nseg + wk.seg) * PSZ;
#pragma unroll
    for (int m = 0; m < MF; m++) {
        __syncthreads();
        st_spill<MF, NFH>(red0, red1, acc, m, wave, lane);
        __syncthreads();
        // the tile's rows only (a split item's last segment reads those alone)
        const int nr = min(16, n - 16 * m);
        for (int i = threadIdx.x; i < nr * NC; i += ST_THREADS) {
            const int row = i / NC, c = i % NC;
            const int f = f0 + c;
            const float g = wave_order_sum<NFH>(red0, row, c), u = wave_order_sum<NFH>(red1, row, c);
            if (wk.nseg > 1) {
                store_tagged(pp + (16 * m + row) * 2 * NC + c, tag, __float_as_uint(g));
                store_tagged(pp + (16 * m + row) * 2 * NC + NC + c, tag, __float_as_uint(u));
            } else if (f < a.F) {
                a.act[(size_t)(slot0 + 16 * m + row) * a.F + f] = silu_mul(g, u);
            }
        }
    }
    if (wk.nseg == 1 || !st_last(a.seg_ctr + wk.li, wk.nseg, sh_last)) return;
    const uint64_t *p0 = a.part + (size_t)wk.li * wk.nseg * PSZ;
    constexpr int NC4 = NC / 4;
    for (int i = threadIdx.x; i < 16 * MF * NC4; i += ST_THREADS) {
        const int row = i / NC4, c = 4 * (i - row * NC4);
        if (row >= n) continue;
        const int o[2] = {row * 2 * NC + c, row * 2 * NC + NC + c};
        float gu[2][4];
        if (!st_seg_sum<PSZ, 2>(p0, o, wk.nseg, tag, a.wait_ticks, gu)) atomicOr(a.err, 8u);
        float *dst = a.act + (size_t)(slot0 + row) * a.F + f0 + c;
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (f0 + c + j < a.F) dst[j] = silu_mul(gu[0][j], gu[1][j]);
    }
    st_item_done(a.seg_gen, wk.L, tag);
}

// NFH = 0: the width that the count of row tiles asks for (st_width).
template <int MF, int NFH>
__global__ __launch_bounds__(ST_THREADS, 2) void moe_stream_gateup_kernel(StreamArgs a)
{
    __shared__ __align__(16) char lds[st_lds<NFH ? NFH : ST_GU_MAX>()];
    __shared__ int sh_last;
    const int n = min(*a.n_tiles, a.tile_cap);
    if constexpr (NFH == 0) {
        switch (st_width<ST_GU_MIN, ST_GU_MAX>(n, a.F, a.G)) {
        case 2: st_gateup<1, 2>(a, n, lds, &sh_last); break;
        case 3: st_gateup<1, 3>(a, n, lds, &sh_last); break;
        case 4: st_gateup<1, 4>(a, n, lds, &sh_last); break;
        case 5: st_gateup<1, 5>(a, n, lds, &sh_last); break;
        case 6: st_gateup<1, 6>(a, n, lds, &sh_last); break;
        default: st_gateup<1, 7>(a, n, lds, &sh_last); break;
        }
    } else {
        st_gateup<MF, NFH>(a, n, lds, &sh_last);
    }
}

// ---------------------------------------------------------------------------
// down: 32 NFH output columns from h0 on (halves h0 and h0 + 16 NFH).
// ---------------------------------------------------------------------------
template <int MF, int NFH>
__device__ __forceinline__ void st_down(const StreamArgs &a, int n_tiles, char *lds, int *sh_last)
{
    constexpr int NH = 16 * NFH, NC = 2 * NH;   // columns of a half, of the item
    const int ncg = (a.H + NC - 1) / NC;
    StWork wk;
    if (!st_work(n_tiles * ncg, a.G, a.nbF, ncg, 16 * MF, a.tile_m0, wk)) return;
    const int tile = wk.item / ncg, cg = wk.item - tile * ncg;
    const int e = a.tile_e[tile], m0 = a.tile_m0[tile];
    const int n = min(16 * MF, a.counts[e] - m0);
    const int slot0 = a.offsets[e] + m0;
    const int h0 = cg * NC;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);

    StSrc<MF, NFH> src;
    src.abase = reinterpret_cast<const char *>(a.act);
    const size_t eb = (size_t)e * a.nbF * a.H;
    src.qb[0] = src.qb[1] = a.dq + eb * QK;
    src.db[0] = src.db[1] = a.dd + eb;
    src.qstep = (uint32_t)a.H * QK;
    src.dstep = (uint32_t)a.H;
    const int c0[2] = {h0, h0 + NH};
    st_offsets<MF, NFH>(src, [&](int r) { return (uint32_t)(slot0 + min(r, n - 1)) * a.F * 4; }, c0,
                        a.H, lane);

    f4_t acc[MF][2 * NFH];
#pragma unroll
    for (int m = 0; m < MF; m++)
#pragma unroll
        for (int j = 0; j < 2 * NFH; j++) acc[m][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int kb0 = wk.nseg > 1 ? wk.seg * a.nbF / wk.nseg : 0;
    const int kb1 = wk.nseg > 1 ? (wk.seg + 1) * a.nbF / wk.nseg : a.nbF;
    const uint32_t tag =
        wk.nseg > 1 ? __hip_atomic_load(a.seg_gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u : 0u;
    st_mainloop<MF, NFH>(src, kb0, kb1 - kb0, wave, acc);
    float (*red0)[16][NH + 1] = reinterpret_cast<float (*)[16][NH + 1]>(lds);
    float (*red1)[16][NH + 1] = red0 + 4;
    // split item: partial [16 MF rows][NC columns] of each segment
    constexpr int PSZ = 16 * MF * NC;
    uint64_t *pp = a.part + (size_t)(wk.li * wk.nseg + wk.seg) * PSZ;
#pragma unroll
    for (int m = 0; m < MF; m++) {
        __syncthreads();
        st_spill<MF, NFH>(red0, red1, acc, m, wave, lane);
        __syncthreads();
        // the tile's rows only (a split item's last segment reads those alone)
        const int nr = min(16, n - 16 * m);
        for (int i = threadIdx.x; i < nr * NC; i += ST_THREADS) {
            const int row = i / NC, c = i % NC;
            const int h = h0 + c;
            const float v = wave_order_sum<NFH>(c < NH ? red0 : red1, row, c < NH ? c : c - NH);
            if (wk.nseg > 1)
                store_tagged(pp + (16 * m + row) * NC + c, tag, __float_as_uint(v));
            else if (h < a.H)
                a.y[(size_t)(slot0 + 16 * m + row) * a.H + h] = v;
        }
    }
    if (wk.nseg == 1 || !st_last(a.seg_ctr + wk.li, wk.nseg, sh_last)) return;
    const uint64_t *p0 = a.part + (size_t)wk.li * wk.nseg * PSZ;
    for (int i = threadIdx.x; i < 16 * MF * (NC / 4); i += ST_THREADS) {
        const int row = i / (NC / 4), c = 4 * (i % (NC / 4));
        if (row >= n) continue;
        const int o[1] = {row * NC + c};
        float v[1][4];
        if (!st_seg_sum<PSZ, 1>(p0, o, wk.nseg, tag, a.wait_ticks, v)) atomicOr(a.err, 8u);
        float *dst = a.y + (size_t)(slot0 + row) * a.H + h0 + c;
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (h0 + c + j < a.H) dst[j] = v[0][j];
    }
    st_item_done(a.seg_gen, wk.L, tag);
}

template <int MF, int NFH>
__global__ __launch_bounds__(ST_THREADS, 2) void moe_stream_down_kernel(StreamArgs a)
{
    __shared__ __align__(16) char lds[st_lds<NFH ? NFH : ST_DN_MAX>()];
    __shared__ int sh_last;
    const int n = min(*a.n_tiles, a.tile_cap);
    if constexpr (NFH == 0) {
        switch (st_width<ST_DN_MIN, ST_DN_MAX>(n, a.H / 2, a.G)) {
        case 2: st_down<1, 2>(a, n, lds, &sh_last); break;
        case 3: st_down<1, 3>(a, n, lds, &sh_last); break;
        default: st_down<1, 4>(a, n, lds, &sh_last); break;
        }
    } else {
        st_down<MF, NFH>(a, n, lds, &sh_last);
    }
}

// ---------------------------------------------------------------------------

static size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// slots per tile: 16 for groups of up to ~16 rows on average, else 32
static int stream_mf(const qq_moe *m, int T) { return (size_t)T * m->K <= (size_t)16 * m->E ? 1 : 2; }

static int stream_cap(const qq_moe *m, int T, int bm) { return T * m->K / bm + m->E; }

size_t stream_work_bytes(const qq_moe *m, int T)
{
    const size_t P = (size_t)T * m->K;
    const size_t cap = (size_t)stream_cap(m, T, 16);
    return al256((size_t)m->E * 4) + al256((size_t)(m->E + 1) * 4) + 2 * al256(P * 4) +
           2 * al256(cap * 4) + 256 + al256(P * m->F * 4) + al256(P * m->H * 4);
}

// work: counts | offsets | perm | inv | tile e | tile m0 | tile count | act | y
StreamDispatch stream_dispatch(const qq_moe *m, int T, char *work)
{
    const size_t P = (size_t)T * m->K;
    StreamDispatch d;
    char *p = work;
    d.counts = reinterpret_cast<int32_t *>(p);  p += al256((size_t)m->E * 4);
    d.offsets = reinterpret_cast<int32_t *>(p); p += al256((size_t)(m->E + 1) * 4);
    d.perm = reinterpret_cast<int32_t *>(p);    p += al256(P * 4);
    d.inv = reinterpret_cast<int32_t *>(p);     p += al256(P * 4);
    d.tiles.bm = 16 * stream_mf(m, T);
    d.tiles.cap = stream_cap(m, T, d.tiles.bm);
    d.tiles.e = reinterpret_cast<int32_t *>(p); p += al256((size_t)stream_cap(m, T, 16) * 4);
    d.tiles.m0 = reinterpret_cast<int32_t *>(p);
    p += al256((size_t)stream_cap(m, T, 16) * 4);
    d.tiles.n = reinterpret_cast<int32_t *>(p);
    return d;
}

// Gate/up features per column half of a workgroup, 16 NFH.  Each workgroup
// keeps a fixed number of blocks in flight, so a kernel whose items fill the
// resident slots (2 per CU) only partly in its last round streams that round
// at a fraction of the rate.  The wider items are taken where they need
// fewer item-rounds x width, counting the row tiles of even routing
// (ceil(T K / 16 / E) per expert, clipped to T K / 16 + E).
static int stream_gateup_nfh(const qq_ctx *ctx, const qq_moe *m, int T)
{
    if (stream_mf(m, T) != 1) return 4;
    const long slots = 2L * ctx->num_cus;
    const long per_e = ((long)T * m->K + 16L * m->E - 1) / (16L * m->E);
    const long tiles = std::min((long)stream_cap(m, T, 16), per_e * m->E);
    long best = 0, best_cost = 0;
    for (const int nfh : {4, 7}) {
        const long items = tiles * ((m->F + 16 * nfh - 1) / (16 * nfh));
        const long cost = ((items + slots - 1) / slots) * nfh;
        if (!best || cost < best_cost) {
            best = nfh;
            best_cost = cost;
        }
    }
    return (int)best;
}

// Whether so few experts are expected to be touched that items of `ncg` column
// groups a row tile leave a sixth or more of the resident workgroups without
// one: the launch then takes its width from the tile count (the widths in one
// kernel cost a full launch about 1.5 us: 83.0 -> 85 us at 64 tokens).
static bool stream_few(const qq_ctx *ctx, const qq_moe *m, int T, int ncg)
{
    const double touched = m->E * (1.0 - pow(1.0 - (double)m->K / m->E, (double)T));
    return stream_mf(m, T) == 1 && touched * ncg <= (2.0 * ctx->num_cus) * 5.0 / 6.0;
}

// Workgroups of a launch: 8 * ceil(items / 8) for the most items that a tile
// count up to cap makes, at `ncg` column groups a tile or (few) at the width it takes.
template <int LO, int HI>
static unsigned stream_grid(bool few, int cap, int ncg, int cols, int G)
{
    int items = cap * ncg;
    for (int n = 1; few && n <= cap; n++) {
        const int w = st_width<LO, HI>(n, cols, G);
        items = std::max(items, n * ((cols + 16 * w - 1) / (16 * w)));
    }
    return 8u * (unsigned)((items + 7) / 8);
}

int launch_moe_stream(qq_ctx *ctx, const qq_moe *m, const float *x, float *hidden, int T,
                      const MaskBits &mask, const int32_t *idx, const double *w, char *work,
                      bool dispatched)
{
    const size_t P = (size_t)T * m->K;
    const int MF = stream_mf(m, T);
    const StreamDispatch d = stream_dispatch(m, T, work);
    const int cap = d.tiles.cap;
    int32_t *counts = d.counts, *offsets = d.offsets, *perm = d.perm, *inv = d.inv;
    const DispatchTiles &tiles = d.tiles;
    char *p = work + al256((size_t)m->E * 4) + al256((size_t)(m->E + 1) * 4) + 2 * al256(P * 4) +
              2 * al256((size_t)stream_cap(m, T, 16) * 4) + 256;
    float *act = reinterpret_cast<float *>(p);         p += al256(P * m->F * 4);
    float *y = reinterpret_cast<float *>(p);

    if (!dispatched) {
        const int rc = launch_dispatch(ctx, m, idx, (int)P, mask, counts, offsets, perm, inv, tiles);
        if (rc) return rc;
    }

    StreamArgs a;
    a.x = x;
    a.act = act;
    a.y = y;
    a.perm = perm;
    a.counts = counts;
    a.offsets = offsets;
    a.tile_e = tiles.e;
    a.tile_m0 = tiles.m0;
    a.n_tiles = tiles.n;
    a.gq = m->gate->qs;
    a.uq = m->up->qs;
    a.dq = m->down->qs;
    a.gd = reinterpret_cast<const uint16_t *>(m->gate->d);
    a.ud = reinterpret_cast<const uint16_t *>(m->up->d);
    a.dd = reinterpret_cast<const uint16_t *>(m->down->d);
    a.H = m->H;
    a.F = m->F;
    a.K = m->K;
    a.nbH = m->H / QK;
    a.nbF = m->F / QK;
    a.part = ctx->seg_part;
    a.seg_ctr = ctx->sync_seg;
    a.seg_gen = ctx->sync_seg + SEG_CTR_WORDS / 4;
    a.err = ctx->sync_err;
    a.wait_ticks = ctx->dec_wait_ticks;
    a.G = 2 * ctx->num_cus;
    a.tile_cap = cap;

    // a split item's partial sums: [16 MF rows][2 x 16 NFH columns]
    static_assert(16 * 2 * 16 * ST_GU_MAX <= SEG_PART_WORDS && 16 * 2 * 16 * ST_DN_MAX <= SEG_PART_WORDS &&
                  32 * 2 * 16 * 4 <= SEG_PART_WORDS, "partial sums of a segment");

    // grids (st_work): 8 * ceil(items / 8) workgroups for the items of up to
    // cap row tiles; split items' segments take the room past the items there are
    const int nfh = stream_gateup_nfh(ctx, m, T);
    const int ncg1 = (m->F + 16 * nfh - 1) / (16 * nfh), ncg2 = (m->H + 127) / 128;
    const bool few1 = stream_few(ctx, m, T, ncg1), few2 = stream_few(ctx, m, T, ncg2);
    const dim3 g1(stream_grid<ST_GU_MIN, ST_GU_MAX>(few1, cap, ncg1, m->F, a.G));
    const dim3 g2(stream_grid<ST_DN_MIN, ST_DN_MAX>(few2, cap, ncg2, m->H / 2, a.G));
    prof_begin(ctx, K_STREAM_GATEUP);
    if (few1)
        QQ_LAUNCH(ctx, (moe_stream_gateup_kernel<1, 0>), g1, dim3(ST_THREADS), 0, a);
    else if (MF == 1 && nfh == 7)
        QQ_LAUNCH(ctx, (moe_stream_gateup_kernel<1, 7>), g1, dim3(ST_THREADS), 0, a);
    else if (MF == 1)
        QQ_LAUNCH(ctx, (moe_stream_gateup_kernel<1, 4>), g1, dim3(ST_THREADS), 0, a);
    else
        QQ_LAUNCH(ctx, (moe_stream_gateup_kernel<2, 4>), g1, dim3(ST_THREADS), 0, a);
    prof_end(ctx);
    QQ_HIP(ctx, hipGetLastError());
    prof_begin(ctx, K_STREAM_DOWN);
    a.seg_ctr = ctx->sync_seg + SEG_CTR_WORDS / 2;
    a.seg_gen = ctx->sync_seg + 3 * SEG_CTR_WORDS / 4;
    if (few2)
        QQ_LAUNCH(ctx, (moe_stream_down_kernel<1, 0>), g2, dim3(ST_THREADS), 0, a);
    else if (MF == 1)
        QQ_LAUNCH(ctx, (moe_stream_down_kernel<1, 4>), g2, dim3(ST_THREADS), 0, a);
    else
        QQ_LAUNCH(ctx, (moe_stream_down_kernel<2, 4>), g2, dim3(ST_THREADS), 0, a);
    prof_end(ctx);
    QQ_HIP(ctx, hipGetLastError());
    return launch_combine(ctx, m, T, y, false, inv, w, hidden);
}

}  // namespace qq
