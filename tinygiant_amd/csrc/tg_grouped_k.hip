/*
 * tg_grouped_k.hip -- Q4_K gate/up and Q6_K down expert phases on int8 MFMA
 * for layers whose experts hold many pairs (a prefill, a long verify batch):
 * moe_phase_a / moe_phase_b of csrc/libtinygiant.c:1279-1384 with the
 * per-block dots of dot_q4k_q8 (:223-272) and dot_q6k_q8 (:384-443), the
 * contraction the reference groups four rows at a time (dot_q4k_q8_x4
 * :276-337, dot_q6k_q8_x4 :445-487) done sixteen pairs at a time.
 *
 * Arithmetic.  v_mfma_i32_16x16x32_i8 sums 32 int8 products exactly.  A
 * Q4_K sub-block is 32 values under one 6-bit scale and min, so one MFMA per
 * sub-block gives the reference's integer sums idot for 16 weight rows x 16
 * pairs, and the scale work is the reference's per group g of two
 * sub-blocks, summed here over the block: d * sum_s sc_s idot_s - dmin *
 * sum_s m_s bs_s, both sums exact (int32, and the min sums, a 16 x 16
 * product of 8-long integer vectors, on two f32 MFMAs of K = 4 whose
 * products and sums stay integers below 2^24).  A Q6_K sub-block is 16
 * values under one int8 scale: each 32-value chunk of a half-block runs
 * twice, the pair operand zero in one half of K each time, so the two
 * sub-block sums come out apart; the 6-bit codes enter unshifted and the
 * -32 offset is folded in with the pair's 16-value sums (sum (c - 32) x sc =
 * sum c x sc - 32 sum sc sum x, the last on two f32 MFMAs), exact in int32
 * per half-block.  Only the f32 additions (per block or half-block, then
 * across waves) are associated differently from the reference's
 * sub-block-by-sub-block sum.
 *
 * Operand layout of v_mfma_i32_16x16x32_i8 (measured on gfx950): A lane l =
 * row l % 16 of A, K = 8 (l / 16) + byte; B lane l = column l % 16, the same
 * K; D lane l, register v = A row 4 (l / 16) + v, B column l % 16.  The pairs'
 * q8 operands go in as A and the weight rows as B, so the four sums of a lane
 * share one weight row (lane % 16) and its scales.
 *
 * Work: one workgroup per (16-row slab, active expert).  The slab is staged
 * in LDS (Q6_K blocks re-spaced to 224 bytes so every field is aligned, each
 * load inside its block, since a buffer load that runs past the matrix end
 * reads zero as a whole); the
 * four waves split the row's blocks (Q4_K) or half-blocks (Q6_K); each pass
 * runs 16 pairs of the expert against the resident slab, their q8 operands
 * read from the q8 rows in global memory; 256 threads add the waves' partial
 * sums in wave order and write one result each.  HBM sees each weight byte
 * once however many pairs the expert holds.
 *
 * All this is the form of k_moe_qa and k_moe_qb.  k_moe_qa_ring (scales in the
 * codes, MFMAs of K = 64) and k_moe_qb_ring (the codes, not the pairs, zeroed
 * in one half of K) form the same integer sums, in persistent workgroups.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "tg_device.hpp"
#include "tg_kernels.h"
#include "tg_xchg.hpp"

namespace tg {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

/* four waves a workgroup: three workgroups (twelve waves, three slabs in
 * flight) share a CU, within its LDS; eight waves a workgroup measured 16%
 * slower (two workgroups a CU) */
constexpr int NW = 4;                    /* waves per workgroup */
constexpr int NT = 64 * NW;
constexpr uint32_t OOB = 0x80000000u;    /* past every buffer: the load reads zero */
constexpr uint32_t Q4B = 144, Q6B = 210; /* bytes per 256-value block */
constexpr uint32_t Q6S = 224;            /* LDS stride of a staged Q6_K block */
/* A gate/up wave's q8 operands of a pass are loaded at once: QA_WB Q4_K
 * blocks of a row (D <= 256 NW QA_WB), in a form for Qwen3's 8 blocks of D
 * (fewer registers) and one for longer rows. */
constexpr int QA_WB_MAX = 3;

__device__ inline long as_long(u32x2 v) { return (long)(((uint64_t)v.y << 32) | v.x); }

/* a wave-uniform read of a read-only table through the constant address
 * space: a scalar load, counted apart from the vector loads */
template <class T>
__device__ inline T ldc(const T *p, size_t i) {
    return ((const __attribute__((address_space(4))) T *)(uintptr_t)p)[i];
}

__device__ inline v4i mma(long a, long b) {
    const v4i z = {0, 0, 0, 0};
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, z, 0, 0, 0);
}

/* LDS bytes: the gate and up slabs (rows 16 bytes apart more than their
 * length, so the 16 lanes reading one sub-block of 16 rows hit distinct
 * banks; each slab rounded up to whole 1 KiB copies), then the waves'
 * partial sums.  Q6_K slabs likewise pad each row of blocks by 16 bytes. */
__host__ __device__ inline uint32_t qa_row_stride(int D) { return (uint32_t)(D / 256) * Q4B + 16u; }
__host__ __device__ inline uint32_t qa_slab_region(int D) { return (16u * qa_row_stride(D) + 1023u) & ~1023u; }
__host__ __device__ inline uint32_t qb_row_stride(int I) { return (uint32_t)(I / 256) * Q6S + 16u; }
__host__ __device__ inline size_t qa_lds_bytes(int D) {
    return 2u * (size_t)qa_slab_region(D) + (size_t)NW * 2 * 4 * 64 * 4;
}
__host__ __device__ inline size_t qb_lds_bytes(int I) { return 64u * (size_t)qb_row_stride(I); }

/* 6-bit scales and mins of a Q4_K block header (get_scale_min_k4,
 * csrc/libtinygiant.c:146-155), four bytes at a time: sc of sub-blocks 0-3,
 * 4-7, then the mins */
struct Q4Hdr {
    float d, dmin;
    uint32_t scl, sch, mnl, mnh;
};
__device__ inline Q4Hdr q4_hdr(u32x4 h) {
    Q4Hdr r;
    const uint32_t m4 = 0x0F0F0F0Fu;
    r.d = ref_f16(h.x & 0xFFFFu);
    r.dmin = ref_f16(h.x >> 16);
    r.scl = h.y & 0x3F3F3F3Fu;
    r.mnl = h.z & 0x3F3F3F3Fu;
    r.sch = (h.w & m4) | ((h.y >> 2) & 0x30303030u);
    r.mnh = ((h.w >> 4) & m4) | ((h.z >> 2) & 0x30303030u);
    return r;
}
/* a word's four bytes (each product below 256) times a factor held in both
 * halves of f */
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ inline int mul_bytes(uint32_t q, uint32_t f) {
    return __builtin_bit_cast(int, (u16x2)(__builtin_bit_cast(u16x2, q) * __builtin_bit_cast(u16x2, f)));
}

__device__ inline int byte_of(uint32_t w, int i) { return (int)((w >> (8 * i)) & 0xFFu); }

}  // namespace

/* Phase A: hidden[p][r] = act(gate_r . xq_p + bg[r], up_r . xq_p + bu[r])
 * for rows r of slab blockIdx.x and every pair p of active expert
 * a.ed[blockIdx.y]; Q4_K gate and up matrices of D = 256 nb columns.  The
 * slabs arrive by direct-to-LDS copies, while the first pass's q8 operands
 * load into registers. */
template <int QA_WB>
__global__ __launch_bounds__(NT) void k_moe_qa(MoeArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const ExpDesc &ex = a.ed[blockIdx.y];
    const int e = ex.e, p0 = ex.p0, np = ex.np;
    const int nb = a.D / 256;
    const uint32_t rb = (uint32_t)nb * Q4B, rs = qa_row_stride(a.D), sreg = qa_slab_region(a.D);
    float *red = (float *)(lds + 2 * sreg);   /* [NW][2][4][64] */
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
    const int r0 = blockIdx.x * 16;

    /* the slabs, 1 KiB of LDS a copy: lane l of copy k fills LDS bytes
     * 1024 k + 16 l, i.e. row (1024 k + 16 l) / rs at that column (the row
     * padding and rows past 16 or past I read zero) */
    {
        const uint32_t mbytes = (uint32_t)a.I * rb, base = (uint32_t)r0 * rb, nins = sreg / 1024u;
        const u32x4 gd = buf_desc((const void *)(uintptr_t)ex.gate, mbytes);
        const u32x4 ud = buf_desc((const void *)(uintptr_t)ex.up, mbytes);
        for (uint32_t k = (uint32_t)w; k < nins; k += NW) {
            const uint32_t P = 1024u * k + 16u * (uint32_t)lane, row = P / rs, col = P - row * rs;
            const uint32_t src = row < 16u && col < rb ? base + row * rb + col : OOB;
            copy_lanes_nt(gd, src, lds_addr(lds + 1024u * k));
            copy_lanes_nt(ud, src, lds_addr(lds + sreg + 1024u * k));
        }
    }
    const Q8Rows &q = a.xq;
    const Buf qs_b = make_buf(q.qs, (uint32_t)((size_t)a.k * nb * 256));
    const Buf s32_b = make_buf(q.s32, (uint32_t)((size_t)a.k * nb * 32));
    const Buf d_b = make_buf(q.d, (uint32_t)((size_t)a.k * nb * 4));
    /* the input row of pair t + c16 (0 past the expert's pairs): the 16 rows
     * come through the scalar path, so waiting for them does not wait for
     * the slab copies queued on the vector path */
    auto pair_row = [&](int t) {
        uint32_t rj[16];
#pragma unroll
        for (int j = 0; j < 16; j++) rj[j] = (uint32_t)ldc(a.p_row, (size_t)min(p0 + t + j, a.P - 1));
        uint32_t r = 0u;
#pragma unroll
        for (int j = 0; j < 16; j++) r = c16 == j && t + j < np ? rj[j] : r;
        return r;
    };
    const float *gbias = a.gbias ? (const float *)(uintptr_t)a.gbias[e] : nullptr;
    const float *ubias = a.ubias ? (const float *)(uintptr_t)a.ubias[e] : nullptr;

    /* pair c16's q8 operands of the wave's blocks b = w + NW i of a pass,
     * all loaded at once: sub-block s = 2 jg + half covers x[64 jg + 32 half
     * ...], this lane's K slice 8 g .. 8 g + 7 */
    long xb[QA_WB][8];
    float bsg0[QA_WB], bsg1[QA_WB];   /* the pair's 32-value sums of sub-blocks g and 4 + g */
    float xd[QA_WB];
    auto load_x = [&](uint32_t prow, bool pv) {
#pragma unroll
        for (int i = 0; i < QA_WB; i++) {
            const int b = w + NW * i;
            const bool v = pv && b < nb;
            const uint32_t qb = prow * (uint32_t)nb + (uint32_t)b;
#pragma unroll
            for (int s = 0; s < 8; s++)
                xb[i][s] = as_long(ld8(qs_b, v ? qb * 256u + 64u * (s >> 1) + 32u * (s & 1) + 8u * g : OOB));
            bsg0[i] = (float)(int)ld4(s32_b, v ? qb * 32u + 4u * g : OOB);
            bsg1[i] = (float)(int)ld4(s32_b, v ? qb * 32u + 16u + 4u * g : OOB);
            xd[i] = __uint_as_float(ld4(d_b, v ? qb * 4u : OOB));
        }
    };
    int t0 = 0;
    bool pv = c16 < np;
    uint32_t prow = pair_row(0);
    load_x(prow, pv);
    wait_copies();
    __syncthreads();

    for (;;) {
        float acc[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < QA_WB; i++) {
            const int b = w + NW * i;
            if (b >= nb) break;   /* uniform per wave */
#pragma unroll 1
            for (int m = 0; m < 2; m++) {
                const uint8_t *sb = lds + m * sreg;
                /* the pairs' q8 operands are the MFMA's A side and the weight
                 * rows its B side, so a lane's four sums belong to one row
                 * (c16) and four pairs (4 g + v): one header a lane */
                const Q4Hdr hr = q4_hdr(*(const u32x4 *)(sb + c16 * rs + b * Q4B));
                float xdv[4];
#pragma unroll
                for (int v = 0; v < 4; v++) xdv[v] = __shfl(xd[i], 4 * g + v, 64);
                /* the min terms sum_s bs[pair][s] m[row][s] of the 16 pairs x 16
                 * rows: two f32 MFMAs of K = 4 (sub-blocks g and 4 + g of this
                 * lane group; products and sums are integers below 2^24, exact) */
                v4f im = {0.f, 0.f, 0.f, 0.f};
                im = __builtin_amdgcn_mfma_f32_16x16x4f32(bsg0[i], (float)byte_of(hr.mnl, g), im, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f32_16x16x4f32(bsg1[i], (float)byte_of(hr.mnh, g), im, 0, 0, 0);
                /* the scale terms sum_s sc[row][s] idot[pair][row][s]: one int8
                 * MFMA per sub-block, summed exactly in int32 */
                const uint8_t *ab = sb + c16 * rs + b * Q4B + 16 + 8 * g;   /* row c16's codes */
                int isc[4] = {0, 0, 0, 0};
#pragma unroll
                for (int jg = 0; jg < 4; jg++) {
                    const u32x2 qq = *(const u32x2 *)(ab + 32 * jg);
                    u32x2 lo, hi;
                    lo.x = qq.x & 0x0F0F0F0Fu;
                    lo.y = qq.y & 0x0F0F0F0Fu;
                    hi.x = (qq.x >> 4) & 0x0F0F0F0Fu;
                    hi.y = (qq.y >> 4) & 0x0F0F0F0Fu;
                    const v4i dl = mma(xb[i][2 * jg], as_long(lo));
                    const v4i dh = mma(xb[i][2 * jg + 1], as_long(hi));
                    const uint32_t scw = jg < 2 ? hr.scl : hr.sch;
                    const int s0 = byte_of(scw, 2 * (jg & 1)), s1 = byte_of(scw, 2 * (jg & 1) + 1);
#pragma unroll
                    for (int v = 0; v < 4; v++) isc[v] += __mul24(s0, dl[v]) + __mul24(s1, dh[v]);
                }
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    /* acc indexed with constants only (m is a loop variable) */
                    const float t = xdv[v] * (hr.d * (float)isc[v] - hr.dmin * im[v]);
                    if (m == 0) acc[0][v] += t;
                    else acc[1][v] += t;
                }
            }
        }
        /* the waves' partial sums (block order), then one result per thread */
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int v = 0; v < 4; v++) red[((w * 2 + m) * 4 + v) * 64 + lane] = acc[m][v];
        /* the next pass's q8 operands load while this one is written out */
        const int t1 = t0 + 16;
        if (t1 < np) {
            pv = t1 + c16 < np;
            prow = pair_row(t1);
            load_x(prow, pv);
        }
        __syncthreads();
        if (tid < 256) {
            /* register ev of D lane el: pair 4 (el / 16) + ev, slab row el % 16 */
            const int ev = tid >> 6, el = tid & 63;
            const int jj = t0 + 4 * (el >> 4) + ev, r = r0 + (el & 15);
            if (jj < np && r < a.I) {
                float gv = 0.f, uv = 0.f;
#pragma unroll
                for (int ww = 0; ww < NW; ww++) {
                    gv += red[((ww * 2 + 0) * 4 + ev) * 64 + el];
                    uv += red[((ww * 2 + 1) * 4 + ev) * 64 + el];
                }
                if (gbias) gv += gbias[r];
                if (ubias) uv += ubias[r];
                a.hidden[(size_t)(p0 + jj) * a.I + r] = act_fn(a.act, gv, uv);
            }
        }
        if (t1 >= np) break;
        t0 = t1;
        __syncthreads();   /* red is rewritten by the next pass */
    }
}

/* Phase A, persistent, for Q4_K gate/up rows of D = 2048 (8 blocks): one
 * workgroup a compute unit walks its list of items (active expert, 16-row
 * slab, pass of up to RING_P = 32 pairs), the slabs streaming through a ring
 * of three LDS slots two items ahead of the item computed, so a compute unit
 * always has weight bytes in flight.
 *
 * Eight compute waves: wave c takes matrix c / 4 (gate, up) and blocks
 * c % 4 and c % 4 + 4 of it, so the partial sums of a block pair meet in
 * LDS in the order of the expert-major kernel (wave order).  They hold the
 * q8 operands of a run of items with the same expert and pass, one or two
 * tiles of 16 pairs, loaded once a run (a compute unit returns its loads in
 * issue order, so operands loaded per item would wait behind the slabs in
 * flight each time; for the same reason the loop must hold no spilled
 * register: a scratch reload waits there too); a workgroup's list is a
 * contiguous stretch of the layer's items ordered expert, pass, slab, so it
 * holds a few runs.  They also finish the previous item (its partial sums,
 * double-buffered in LDS, the activation, the hidden values), one result a
 * lane, one barrier an item.  Two copy waves issue the slab copies
 * (direct-to-LDS, one matrix each) and nothing else, so each waits for its
 * own with exact counts.
 *
 * A slab's LDS image swizzles each row's 16-byte units within aligned
 * groups of eight (unit u of row r at 72 r + (u ^ ((r >> 1) & 7))): the 16
 * rows a lane group reads at one column then fall on distinct banks.
 *
 * Bound: an item of one tile takes 1.6 us, the slab's 36 KiB at a compute
 * unit's share of HBM (1.5 us); of two tiles 2.3 us, VALU and MFMA issue of
 * the two compute waves of a SIMD.  With one tile a pass every further 16
 * pairs of an expert streamed its slabs again: 509 tokens (313 passes of 16
 * pairs, 204 of 32) 107 -> 91 us, the layer with both rings 245 -> 194; 33
 * tokens 33 -> 32 us and 80 -> 72. */
constexpr int RG_NB = 8;                              /* Q4_K blocks of a row */
constexpr int RG_UNITS = RG_NB * 9;                   /* 16-byte units of a 1152-byte row */
constexpr int RG_SLAB = 16 * RG_UNITS * 16;           /* 18,432 bytes: one matrix's 16 rows */
constexpr int RG_COPIES = RG_SLAB / 1024;             /* 18 copies of 1 KiB */
constexpr int RG_SLOTS = 3;
constexpr int RG_CW = 8, RG_YW = 2;                   /* compute and copy waves */
constexpr int RG_LC = RG_COPIES;                      /* copies a copy wave issues per item (its matrix's slab) */
constexpr int RG_NT = 64 * (RG_CW + RG_YW);
static_assert((RG_SLOTS - 2) * RG_LC <= 63, "a vmcnt count");
static_assert(RG_SLAB % 1024 == 0, "whole copies");
static_assert(RG_UNITS % 8 == 0, "the swizzle stays inside a row");

__device__ inline uint32_t rg_unit(int r, int u) { return (uint32_t)(RG_UNITS * r + (u ^ ((r >> 1) & 7))); }

struct RgX {   /* a compute lane's q8 operands of one run, blocks c % 4 and c % 4 + 4 of its pair in each tile */
    v4i xb[RING_T][2][2][2];  /* [tile][block][half of the block][low, high nibbles]: 16 values */
    uint32_t bs[RING_T][2];   /* 32-value sums (below 2^13) of sub-blocks g and 4 + g, 16 bits each */
    int nt;   /* tiles that hold pairs */
};

__global__ __launch_bounds__(RG_NT) void k_moe_qa_ring(MoeArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t ring[RG_SLOTS][2][RG_SLAB];
    __shared__ __attribute__((aligned(16))) float red[2][RING_T][RG_CW][4][64];   /* by item parity */
    __shared__ __attribute__((aligned(16))) float xdl[RG_CW][RING_T][2][16];      /* the run's q8 scales */
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4,
              c16 = lane & 15;
    const bool copier = w >= RG_CW;
    const int wg = ring_wg();
    const int i0 = ldc(a.rg_off, wg), n = ldc(a.rg_off, wg + 1) - i0;
    if (n <= 0) return;   /* uniform */
    const uint32_t mbytes = (uint32_t)a.I * (RG_NB * Q4B);
    const Q8Rows &q = a.xq;
    const Buf qs_b = make_buf(q.qs, (uint32_t)((size_t)a.k * RG_NB * 256));
    const Buf s32_b = make_buf(q.s32, (uint32_t)((size_t)a.k * RG_NB * 32));
    const Buf d_b = make_buf(q.d, (uint32_t)((size_t)a.k * RG_NB * 4));
    const int mw = (w >> 2) & 1, bw = w & 3;   /* a compute wave's matrix and first block */

    /* item j of the list (j < n): expert index, slab, pass */
    auto item = [&](int j) { return ldc(a.rg_items, (size_t)(i0 + j)); };
    /* What a copy wave needs of an item comes through the scalar path in
     * stages, each from loads issued an item earlier (an item code, then its
     * expert's entry): a chain of dependent scalar loads in one item's step
     * would stall the wave for each round trip, and the barrier with it. */
    struct Info {   /* its matrix (gate for wave RG_CW, up for the next) and slab */
        uint64_t base;
        int s;
    };
    auto info_code = [&](int it) __attribute__((always_inline)) {
        Info f;
        f.base = w - RG_CW ? ldc(&a.ed[it >> 16].up, 0) : ldc(&a.ed[it >> 16].gate, 0);
        f.s = (it >> 8) & 255;
        return f;
    };
    /* the copy wave's matrix slab of item j, 18 KiB */
    auto issue_copies = [&](int j, const Info &f) __attribute__((always_inline)) {
        const int s = f.s, m = w - RG_CW;
        const u32x4 desc = buf_desc((const void *)(uintptr_t)f.base, mbytes);
        uint8_t *dst = &ring[j % RG_SLOTS][m][0];
#pragma unroll
        for (int k = 0; k < RG_LC; k++) {
            const int P = 64 * k + lane, r = P / RG_UNITS, u = (P % RG_UNITS) ^ ((r >> 1) & 7);
            copy_lanes_nt(desc, (uint32_t)(s * 16 + r) * (RG_NB * Q4B) + 16u * (uint32_t)u, lds_addr(dst + 1024 * k));
        }
    };
    /* the loader wave waits for item j's copies, k items' copies issued after them */
    auto wait_copies_behind = [&](int k) __attribute__((always_inline)) {
        if (k >= 1) wait_copies_but<RG_LC>();
        else wait_copies_but<0>();
    };
    static_assert(RG_SLOTS - 2 == 1, "wait_copies_behind covers the items in flight");
    /* the compute lane's operands of run r: its pair c16 of each tile, whose
     * input row the run's record holds (one round trip of scalar loads) */
    auto load_x = [&](int r, RgX &x) __attribute__((always_inline)) {
        const int *rc = a.rg_runs + (size_t)RING_REC * r;
        const int nv = ldc(rc, 1);
        x.nt = nv > 16 ? 2 : 1;
        uint32_t bs0[RING_T][2], bs1[RING_T][2], xd[RING_T][2];
#pragma unroll
        for (int t = 0; t < RING_T; t++) {
            if (t >= x.nt) break;   /* uniform */
            uint32_t rj[16];
#pragma unroll
            for (int jj = 0; jj < 16; jj++) rj[jj] = (uint32_t)ldc(rc, 2 + 16 * t + jj);
            uint32_t prow = 0u;
#pragma unroll
            for (int jj = 0; jj < 16; jj++) prow = c16 == jj ? rj[jj] : prow;
            const bool pv = 16 * t + c16 < nv;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                /* one offset a lane and buffer, the rest in the instructions */
                const uint32_t qb = prow * RG_NB + (uint32_t)(bw + 4 * h);
                const uint32_t oq = pv ? qb * 256u + 64u * (g >> 1) + 16u * (g & 1) : OOB, os = pv ? qb * 32u + 4u * g : OOB;
#pragma unroll
                for (int s = 0; s < 4; s++)
                    x.xb[t][h][s >> 1][s & 1] = __builtin_bit_cast(v4i, ld16(qs_b, oq + 128u * (s >> 1) + 32u * (s & 1)));
                bs0[t][h] = ld4(s32_b, os);
                bs1[t][h] = ld4(s32_b, os + 16u);
                xd[t][h] = ld4(d_b, pv ? qb * 4u : OOB);
            }
        }
        /* taken as the values of an empty asm statement: the compiler waits
         * for the loads there and not at their uses */
#pragma unroll
        for (int t = 0; t < RING_T; t++) {
            if (t >= x.nt) break;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                v4i(&xb)[2][2] = x.xb[t][h];
                asm volatile(""
                             : "+v"(xb[0][0]), "+v"(xb[0][1]), "+v"(xb[1][0]), "+v"(xb[1][1]), "+v"(bs0[t][h]), "+v"(bs1[t][h]), "+v"(xd[t][h]));
                x.bs[t][h] = (bs0[t][h] & 0xFFFFu) | (bs1[t][h] << 16);
                /* the pairs' scales, where a lane finds those of its four result
                 * pairs side by side (the wave's own words, in order) */
                xdl[w][t][h][c16] = __uint_as_float(xd[t][h]);
            }
        }
    };
    /* compute item j from its slot with operands x: the wave's two blocks of
     * its matrix against NT tiles of pairs, their sums to red.  The codes and
     * scales are unpacked once for all tiles. */
    auto compute = [&](int j, const RgX &x, auto tiles) __attribute__((always_inline)) {
        constexpr int NT_ = decltype(tiles)::value;
        const uint8_t *sb = &ring[j % RG_SLOTS][mw][0];
        /* byte 2 (g / 2) (or the next) of a word of scales in both its halves */
        const uint32_t sel0 = 0x0C000C00u + 0x00020002u * (uint32_t)(g >> 1), sel1 = sel0 + 0x00010001u;
        /* every LDS read of the item first: read where they are used, each
         * would add its latency to the item (12 reads, 2 waves a SIMD) */
        u32x4 hd[2];
        u32x4 qc[2][2];   /* 16 bytes of codes of each half block */
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int b = bw + 4 * h;
            hd[h] = *(const u32x4 *)(sb + 16 * rg_unit(c16, 9 * b));
#pragma unroll
            for (int p = 0; p < 2; p++) qc[h][p] = *(const u32x4 *)(sb + 16 * rg_unit(c16, 9 * b + 1 + 4 * p + g));
        }
        v4f xdv[NT_][2];
#pragma unroll
        for (int t = 0; t < NT_; t++)
#pragma unroll
            for (int h = 0; h < 2; h++) xdv[t][h] = *(const v4f *)&xdl[w][t][h][4 * g];
        __builtin_amdgcn_sched_barrier(0);
        float acc[NT_][4];
#pragma unroll
        for (int t = 0; t < NT_; t++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[t][v] = 0.f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const Q4Hdr hr = q4_hdr(hd[h]);
            /* sum_s sc[row][s] idot[pair][row][s], exact in int32, without a
             * multiply per (pair, row, sub-block): the weight codes are scaled
             * before the product.  A 6-bit scale is 8 h + l, and a code times
             * h or l stays below 128, so x . (q l) and x . (q h) accumulate
             * over the whole block inside the MFMAs and meet at the end as
             * l + 8 h.  The scaling is shared by all pairs.  With the scales
             * inside, one MFMA may mix sub-blocks: a lane takes 16 bytes of
             * codes as they lie (bytes 16 g of half p: 16 values of sub-block
             * 4 p + 2 (g / 2) in the low nibbles, of the next in the high
             * ones), so its q8 values are 16-byte pieces too. */
            v4i il[NT_], ih[NT_];
#pragma unroll
            for (int t = 0; t < NT_; t++) il[t] = ih[t] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const uint32_t sc = p ? hr.sch : hr.scl, s3 = sc & 0x07070707u, s8 = (sc >> 3) & 0x07070707u;
#pragma unroll
                for (int n = 0; n < 2; n++) {
                    u32x4 q4 = qc[h][p];
                    if (n) q4 >>= 4;
                    q4 &= 0x0F0F0F0Fu;
                    const uint32_t fl = __builtin_amdgcn_perm(0u, s3, n ? sel1 : sel0);
                    const uint32_t fh = __builtin_amdgcn_perm(0u, s8, n ? sel1 : sel0);
                    const v4i cl = {mul_bytes(q4.x, fl), mul_bytes(q4.y, fl), mul_bytes(q4.z, fl), mul_bytes(q4.w, fl)};
                    const v4i ch = {mul_bytes(q4.x, fh), mul_bytes(q4.y, fh), mul_bytes(q4.z, fh), mul_bytes(q4.w, fh)};
#pragma unroll
                    for (int t = 0; t < NT_; t++) {
                        il[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.xb[t][h][p][n], cl, il[t], 0, 0, 0);
                        ih[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.xb[t][h][p][n], ch, ih[t], 0, 0, 0);
                    }
                }
            }
            const float m0 = (float)byte_of(hr.mnl, g), m1 = (float)byte_of(hr.mnh, g);
            v4f im[NT_];
#pragma unroll
            for (int t = 0; t < NT_; t++) {
                im[t] = v4f{0.f, 0.f, 0.f, 0.f};
                im[t] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)(int)(int16_t)x.bs[t][h], m0, im[t], 0, 0, 0);
                im[t] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)((int)x.bs[t][h] >> 16), m1, im[t], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < NT_; t++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    acc[t][v] += xdv[t][h][v] * (hr.d * (float)(il[t][v] + 8 * ih[t][v]) - hr.dmin * im[t][v]);
        }
#pragma unroll
        for (int t = 0; t < NT_; t++)
#pragma unroll
            for (int v = 0; v < 4; v++) red[j & 1][t][w][v][lane] = acc[t][v];
    };
    /* finishing item j: a compute wave's lane takes one (pair, row) result,
     * the gate and up waves' sums in wave order, the activation, the hidden
     * value; wave w has tile w / 4, pairs 4 (w % 4) + g and row c16 of the
     * slab, whose sums sit in lane 16 (w % 4) + c16, register g.  (Two
     * finishing waves of their own set the pace: 1.4 us an item of one tile,
     * 2.3 of two, behind compute waves that took 1.4 and 2.0.) */
    struct Done {   /* the item to finish: its first pair, pairs from there, first row, biases */
        int pf, nv, r;
        float gb, ub;
    };
    auto finish = [&](int j, const Done &f) __attribute__((always_inline)) {
        const int t = w >> 2;
        if (16 * t >= f.nv) return;   /* uniform */
        int ln = lane;
        asm volatile("" : "+v"(ln));   /* what follows of it is computed here, not kept in registers */
        const int g = ln >> 4, c16 = ln & 15, jj = 16 * t + 4 * (w & 3) + g;
        const float *p = &red[j & 1][t][0][g][16 * (w & 3) + c16];
        float gv = 0.f, uv = 0.f;
#pragma unroll
        for (int ww = 0; ww < 4; ww++) {
            gv += p[ww * 256];
            uv += p[(4 + ww) * 256];
        }
        if (a.gbias) {
            gv += f.gb;
            uv += f.ub;
        }
        if (jj < f.nv) a.hidden[(size_t)(f.pf + jj) * a.I + f.r + c16] = act_fn(a.act, gv, uv);
    };
    /* a run: items of one expert and pass */
    auto run_end = [&](int s) { return min(ldc(a.rg_rend, (size_t)(i0 + s)), i0 + n) - i0; };

    /* The two roles run loops of their own (so the compiler's waits for the
     * compute waves' operand loads never land in the copy waves' code),
     * meeting at one barrier an item.  Between the barriers of items i and
     * i + 1 the compute waves finish item i - 1 (reading red[(i - 1) % 2]) and
     * compute item i (reading slot i % RG_SLOTS, writing red[i % 2]) while
     * the copy waves copy item i + 2 into item i - 1's slot: each wave
     * reaches the next barrier only after its part. */
    if (copier) {
        for (int j = 0; j < RG_SLOTS - 1 && j < n; j++) issue_copies(j, info_code(item(j)));
        Info fc = info_code(item(min(RG_SLOTS - 1, n - 1)));   /* item i + RG_SLOTS - 1 */
        int code = item(min(RG_SLOTS, n - 1));                  /* item i + RG_SLOTS */
        for (int i = 0; i < n; i++) {
            wait_copies_behind(min(RG_SLOTS - 2, n - 1 - i));
            /* a copy wave writes no LDS itself: its barrier leaves the scalar
             * reads of the next items' info in flight */
            asm volatile("s_barrier" ::: "memory");
            if (i + RG_SLOTS - 1 < n) issue_copies(i + RG_SLOTS - 1, fc);
            fc = info_code(code);
            code = item(min(i + RG_SLOTS + 1, n - 1));
        }
        asm volatile("s_barrier" ::: "memory");
        wait_copies();   /* no copy outlives the workgroup */
        return;
    }
    /* A run's operands are loaded when it starts, behind the slabs in flight.
     * (Loading them three items earlier into registers of their own did not
     * shorten the wait: their bytes only delay the slabs; two tiles leave no
     * registers for it.) */
    RgX cur;
    Done done = {0, 0, 0, 0.f, 0.f};
    int run = ldc(a.rg_run0, wg);   /* the run of item 0; the runs follow in order */
    int slab = (item(0) >> 8) & 255;
    for (int i = 0; i < n; run++, slab = 0) {
        load_x(run, cur);
        const int re = run_end(i);
        const int *rc = a.rg_runs + (size_t)RING_REC * run;
        const int pf = ldc(rc, 0), nv = ldc(rc, 1), e = ldc(rc, 2 + RING_P);
        /* a null entry: an empty buffer, which reads zero */
        const uint64_t qg = a.gbias ? ldc(a.gbias, e) : 0, qu = a.ubias ? ldc(a.ubias, e) : 0;
        const Buf gb = make_buf((const void *)(uintptr_t)qg, qg ? (uint32_t)a.I * 4u : 0u);
        const Buf ub = make_buf((const void *)(uintptr_t)qu, qu ? (uint32_t)a.I * 4u : 0u);
        auto step = [&](auto tiles) __attribute__((always_inline)) {
            for (; i < re; i++, slab++) {
                bar_lds();   /* item i's slab has landed, item i - 1's sums are in LDS */
                finish(i - 1, done);   /* nothing before the first item: no pairs */
                done.pf = pf;
                done.nv = nv;
                done.r = 16 * slab;
                if (a.gbias) {   /* both or neither */
                    done.gb = __uint_as_float(ld4(gb, (uint32_t)(16 * slab + c16) * 4u));
                    done.ub = __uint_as_float(ld4(ub, (uint32_t)(16 * slab + c16) * 4u));
                }
                compute(i, cur, tiles);
            }
        };
        if (cur.nt == 1) step(std::integral_constant<int, 1>());
        else step(std::integral_constant<int, 2>());
    }
    bar_lds();   /* item n - 1's sums are in LDS */
    finish(n - 1, done);
}

/* Phase B: part[p][r] = w_p * (down_r . hq_p + bd[r]) for the 64 rows r of
 * slab blockIdx.x and every pair p of active expert a.ed[blockIdx.y]; Q6_K
 * down matrix of I = 256 nbi columns.  Wave w owns rows 16 w .. 16 w + 15 of
 * the slab over the whole row, so its MFMA sums are the rows' results and no
 * partial sums cross waves.  The slab's loads go out first, then the first
 * pass's q8 operands, then the slab is stored to LDS. */
constexpr int QB_ROWS = 64;                 /* rows of a down slab: one 16-row tile a wave */
constexpr int QB_PIECES = 13;               /* 16-byte pieces of a block's bytes 0-207 */
constexpr int QB_NPC = 10;                  /* pieces per thread in flight while the slab is staged */
constexpr int QB_CH = 6;                    /* half-blocks whose q8 operands a wave holds at once */
template <int>
__global__ __launch_bounds__(NT) void k_moe_qb(MoeArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const ExpDesc &ex = a.ed[blockIdx.y];
    const int e = ex.e, p0 = ex.p0, np = ex.np;
    const int nbi = a.I / 256, nhb = 2 * nbi;
    /* n / nbi for the slab's block indices n < 64 * 12 as (n * inv) >> 16:
     * inv exceeds 2^16 / nbi by less than 1, so the product's error stays
     * below 768 / 2^16 < 1 / nbi */
    const uint32_t inv = (65536u + (uint32_t)nbi - 1u) / (uint32_t)nbi;
    auto div_nbi = [&](int n) { return (int)(((uint32_t)n * inv) >> 16); };
    const uint32_t rb = (uint32_t)nbi * Q6B, rs = qb_row_stride(a.I);
    /* LDS offset of block blk of slab row row */
    auto blk_at = [&](int row, int blk) { return (uint32_t)row * rs + (uint32_t)blk * Q6S; };
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4,
              c16 = lane & 15;
    const int r0 = blockIdx.x * QB_ROWS;

    /* the slab, each block at a 224-byte stride: bytes 0-207 as 13 pieces,
     * then d at 208 (a load that ran past byte 209 would read zero in the
     * matrix's last block; rows past D read zero) */
    const Buf dw = make_buf_uniform((const void *)(uintptr_t)ex.down, (uint32_t)a.D * rb);
    const int nch = QB_ROWS * nbi * QB_PIECES;
    auto piece_src = [&](int c) {
        const int piece = c % QB_PIECES, rbk = c / QB_PIECES, row = div_nbi(rbk), blk = rbk - row * nbi;
        return (uint32_t)(r0 + row) * rb + (uint32_t)blk * Q6B + 16u * piece;
    };
    auto piece_dst = [&](int c) {
        const int rbk = c / QB_PIECES, row = div_nbi(rbk);
        return blk_at(row, rbk - row * nbi) + 16 * (c % QB_PIECES);
    };
    u32x4 pc[QB_NPC];
#pragma unroll
    for (int i = 0; i < QB_NPC; i++) {
        const int c = tid + NT * i;
        pc[i] = ld16(dw, c < nch ? piece_src(c) : OOB);
    }
    uint32_t dd[(QB_ROWS * 12 + NT - 1) / NT];   /* d of the slab's blocks (I <= 3072) */
#pragma unroll
    for (int i = 0; i < (QB_ROWS * 12 + NT - 1) / NT; i++) {
        const int rbk = tid + NT * i;
        const int row = div_nbi(rbk);
        dd[i] = rbk < QB_ROWS * nbi ? ld2(dw, (uint32_t)(r0 + row) * rb + (uint32_t)(rbk - row * nbi) * Q6B + 208u) : 0u;
    }

    const Q8Rows &q = a.hq;
    const Buf qs_b = make_buf(q.qs, (uint32_t)((size_t)a.P * nbi * 256));
    const Buf s16_b = make_buf(q.s16, (uint32_t)((size_t)a.P * nbi * 64));
    const Buf d_b = make_buf(q.d, (uint32_t)((size_t)a.P * nbi * 4));
    const Buf pw_b = make_buf(a.p_w, (uint32_t)a.P * 4u);
    const float *dbias = a.dbias ? (const float *)(uintptr_t)a.dbias[e] : nullptr;
    /* pair c16's q8 operands of half-blocks c0 .. c0 + QB_CH - 1: chunk m of
     * half h of block bi covers x[128 h + 32 m ...], this lane's K slice
     * 8 g .. 8 g + 7; the 16-value sums of sub-blocks 8 h + g and 8 h + 4 + g */
    long xb[QB_CH][4];
    int s16g[QB_CH][2];
    float xd[QB_CH];
    auto load_x = [&](uint32_t prow, bool pv, int c0) {
#pragma unroll
        for (int i = 0; i < QB_CH; i++) {
            const int hb = c0 + i;
            const bool v = pv && hb < nhb;
            const int bi = hb >> 1, h = hb & 1;
            const uint32_t qb = prow * (uint32_t)nbi + (uint32_t)bi;
#pragma unroll
            for (int m = 0; m < 4; m++)
                xb[i][m] = as_long(ld8(qs_b, v ? qb * 256u + 128u * h + 32u * m + 8u * g : OOB));
            /* each its own load: a select among loaded words would wait for the load */
            s16g[i][0] = (int)ld4(s16_b, v ? qb * 64u + 32u * h + 4u * g : OOB);
            s16g[i][1] = (int)ld4(s16_b, v ? qb * 64u + 32u * h + 16u + 4u * g : OOB);
            xd[i] = __uint_as_float(ld4(d_b, v ? qb * 4u : OOB));
        }
    };
    int t0 = 0;
    bool pv = c16 < np;
    uint32_t prow = (uint32_t)(pv ? p0 + c16 : 0);
    load_x(prow, pv, 0);
#pragma unroll
    for (int i = 0; i < QB_NPC; i++) {
        const int c = tid + NT * i;
        if (c < nch) *(u32x4 *)(lds + piece_dst(c)) = pc[i];
    }
    for (int c = tid + NT * QB_NPC; c < nch; c += NT)   /* rows of more than 3 blocks */
        *(u32x4 *)(lds + piece_dst(c)) = ld16(dw, piece_src(c));
#pragma unroll
    for (int i = 0; i < (QB_ROWS * 12 + NT - 1) / NT; i++) {
        const int rbk = tid + NT * i;
        const int row = div_nbi(rbk);
        if (rbk < QB_ROWS * nbi) *(uint32_t *)(lds + blk_at(row, rbk - row * nbi) + 208) = dd[i];
    }
    __syncthreads();

    const int tr = 16 * w;   /* the wave's first slab row */
    for (;;) {
        /* the weights of the lane's four pairs, waited for only at the end */
        float pwv[4];
#pragma unroll
        for (int v = 0; v < 4; v++)
            pwv[v] = __uint_as_float(ld4(pw_b, t0 + 4 * g + v < np ? (uint32_t)(p0 + t0 + 4 * g + v) * 4u : OOB));
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
        for (int c0 = 0; c0 < nhb; c0 += QB_CH) {
            if (c0 > 0) load_x(prow, pv, c0);   /* rows of more than 3 blocks */
#pragma unroll
            for (int i = 0; i < QB_CH; i++) {
                const int hb = c0 + i;
                if (hb >= nhb) break;   /* uniform */
                const int bi = hb >> 1, h = hb & 1;
                /* row c16's codes: ql bytes 64 h + 32 (m & 1) + 8 g, qh bytes 32 h + 8 g */
                const uint8_t *ab = lds + blk_at(tr + c16, bi);
                const u32x2 ql0 = *(const u32x2 *)(ab + 64 * h + 8 * g);
                const u32x2 ql1 = *(const u32x2 *)(ab + 64 * h + 32 + 8 * g);
                const u32x2 qh = *(const u32x2 *)(ab + 128 + 32 * h + 8 * g);
                /* the pairs' q8 operands are the MFMA's A side and the weight
                 * rows its B side, so a lane's four sums belong to row c16
                 * and pairs 4 g + v: its scales are row c16's */
                const u32x2 scr = *(const u32x2 *)(ab + 192 + 8 * h);   /* sub-block scales 8 h .. 8 h + 7 */
                const float dv = ref_f16(*(const uint32_t *)(ab + 208) & 0xFFFFu);
                float xdv[4];
#pragma unroll
                for (int v = 0; v < 4; v++) xdv[v] = __shfl(xd[i], 4 * g + v, 64);
                /* the -32 offset terms sum_s s16[pair][s] sc[row][s] over the
                 * half's 8 sub-blocks: two f32 MFMAs of K = 4 (sub-blocks g
                 * and 4 + g; integers below 2^24, exact) */
                v4f cf = {0.f, 0.f, 0.f, 0.f};
                cf = __builtin_amdgcn_mfma_f32_16x16x4f32((float)s16g[i][0], (float)(int8_t)(scr.x >> (8 * g)), cf, 0,
                                                          0, 0);
                cf = __builtin_amdgcn_mfma_f32_16x16x4f32((float)s16g[i][1], (float)(int8_t)(scr.y >> (8 * g)), cf, 0,
                                                          0, 0);
                int ai[4] = {0, 0, 0, 0};
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const u32x2 ql = (m & 1) ? ql1 : ql0;
                    const int sl = 4 * (m >> 1), sh = 2 * m;
                    u32x2 c;
                    c.x = ((ql.x >> sl) & 0x0F0F0F0Fu) | (((qh.x >> sh) & 0x03030303u) << 4);
                    c.y = ((ql.y >> sl) & 0x0F0F0F0Fu) | (((qh.y >> sh) & 0x03030303u) << 4);
                    /* K slots 0-15 (lane groups 0, 1) are sub-block 2 m, 16-31 sub-block 2 m + 1 */
                    const long x0 = g < 2 ? xb[i][m] : 0l, x1 = g < 2 ? 0l : xb[i][m];
                    const v4i d0 = mma(x0, as_long(c)), d1 = mma(x1, as_long(c));
                    const uint32_t sw = m < 2 ? scr.x : scr.y;
                    const int sc0 = (int)(int8_t)(sw >> (16 * (m & 1))), sc1 = (int)(int8_t)(sw >> (16 * (m & 1) + 8));
#pragma unroll
                    for (int v = 0; v < 4; v++) ai[v] += __mul24(sc0, d0[v]) + __mul24(sc1, d1[v]);   /* |.| < 2^24 */
                }
                /* sum (c - 32) x sc, exact in int32 */
#pragma unroll
                for (int v = 0; v < 4; v++) acc[v] += dv * xdv[v] * (float)(ai[v] - 32 * (int)cf[v]);
            }
        }
        /* row r0 + tr + c16 of pairs t0 + 4 g + v, in the half-blocks' order */
        const int r = r0 + tr + c16;
        if (r < a.D) {
            const float bias = dbias ? dbias[r] : 0.f;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int jj = t0 + 4 * g + v;
                if (jj < np) a.part[(size_t)(p0 + jj) * a.D + r] = pwv[v] * (acc[v] + bias);
            }
        }
        t0 += 16;
        if (t0 >= np) break;
        pv = t0 + c16 < np;
        prow = (uint32_t)(pv ? p0 + t0 + c16 : 0);
        load_x(prow, pv, 0);
    }
}

/* Phase B, persistent, for Q6_K down rows of I = 768 (3 blocks, 630 bytes
 * a row) without a down bias: one workgroup a compute unit walks its list
 * of items (active expert, 32-row slab, pass of up to 32 pairs), the slabs
 * (20,160 contiguous bytes) streaming through a ring of five LDS slots four
 * items ahead, as the gate/up ring does.  Twelve compute waves take one
 * 128-value half-block of one 16-row tile each (wave c: half-block c % 6,
 * block c % 6 / 2, tile c / 6; three a SIMD), with k_moe_qb's arithmetic,
 * and leave each
 * half-block's term d x d_x x (sum - 32 x offsets) in LDS.  Two copy waves
 * issue the slab copies and wait for them with exact counts (they issue no
 * other memory operation, which would enter the counts).  The compute waves
 * also finish the previous item: the six terms added in half-block order
 * (k_moe_qb's order), times the pair's weight (two finishing waves took as
 * long as an item's copies and products: 103 -> 86 us at 509 tokens with
 * their work left out).  The slab
 * keeps the matrix's layout in LDS (the copies read 16-byte-aligned sources
 * only), so fields of odd rows and odd blocks lie at 2 mod 4 and are read
 * as covering dwords, shifted. */
constexpr int DR_NB = 3;                                  /* Q6_K blocks of a 768-value row */
constexpr int DR_RB = DR_NB * (int)Q6B;                   /* 630 bytes a row */
constexpr int DR_ROWS = 32;
constexpr int DR_SLAB = DR_ROWS * DR_RB;                  /* 20,160 bytes */
constexpr int DR_COPIES = (DR_SLAB + 1023) / 1024;        /* 20 copies, the last of DR_LAST lanes */
constexpr int DR_LAST = (DR_SLAB - 1024 * (DR_COPIES - 1)) / 16;
constexpr int DR_SLOTS = 5;
constexpr int DR_HB = 2 * DR_NB;                        /* half-blocks of a row */
constexpr int DR_CW = 2 * DR_HB, DR_YW = 2;             /* compute and copy waves */
constexpr int DR_LC = DR_COPIES / DR_YW;                  /* copies a copy wave issues per item */
constexpr int DR_NT = 64 * (DR_CW + DR_YW);
static_assert(DR_SLAB % 16 == 0 && DR_LAST > 0 && DR_LAST <= 64, "whole 16-byte pieces");
static_assert(DR_COPIES % DR_YW == 0, "equal copy counts per copy wave");
static_assert((DR_SLOTS - 2) * DR_LC <= 63, "a vmcnt count");

/* 8 bytes at LDS offset o (o even) of base: the covering dwords, then the
 * bytes shifted out of them (o and `at` alike mod 4) */
struct Dr8 {
    uint32_t d0, d1, d2;
};
__device__ inline Dr8 dr_read8(const uint8_t *base, uint32_t o) {
    const uint32_t *p = (const uint32_t *)(base + (o & ~3u));
    return Dr8{p[0], p[1], p[2]};
}
__device__ inline u32x2 dr_shift8(const Dr8 &d, uint32_t at) {
    return u32x2{__builtin_amdgcn_alignbyte(d.d1, d.d0, at & 3u), __builtin_amdgcn_alignbyte(d.d2, d.d1, at & 3u)};
}

struct DrX {   /* a compute lane's q8 operands of one run: pair c16 of each tile, its wave's half-block */
    long xb[RING_T][4];   /* K slice 8 g of chunk m */
    float s16a[RING_T], s16b[RING_T], xd[RING_T];
    int nt;                              /* tiles that hold pairs */
};

__global__ __launch_bounds__(DR_NT) void k_moe_qb_ring(MoeArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t ring[DR_SLOTS][DR_SLAB];
    __shared__ __attribute__((aligned(16))) float red[2][RING_T][DR_HB][2][4][64];   /* by item parity */
    __shared__ __attribute__((aligned(16))) float xdl[DR_CW][RING_T][16];            /* the run's q8 scales */
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4,
              c16 = lane & 15;
    const bool copier = w >= DR_CW;
    const int wg = ring_wg();
    const int i0 = ldc(a.rb_off, wg), n = ldc(a.rb_off, wg + 1) - i0;
    if (n <= 0) return;   /* uniform */
    const uint32_t mbytes = (uint32_t)a.D * DR_RB;
    const Q8Rows &q = a.hq;
    const Buf qs_b = make_buf(q.qs, (uint32_t)((size_t)a.P * DR_NB * 256));
    const Buf s16_b = make_buf(q.s16, (uint32_t)((size_t)a.P * DR_NB * 64));
    const Buf d_b = make_buf(q.d, (uint32_t)((size_t)a.P * DR_NB * 4));
    const Buf pw_b = make_buf(a.p_w, (uint32_t)a.P * 4u);
    const int hbw = w % DR_HB, bi = hbw >> 1, h = hbw & 1, tw = w / DR_HB;   /* a compute wave's half-block, tile */

    auto item = [&](int j) { return ldc(a.rb_items, (size_t)(i0 + j)); };
    /* What a copy wave needs of an item comes through the scalar path in
     * stages, each from loads issued an item earlier: an item code, then its
     * expert's table entry.  A chain of dependent scalar loads in one item's
     * step would stall the wave for each load's round trip (about a
     * microsecond under the weight stream) and the barrier with it. */
    struct Info {   /* the matrix and slab */
        uint64_t base;
        int s;
    };
    auto info_code = [&](int it) __attribute__((always_inline)) {
        Info f;
        f.base = ldc(&a.ed[it >> 16].down, 0);
        f.s = (it >> 8) & 255;
        return f;
    };
    /* the copy wave's share of item j's copies */
    auto issue_copies = [&](int j, const Info &f) __attribute__((always_inline)) {
        const u32x4 desc = buf_desc((const void *)(uintptr_t)f.base, mbytes);
        uint8_t *dst = &ring[j % DR_SLOTS][0];
        const uint32_t src = (uint32_t)f.s * DR_SLAB + 16u * (uint32_t)lane;
#pragma unroll
        for (int kk = 0; kk < DR_LC; kk++) {
            const int k = DR_LC * (w - DR_CW) + kk;
            if (k < DR_COPIES - 1 || lane < DR_LAST) copy_lanes_nt(desc, src + 1024u * k, lds_addr(dst + 1024 * k));
        }
    };
    auto wait_copies_behind = [&](int k) __attribute__((always_inline)) {
        if (k >= 3) wait_copies_but<3 * DR_LC>();
        else if (k == 2) wait_copies_but<2 * DR_LC>();
        else if (k == 1) wait_copies_but<DR_LC>();
        else wait_copies_but<0>();
    };
    static_assert(DR_SLOTS - 2 == 3, "wait_copies_behind covers the items in flight");
    /* the compute lane's operands of run r: its pair c16 of each tile (the
     * run's first pair and count from its record) */
    auto load_x = [&](int r, DrX &x) __attribute__((always_inline)) {
        const int *rc = a.rb_runs + (size_t)RING_REC * r;
        const int pf = ldc(rc, 0), nv = ldc(rc, 1);
        x.nt = nv > 16 ? 2 : 1;
#pragma unroll
        for (int t = 0; t < RING_T; t++) {
            if (t >= x.nt) break;   /* uniform */
            const bool pv = 16 * t + c16 < nv;
            const uint32_t qb = (uint32_t)(pf + 16 * t + c16) * DR_NB + (uint32_t)bi;
            const uint32_t oq = pv ? qb * 256u + 128u * h + 8u * g : OOB, os = pv ? qb * 64u + 32u * h + 4u * g : OOB;
#pragma unroll
            for (int m = 0; m < 4; m++) x.xb[t][m] = as_long(ld8(qs_b, oq + 32u * m));
            x.s16a[t] = (float)(int)ld4(s16_b, os);
            x.s16b[t] = (float)(int)ld4(s16_b, os + 16u);
            x.xd[t] = __uint_as_float(ld4(d_b, pv ? qb * 4u : OOB));
        }
    };
    /* compute item j from its slot: the wave's half-block of its row tile
     * against NT tiles of pairs, the codes unpacked once for all of them */
    auto compute = [&](int j, const DrX &x, auto tiles) __attribute__((always_inline)) {
        constexpr int NT_ = decltype(tiles)::value;
        const uint8_t *sb = &ring[j % DR_SLOTS][0];
        const uint32_t lo = g < 2 ? ~0u : 0u;
        const uint32_t rb = (uint32_t)(16 * tw + c16) * DR_RB + (uint32_t)bi * Q6B;   /* row c16's block */
        /* every LDS read of the item first */
        const Dr8 r0 = dr_read8(sb, rb + 64u * h + 8u * g), r1 = dr_read8(sb, rb + 64u * h + 32u + 8u * g);
        const Dr8 r2 = dr_read8(sb, rb + 128u + 32u * h + 8u * g), r3 = dr_read8(sb, rb + 192u + 8u * h);
        const uint32_t dw = *(const uint32_t *)(sb + ((rb + 208u) & ~3u));
        __builtin_amdgcn_sched_barrier(0);
        const u32x2 ql0 = dr_shift8(r0, rb), ql1 = dr_shift8(r1, rb), qh = dr_shift8(r2, rb), scr = dr_shift8(r3, rb);
        const float dv = ref_f16((rb & 2u) ? (dw >> 16) : (dw & 0xFFFFu));
        const float sa = (float)(int8_t)(scr.x >> (8 * g)), sb4 = (float)(int8_t)(scr.y >> (8 * g));
        v4f cf[NT_];
        int ai[NT_][4];
#pragma unroll
        for (int t = 0; t < NT_; t++) {
            cf[t] = v4f{0.f, 0.f, 0.f, 0.f};
            cf[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.s16a[t], sa, cf[t], 0, 0, 0);
            cf[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.s16b[t], sb4, cf[t], 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) ai[t][v] = 0;
        }
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const u32x2 ql = (m & 1) ? ql1 : ql0;
            const int sl = 4 * (m >> 1), sh = 2 * m;
            u32x2 c;
            c.x = ((ql.x >> sl) & 0x0F0F0F0Fu) | (((qh.x >> sh) & 0x03030303u) << 4);
            c.y = ((ql.y >> sl) & 0x0F0F0F0Fu) | (((qh.y >> sh) & 0x03030303u) << 4);
            /* K slots 0-15 (lane groups 0, 1) are sub-block 2 m, 16-31
             * sub-block 2 m + 1: the codes are zeroed in one half of K */
            const u32x2 c0 = {c.x & lo, c.y & lo}, c1 = {c.x & ~lo, c.y & ~lo};
            const uint32_t sw = m < 2 ? scr.x : scr.y;
            const int sc0 = (int)(int8_t)(sw >> (16 * (m & 1))), sc1 = (int)(int8_t)(sw >> (16 * (m & 1) + 8));
            if (NT_ > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < NT_; t++) {
                const v4i d0 = mma(x.xb[t][m], as_long(c0)), d1 = mma(x.xb[t][m], as_long(c1));
#pragma unroll
                for (int v = 0; v < 4; v++) ai[t][v] += __mul24(sc0, d0[v]) + __mul24(sc1, d1[v]);   /* |.| < 2^24 */
            }
        }
#pragma unroll
        for (int t = 0; t < NT_; t++) {
            const v4f xdv = *(const v4f *)&xdl[w][t][4 * g];   /* of pairs 4 g .. 4 g + 3 */
#pragma unroll
            for (int v = 0; v < 4; v++)
                red[j & 1][t][hbw][tw][v][lane] = dv * xdv[v] * (float)(ai[t][v] - 32 * (int)cf[t][v]);
        }
    };
    /* finishing item j: a compute lane takes one or two (pair, row) results
     * o = tid and tid + 64 DR_CW of the slab (tile of pairs o / 512, row tile
     * o / 256 % 2, pair o / 16 % 16, row o % 16): the six half-block terms in
     * order, times the pair's weight; the term of pair 4 g + v and row c16
     * sits in lane 16 g + c16, register v */
    struct Done {   /* the item to finish: its first pair, pairs from there, first row, the lane's pair weights */
        int pf, nv, r;
        float pw[2];
    };
    auto out_pair = [&](int u) { return 16 * ((tid + 64 * DR_CW * u) >> 9) + (((tid + 64 * DR_CW * u) >> 4) & 15); };
    auto finish = [&](int j, const Done &f) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int ow = w + DR_CW * u;   /* o / 64, uniform */
            if (ow >= 8 * RING_T || 16 * (ow >> 3) >= f.nv) break;
            int lx = lane;
            asm volatile("" : "+v"(lx));   /* what follows of it is computed here, not kept in registers */
            const int t = ow >> 3, tq = (ow >> 2) & 1, v = lx >> 4, c16 = lx & 15, jj = 4 * (ow & 3) + v;
            const int ln = 16 * (ow & 3) + c16;
            float acc = 0.f;
#pragma unroll
            for (int c = 0; c < DR_HB; c++) acc += red[j & 1][t][c][tq][v][ln];
            if (16 * t + jj < f.nv) a.part[(size_t)(f.pf + 16 * t + jj) * a.D + f.r + 16 * tq + c16] = f.pw[u] * (acc + 0.f);
        }
    };
    auto run_end = [&](int s0) { return min(ldc(a.rb_rend, (size_t)(i0 + s0)), i0 + n) - i0; };

    /* as in the gate/up ring: between the barriers of items i and i + 1 the
     * compute waves finish item i - 1 (red[(i - 1) % 2]) and compute item i
     * (slot i % DR_SLOTS, red[i % 2]) while the copy waves copy item
     * i + DR_SLOTS - 1 into item i - 1's slot */
    if (copier) {
        for (int j = 0; j < DR_SLOTS - 1 && j < n; j++) issue_copies(j, info_code(item(j)));
        Info fc = info_code(item(min(DR_SLOTS - 1, n - 1)));   /* item i + DR_SLOTS - 1 */
        int code = item(min(DR_SLOTS, n - 1));                  /* item i + DR_SLOTS */
        for (int i = 0; i < n; i++) {
            wait_copies_behind(min(DR_SLOTS - 2, n - 1 - i));
            asm volatile("s_barrier" ::: "memory");   /* a copy wave writes no LDS itself */
            if (i + DR_SLOTS - 1 < n) issue_copies(i + DR_SLOTS - 1, fc);
            fc = info_code(code);
            code = item(min(i + DR_SLOTS + 1, n - 1));
        }
        asm volatile("s_barrier" ::: "memory");
        wait_copies();   /* no copy outlives the workgroup */
        return;
    }
    auto settle = [&](DrX &x) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < RING_T; t++) {
            if (t >= x.nt) break;
            long(&xb)[4] = x.xb[t];
            asm volatile(""
                         : "+v"(xb[0]), "+v"(xb[1]), "+v"(xb[2]), "+v"(xb[3]), "+v"(x.s16a[t]), "+v"(x.s16b[t]),
                           "+v"(x.xd[t]));
            xdl[w][t][c16] = x.xd[t];   /* the wave's own words, in order */
        }
    };
    DrX cur;
    Done done = {0, 0, 0, {0.f, 0.f}};
    int run = ldc(a.rb_run0, wg);   /* the run of item 0; the runs follow in order */
    int slab = (item(0) >> 8) & 255;
    for (int i = 0; i < n; run++, slab = 0) {
        load_x(run, cur);
        const int re = run_end(i);
        const int *rc = a.rb_runs + (size_t)RING_REC * run;
        const int pf = ldc(rc, 0), nv = ldc(rc, 1);
        float pw[2];
#pragma unroll
        for (int u = 0; u < 2; u++)
            pw[u] = __uint_as_float(ld4(pw_b, out_pair(u) < nv ? (uint32_t)(pf + out_pair(u)) * 4u : OOB));
        settle(cur);
        asm volatile("" : "+v"(pw[0]), "+v"(pw[1]));
        auto step = [&](auto tiles) __attribute__((always_inline)) {
            for (; i < re; i++, slab++) {
                bar_lds();   /* item i's slab has landed, item i - 1's terms are in LDS */
                finish(i - 1, done);   /* nothing before the first item: no pairs */
                done = Done{pf, nv, DR_ROWS * slab, {pw[0], pw[1]}};
                compute(i, cur, tiles);
            }
        };
        if (cur.nt == 1) step(std::integral_constant<int, 1>());
        else step(std::integral_constant<int, 2>());
    }
    bar_lds();   /* item n - 1's terms are in LDS */
    finish(n - 1, done);
}

bool qb_ring_shape(int I, int D) { return I == DR_NB * 256 && D % DR_ROWS == 0 && D / DR_ROWS <= 256; }

/* The MFMA phases need Q4_K gate/up and Q6_K down matrices of whole blocks,
 * slabs within the device's LDS, and 31-bit buffer ranges. */
bool qk_grouped_fits(const MoeArgs &a) {
    static int max_lds = -1;
    if (max_lds < 0) {
        int dev = 0;
        max_lds = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
            max_lds = 0;
    }
    if (a.gate_fmt != TG_FMT_Q4K || a.D % 256 || a.I % 256 || a.n_act_a <= 0) return false;
    if (a.D > 256 * NW * QA_WB_MAX || a.I > 3072) return false;   /* a pass's operands and the slab's d in registers */
    const uint64_t lim = 1ull << 31;
    return qa_lds_bytes(a.D) <= (size_t)max_lds && qb_lds_bytes(a.I) <= (size_t)max_lds &&
           (uint64_t)a.I * (a.D / 256) * Q4B < lim && (uint64_t)a.D * (a.I / 256) * Q6B < lim &&
           (uint64_t)a.P * a.I < lim && (uint64_t)a.k * a.D < lim && (uint64_t)a.P * (a.I / 256) * 64 < lim;
}

bool qa_ring_shape(int gate_fmt, int D, int I) { return gate_fmt == TG_FMT_Q4K && D == 256 * RG_NB && I % 16 == 0 && I <= 4096; }

/* Items in the order expert (busiest first), pass, slab, cut into at most G
 * contiguous stretches of about equal cost (RingCost; workgroups past the
 * last stretch get none): each workgroup's stretch is a few runs of one
 * (expert, pass), and the passes of an expert run at about the same time on
 * neighbouring workgroups, so their slabs' second reads come from the caches.
 * rend[i] is the end of item i's run (the items of its expert and pass): a
 * workgroup finds where its run ends with one load, not by scanning the items
 * that follow.  runs holds each run's record (first pair, the pairs from
 * there on, the input rows of its first RING_P pairs, the expert) in list
 * order and run0[w] the run of workgroup w's first item, so a compute wave
 * reaches a run's operands with one round trip of scalar loads. */
void ring_items(const ExpDesc *ed, int n_act, int slabs, int G, const int *p_row, int P, int pass_pairs,
                const RingCost &c, RingLists &r) {
    r.items.clear();
    r.rend.clear();
    r.runs.clear();
    for (int ei = 0; ei < n_act; ei++)
        for (int t = 0; t < std::max(1, (ed[ei].np + pass_pairs - 1) / pass_pairs); t++) {
            const int run = (int)(r.runs.size() / RING_REC), pf = ed[ei].p0 + pass_pairs * t;
            r.runs.push_back(pf);
            r.runs.push_back(ed[ei].np - pass_pairs * t);
            for (int j = 0; j < RING_P; j++) r.runs.push_back(p_row[std::min(pf + j, P - 1)]);
            r.runs.push_back(ed[ei].e);
            r.runs.resize((size_t)(run + 1) * RING_REC, 0);
            for (int s = 0; s < slabs; s++) r.items.push_back(ei << 16 | s << 8 | t);
            r.rend.resize(r.items.size(), (int)r.items.size());
        }
    /* The cut: the smallest time T (found to 1 %) in which G workgroups get
     * through the list in order, each taking items while they fit.  A run
     * costs its start (its operands) in every workgroup that touches it. */
    const int runs = (int)(r.runs.size() / RING_REC);
    auto two = [&](int run) { return r.runs[(size_t)RING_REC * run + 1] > 16; };
    auto cut = [&](int64_t T, bool write) {
        int w = -1;
        int64_t room = 0;
        for (int run = 0; run < runs; run++) {
            const int64_t start = two(run) ? c.start2 : c.start1, each = two(run) ? c.item2 : c.item1;
            for (int left = slabs; left > 0;) {
                if (room < start + each) {
                    if (++w == G) return false;
                    room = T;
                    if (write) {
                        r.off[w] = run * slabs + slabs - left;
                        r.run0[w] = run;
                    }
                }
                const int take = (int)std::min<int64_t>(left, (room - start) / each);
                room -= start + take * each;
                left -= take;
            }
        }
        return true;
    };
    int64_t lo = std::max(c.start1 + c.item1, c.start2 + c.item2), all = 0;
    for (int run = 0; run < runs; run++) all += two(run) ? c.start2 + slabs * c.item2 : c.start1 + slabs * c.item1;
    lo = std::max(lo, all / G);   /* cut(lo - 1) fails */
    int64_t hi = lo;
    while (!cut(hi, false)) {
        lo = hi;
        hi += hi / 4;
    }
    while (hi - lo > hi / 100 + 1) {
        const int64_t mid = (lo + hi) / 2;
        (cut(mid, false) ? hi : lo) = mid;
    }
    r.off.assign(G + 1, (int)r.items.size());
    r.run0.assign(G + 1, 0);
    cut(hi, true);
}

void launch_moe_a_qk(const MoeArgs &a, hipStream_t st) {
    if (a.rg_items && qa_ring_shape(a.gate_fmt, a.D, a.I)) {
        hipLaunchKernelGGL(k_moe_qa_ring, dim3(a.rg_n), dim3(RG_NT), 0, st, a);
        return;
    }
    const dim3 grid((a.I + 15) / 16, a.n_act_a);
    if (a.D <= 256 * NW * 2) hipLaunchKernelGGL(k_moe_qa<2>, grid, dim3(NT), qa_lds_bytes(a.D), st, a);
    else hipLaunchKernelGGL(k_moe_qa<QA_WB_MAX>, grid, dim3(NT), qa_lds_bytes(a.D), st, a);
}

void launch_moe_b_qk(const MoeArgs &a, hipStream_t st) {
    if (a.rb_items && !a.dbias && qb_ring_shape(a.I, a.D)) {
        hipLaunchKernelGGL(k_moe_qb_ring, dim3(a.rb_n), dim3(DR_NT), 0, st, a);
        return;
    }
    hipLaunchKernelGGL(k_moe_qb<0>, dim3((a.D + QB_ROWS - 1) / QB_ROWS, a.n_act_a), dim3(NT), qb_lds_bytes(a.I), st,
                       a);
}

}  // namespace tg
