/*
 * tg_grouped.hip -- MXFP4 expert phases on block-scaled MFMA with the weights
 * staged in LDS: moe_phase_a / moe_phase_b of csrc/libtinygiant.c:1279-1384
 * with the per-block dot of dot_mxfp4_q8 (:533-547), for any number of pairs
 * per expert (a verify batch, a prefill).
 *
 * Arithmetic.  An MXFP4 block holds 32 e2m1 codes under one e8m0 exponent e.
 * The reference's term for a block is  d_x * half(e) * sum_i kv[c_i] * x_i
 * with kv[c] = 2 * e2m1(c), half(e) = 2^(e-128) and x_i the q8 integers.
 * v_mfma_scale_f32_16x16x128_f8f6f4 multiplies e2m1 A operands under e8m0
 * scales 2^(e-127) by fp8 B operands, so with A = the raw codes and scale e
 * each product is exactly kv[c] * half(e) * b.  A q8 integer x in [-127, 127]
 * is 16 * hi + lo with hi = x >> 4 in [-8, 7] and lo = x & 15, both exact in
 * fp8 e4m3; the hi half runs with B scale 2^4.  The block sums are exact;
 * only the f32 additions of four blocks inside the MFMA and of the q8 scale
 * groups differ in order from the reference's block-by-block sum.
 *
 * Operand layout (measured on gfx950): A lane l = weight row l % 16 and
 * K = 32 (l / 16) + j for nibble j of its four dwords (low nibble first), so
 * the 16 code bytes of a block are the lane's A operand as they lie in memory
 * (K = 2t: value t, K = 2t + 1: value 16 + t); the lane's A scale is the
 * e8m0 of (row l % 16, K block l / 16).  B lane l = pair l % 16, bytes 0..15
 * at K = 16 (l / 16) + j, bytes 16..31 at K = 64 + 16 (l / 16) + j - 16.
 * D lane l, register v = weight row 4 (l / 16) + v, pair l % 16.
 *
 * Work item = 16 weight rows of one expert (a "slab": 16 consecutive rows are
 * one contiguous, 16-byte aligned byte range).  Persistent workgroups walk
 * cost-balanced runs of items; each holds the next item's slabs in registers
 * (coalesced 16-byte loads, in flight while the current item computes) and
 * stores them to LDS; its NWAVE waves split the blocks of a row into ranges
 * and run the expert's pairs against the resident slab, 16 per pass; 256
 * threads then add the waves' partial sums in wave order and write one
 * result each.
 * HBM sees each weight byte once however many pairs the expert holds; the
 * fp8 halves of a pass stay in registers from one item to the next of the
 * same expert.  Rows of up to 90 blocks take k_moe_mx_ring (slabs copied into
 * an LDS ring), longer ones and layers whose experts' down formats differ
 * k_moe_mx (slabs through registers).
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "tg_device.hpp"
#include "tg_kernels.h"
#include "tg_xchg.hpp"

namespace tg {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int MXB = 17;                 /* bytes per MXFP4 block */
constexpr int GB = 4;                   /* blocks per MFMA (K = 128) */
constexpr int NWAVE = 8;                /* waves per workgroup, each one range of blocks */
constexpr int NT = 64 * NWAVE;
constexpr int CHUNKS = 4;               /* 16-byte slab chunks per thread and matrix */
constexpr uint32_t MAX_SLAB = CHUNKS * NT * 16;
constexpr int XB = 12;                  /* blocks of q8 operands per batch */
constexpr int NG = XB / GB;
constexpr uint32_t OOB = 0x80000000u;   /* past every buffer: the load reads zero */
constexpr int FMT_FP8 = 0, FMT_FP4 = 4; /* MFMA operand formats */
constexpr int NPRE = 4;                 /* passes whose pair rows and weights are fetched with the expert */
constexpr int SCALE_1 = 127, SCALE_16 = 131;

/* Slab bytes are read once per call: nontemporal loads (measured 3-6%
 * faster on a 64-token gpt-oss prefill than regular ones; the Q4_K / Q6_K
 * phases, whose lanes share 16-byte pieces of a line, lose with them). */
constexpr int CPOL_NT = 2;
__device__ inline u32x4 ld16_nt(Buf b, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b128(b.r, (int)off, 0, CPOL_NT);
}

/* Read-only tables through explicit address spaces: wave-uniform reads of
 * the constant space become scalar loads (counted apart from the vector
 * loads), per-lane reads of the global space in-order vector loads. */
template <class T>
__device__ inline T ldc(const T *p, size_t i) {
    return ((const __attribute__((address_space(4))) T *)(uintptr_t)p)[i];
}
template <class T>
__device__ inline T ldg(const T *p, size_t i) {
    return ((const __attribute__((address_space(1))) T *)(uintptr_t)p)[i];
}

}  // namespace

/* q8_split_store of rows that were quantized elsewhere.  One wave per 256
 * values. */
__global__ __launch_bounds__(256) void k_mx_split(Q8Rows q, int nrows, int nblk, uint8_t *dst) {
    const int wave = (int)((blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 6), lane = threadIdx.x & 63;
    if (wave >= nrows * q.nb) return;   /* uniform per wave */
    const uint32_t packed = reinterpret_cast<const uint32_t *>(q.qs + (size_t)wave * 256)[lane];
    q8_split_store(packed, lane, dst, nblk, wave / q.nb, wave % q.nb);
}

/* The e8m0 scale byte 255 means 2^127 to the reference (e8m0_to_fp32_half,
 * csrc/libtinygiant.c:516-519) and NaN to the block-scaled MFMA (OCP MX), and
 * 2^127 times the products overflows the MFMA's f32 sums where the
 * reference's integer block sum times its scales may stay finite: a layer
 * with such a block takes the v_dot4 phases.  One thread per block. */
__global__ __launch_bounds__(256) void k_mx_scan_e255(const uint8_t *__restrict__ p, uint64_t nblocks,
                                                      unsigned *flag) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    const bool hit = i < nblocks && p[i * MXB] == 255;
    if (__ballot(hit) && (threadIdx.x & 63) == __builtin_ctzll(__ballot(hit))) atomicOr(flag, 1u);
}

void launch_mx_scan_e255(const uint8_t *p, uint64_t nbytes, unsigned *flag_dev, hipStream_t st) {
    const uint64_t nb = nbytes / MXB;
    if (nb == 0) return;
    hipLaunchKernelGGL(k_mx_scan_e255, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, st, p, nb, flag_dev);
}

void launch_mx_split(const Q8Rows &q, int nrows, int ncols, uint8_t *dst, hipStream_t st) {
    const int waves = nrows * q.nb;
    if (waves <= 0) return;
    hipLaunchKernelGGL(k_mx_split, dim3((waves + 3) / 4), dim3(256), 0, st, q, nrows, ncols / 32, dst);
}

namespace {

/* fp8 halves of one batch of XB blocks of a wave's range (NG groups of GB
 * blocks), MT tiles of pairs, plus the q8 scale of each group */
template <int MT>
struct XBatch {
    v8i hi[MT][NG], lo[MT][NG];
    float d[MT][NG];
};

struct XSrc {
    Buf sp;           /* fp8 halves, [rows][nblk][2][32] */
    Buf d;            /* q8 scales */
    int nblk, nb8;
};

template <int MT>
__device__ inline void load_batch(XBatch<MT> &s, const XSrc &o, int b0, int b1, int nt, const int *xrow, int g) {
#pragma unroll
    for (int t = 0; t < MT; t++) {
        if (t > 0 && t >= nt) break;
        const bool ok = xrow[t] >= 0;
        const uint32_t row = (uint32_t)(ok ? xrow[t] : 0);
        const uint32_t rbase = row * (uint32_t)o.nblk * 64u + 16u * (g & 1);
#pragma unroll
        for (int q = 0; q < NG; q++) {
            const int ba = b0 + GB * q + (g >> 1), bb = ba + 2;   /* blocks of bytes 0..15 and 16..31 */
            const uint32_t oa = ok && ba < b1 ? rbase + (uint32_t)ba * 64u : OOB;
            const uint32_t ob = ok && bb < b1 ? rbase + (uint32_t)bb * 64u : OOB;
            const uint32_t oa2 = oa == OOB ? OOB : oa + 32u, ob2 = ob == OOB ? OOB : ob + 32u;
            const int bq = b0 + GB * q;
            const uint32_t od = ok && bq < b1 ? (row * o.nb8 + (uint32_t)(bq >> 3)) * 4u : OOB;
            const u32x4 h0 = ld16(o.sp, oa), h1 = ld16(o.sp, ob), l0 = ld16(o.sp, oa2), l1 = ld16(o.sp, ob2);
            const uint32_t dv = ld4(o.d, od);
            s.hi[t][q] = v8i{(int)h0.x, (int)h0.y, (int)h0.z, (int)h0.w, (int)h1.x, (int)h1.y, (int)h1.z, (int)h1.w};
            s.lo[t][q] = v8i{(int)l0.x, (int)l0.y, (int)l0.z, (int)l0.w, (int)l1.x, (int)l1.y, (int)l1.z, (int)l1.w};
            s.d[t][q] = __uint_as_float(dv);
        }
    }
}

/* One batch of NG groups starting at block b0: every LDS read of the batch
 * first (the lane's block codes and e byte of each group and matrix), then
 * per group and matrix two chained MFMAs per tile.  A block past b1 reads
 * the last block's codes against B operands and a q8 scale of zero. */
template <int NM, int MT>
__device__ inline void mma_batch(const uint32_t *lds, uint32_t sstride, uint32_t rb, const XBatch<MT> &s, int b0,
                                 int b1, int nt, int lane, float (&acc)[NM][MT][4]) {
    const int g = lane >> 4, c16 = lane & 15;
    uint32_t w[NG][NM][5], sft[NG][NM];
#pragma unroll
    for (int q = 0; q < NG; q++) {
        const int b = min(b0 + GB * q + g, b1 - 1);
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const uint32_t pos = m * sstride + (uint32_t)c16 * rb + (uint32_t)b * MXB;   /* the block's e byte */
            const uint32_t *dw = lds + (pos >> 2);
#pragma unroll
            for (int i = 0; i < 5; i++) w[q][m][i] = dw[i];
            sft[q][m] = pos & 3u;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NG; q++)
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const uint32_t s8 = 8u * (sft[q][m] + 1u);   /* codes start one byte after e: 8 .. 32 bits */
            const uint32_t *ww = w[q][m];
            v8i av;
            av[0] = (int)(uint32_t)((((uint64_t)ww[1] << 32) | ww[0]) >> s8);
            av[1] = (int)(uint32_t)((((uint64_t)ww[2] << 32) | ww[1]) >> s8);
            av[2] = (int)(uint32_t)((((uint64_t)ww[3] << 32) | ww[2]) >> s8);
            av[3] = (int)(uint32_t)((((uint64_t)ww[4] << 32) | ww[3]) >> s8);
            av[4] = av[5] = av[6] = av[7] = 0;
            const int e = (int)((ww[0] >> (8u * sft[q][m])) & 0xFFu);
#pragma unroll
            for (int t = 0; t < MT; t++) {
                if (t > 0 && t >= nt) break;   /* uniform; tile 0 always holds a pair */
                const v4f z = {0.f, 0.f, 0.f, 0.f};
                v4f r = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, s.hi[t][q], z, FMT_FP4, FMT_FP8, 0, e,
                                                                        0, SCALE_16);
                r = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, s.lo[t][q], r, FMT_FP4, FMT_FP8, 0, e, 0,
                                                                    SCALE_1);
                const float d = s.d[t][q];
                acc[m][t][0] += d * r[0];
                acc[m][t][1] += d * r[1];
                acc[m][t][2] += d * r[2];
                acc[m][t][3] += d * r[3];
            }
        }
}

/* 16-byte staging chunks per thread and matrix for rows of rb bytes */
__host__ __device__ inline int mx_chunks(uint32_t rb) { return 16u * rb <= 3u * NT * 16 ? 3 : CHUNKS; }

/* LDS bytes of one matrix's slab: 16 rows, 16 bytes of slack for the last
 * lane's five-dword read, and room for every staging chunk (the stores are
 * unconditional; chunks past the slab hold zeros) */
__host__ __device__ inline uint32_t mx_slab_stride(uint32_t rb) {
    const uint32_t need = 16u * rb + 16u, chunks = (uint32_t)mx_chunks(rb) * NT * 16;
    return ((need > chunks ? need : chunks) + 15u) & ~15u;
}

size_t mx_lds_bytes(int nm, int mt, int cols) {
    const int nblk = cols / 32;
    return (size_t)nm * mx_slab_stride((uint32_t)nblk * MXB)   /* slabs */
           + (size_t)NWAVE * nm * mt * 4 * 64 * 4;             /* partial sums of every wave */
}

}  // namespace

/* DOWN = false, phase A (gate/up, NM = 2):
 *   hidden[p][r] = act(gate_r . xq_p + bg[r], up_r . xq_p + bu[r])
 * DOWN = true, phase B (NM = 1), experts whose down matrix is MXFP4:
 *   part[p][r] = w_p * (down_r . hq_p + bd[r])
 * Persistent: workgroup i takes a contiguous run of items of about equal
 * cost (slab load plus passes of 16 pairs); an item is (active expert,
 * 16-row slab).  NT threads; dynamic LDS = mx_lds_bytes; CH 16-byte chunks
 * per thread and matrix hold a slab (16 * CH * NT bytes at most). */
template <int NM, int MT, int CH, bool DOWN>
__global__ __launch_bounds__(NT) void k_moe_mx(MoeArgs a) {
    static_assert(MT == 1, "the epilogue maps one tile of 16 pairs onto 256 threads");
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const int rows = DOWN ? a.D : a.I, cols = DOWN ? a.I : a.D;
    const int nblk = cols / 32;
    const uint32_t rb = (uint32_t)nblk * MXB;
    const uint32_t slab = 16u * rb, sstride = mx_slab_stride(rb);
    const int nslab = (rows + 15) / 16;
    const int *act = DOWN ? a.mx_act + a.n_act_a : a.mx_act;
    const int nact = DOWN ? a.n_act_b : a.n_act_a;
    const int nitems = nact * nslab;
    float *red = (float *)((uint8_t *)lds + NM * sstride);   /* [NWAVE][NM][4][64] */
    /* w is wave-uniform (readfirstlane), so every condition below that
     * decides which loads a wave issues is a scalar branch */
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4,
              c16 = lane & 15;
    const uint32_t mbytes = (uint32_t)rows * rb;              /* rows past the end read zero */
    /* epilogue thread (tid < 256): register ev of D lane el, i.e. weight row
     * 4 (el / 16) + ev of the slab and pair el % 16 of the tile */
    const int ev = tid >> 6, el = tid & 63;

    /* this wave's block range, a multiple of GB blocks long */
    const int cw = (((nblk + NWAVE - 1) / NWAVE) + GB - 1) / GB * GB;
    const int b0w = min(nblk, w * cw), b1w = min(nblk, b0w + cw);
    XSrc xs;
    const Q8Rows &q = DOWN ? a.hq : a.xq;
    const int qrows = DOWN ? a.P : a.k;
    xs.nblk = nblk;
    xs.nb8 = q.nb;
    xs.sp = make_buf(DOWN ? a.hp : a.xp, (uint32_t)((size_t)qrows * nblk * 64));
    xs.d = make_buf(q.d, (uint32_t)((size_t)qrows * q.nb * 4));

    /* the expert of the item being issued, and its matrices */
    int iss_ai = -1;
    Buf iss_w[NM];
    u32x4 vA[NM][CH], vB[NM][CH];   /* slabs of two items ahead, alternating */
    auto set_issuer = [&](int ai) {
        iss_ai = ai;
        const int e = ldc(act, ai);
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const uint64_t base = DOWN ? ldc(a.down, e) : (m ? ldc(a.up, e) : ldc(a.gate, e));
            iss_w[m] = make_buf((const void *)(uintptr_t)base, mbytes);
        }
    };
    XBatch<MT> xb;
    int xrow[MT];
    /* this workgroup's run of items: an equal share of the total cost */
    const int *cum = DOWN ? a.mx_cum + a.n_act_a + 1 : a.mx_cum;
    auto item_at = [&](long c) {
        int lo = 0, hi = nact;   /* largest i with cum[i] <= c */
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (ldc(cum, mid) <= c) lo = mid;
            else hi = mid;
        }
        const int per = (ldc(cum, lo + 1) - ldc(cum, lo)) / nslab;
        return min(nitems, lo * nslab + (int)((c - ldc(cum, lo) + per - 1) / per));
    };
    const long total = nact ? ldc(cum, nact) : 0;
    int it = nact ? item_at(total * blockIdx.x / gridDim.x) : 0;
    const int it_end = blockIdx.x + 1 == gridDim.x ? nitems : (nact ? item_at(total * (blockIdx.x + 1) / gridDim.x) : 0);
    if (it >= it_end) return;   /* uniform */

    /* an item's slabs; an item past the run reads zeros (no memory access),
     * so every item issues the same loads */
    auto issue = [&](u32x4 (&v)[NM][CH], int item) {
        const bool ok = item < it_end;
        if (ok && item / nslab != iss_ai) set_issuer(item / nslab);
        const uint32_t off = (uint32_t)(item % nslab) * 16u * rb;
#pragma unroll
        for (int m = 0; m < NM; m++) {
#pragma unroll
            for (int c = 0; c < CH; c++) {
                const uint32_t i = (uint32_t)(tid + NT * c) * 16u;
                v[m][c] = ld16_nt(iss_w[m], ok && i < slab ? off + i : OOB);
            }
        }
    };

    /* per-expert state: the expert's pairs, biases (empty buffers read
     * zero) and the input rows of its first 16 pairs */
    struct Expert {
        int ai, p0, ne;
        bool has0, has1;
        Buf bias[2];
    };
    const Buf prow_buf = make_buf(a.p_row, (uint32_t)a.P * 4u), pw_buf = make_buf(a.p_w, (uint32_t)a.P * 4u);
    auto expert = [&](int ai) {
        Expert x;
        x.ai = ai;
        const int e = ldc(act, ai);
        x.p0 = ldc(a.p_off, e);
        x.ne = ldc(a.p_off, e + 1) - x.p0;
        const float *b0p = DOWN ? (a.dbias ? (const float *)(uintptr_t)ldc(a.dbias, e) : nullptr)
                                : (a.gbias ? (const float *)(uintptr_t)ldc(a.gbias, e) : nullptr);
        const float *b1p = DOWN ? nullptr : (a.ubias ? (const float *)(uintptr_t)ldc(a.ubias, e) : nullptr);
        x.has0 = b0p != nullptr;
        x.has1 = b1p != nullptr;
        x.bias[0] = make_buf(b0p, b0p ? (uint32_t)rows * 4u : 0u);
        x.bias[1] = make_buf(b1p, b1p ? (uint32_t)rows * 4u : 0u);
        return x;
    };
    /* input row of pair j of an expert (phase A: its q8 row, phase B: the
     * pair itself), unmasked (zero past the expert's pairs) and with -1
     * there; the pair's router weight */
    auto pair_row_raw = [&](const Expert &x, int j) -> int {
        if (DOWN) return x.p0 + j;
        return (int)ld4(prow_buf, j < x.ne ? (uint32_t)(x.p0 + j) * 4u : OOB);
    };
    auto pair_row = [&](const Expert &x, int j) -> int {
        const int r = pair_row_raw(x, j);
        return j < x.ne ? r : -1;
    };
    auto pair_w = [&](const Expert &x, int j) -> float {
        return __uint_as_float(ld4(pw_buf, j < x.ne ? (uint32_t)(x.p0 + j) * 4u : OOB));
    };
    /* epilogue thread (tid < 256) row of an item's slab */
    auto ep_row = [&](int item) { return (item % nslab) * 16 + 4 * (el >> 4) + ev; };

    /* pair rows (unmasked: the mask is applied where a pass takes them, so
     * the load is not waited for at once) and (phase B) weights of an
     * expert's first NPRE passes */
    int xrows[NPRE], nxrows[NPRE];
    float wts[NPRE], nwts[NPRE];
    auto fetch_pairs = [&](const Expert &x, int (&rr)[NPRE], float (&ww)[NPRE]) {
#pragma unroll
        for (int k = 0; k < NPRE; k++) {
            rr[k] = pair_row_raw(x, 16 * k + c16);
            ww[k] = DOWN ? pair_w(x, 16 * k + (el & 15)) : 0.f;
        }
    };

    /* first item: its slabs, q8 operands, biases and pair weights, then the
     * second item's slabs */
    Expert cur = expert(it / nslab), nxt = cur;
    fetch_pairs(cur, xrows, wts);
    wait_copies();   /* a wait the compiler sees: the pair loads are not pending in the item loop */
    xrow[0] = c16 < cur.ne ? xrows[0] : -1;
    issue(vA, it);
    load_batch<MT>(xb, xs, b0w, min(b1w, b0w + XB), 1, xrow, g);
    int er = ep_row(it);
    float bias0 = __uint_as_float(ld4(cur.bias[0], (uint32_t)er * 4u));
    float bias1 = __uint_as_float(ld4(cur.bias[1], (uint32_t)er * 4u));
    float wt = wts[0];
    __builtin_amdgcn_sched_barrier(0);
    issue(vB, it + 1);

    /* Per item, loads are issued in one fixed order: the next expert's pair
     * rows (when it changes), then after the compute the next item's q8
     * operands (unless kept) and biases, then the slabs two items ahead (past
     * the run they read zeros).  Loads complete in order, so the compiler's
     * wait for an item's slab leaves the next item's slab in flight, and
     * every slab has a whole item of lead. */
    float acc[NM][MT][4];
    /* one pass: the partial sums of every wave to LDS, then 256 threads add
     * them in wave order and write one result each */
    auto finish = [&](int t0) {
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int vv = 0; vv < 4; vv++) red[((w * NM + m) * 4 + vv) * 64 + lane] = acc[m][0][vv];
        bar_lds();
        const int j = t0 + (el & 15);
        if (tid < 256 && j < cur.ne && er < rows) {
            float r2[NM];
#pragma unroll
            for (int m = 0; m < NM; m++) {
                float sum = red[(m * 4 + ev) * 64 + el];
#pragma unroll
                for (int ww = 1; ww < NWAVE; ww++) sum += red[((ww * NM + m) * 4 + ev) * 64 + el];
                r2[m] = sum;
            }
            const int p = cur.p0 + j;
            if (DOWN) {
                a.part[(size_t)p * a.D + er] = wt * (r2[0] + (cur.has0 ? bias0 : 0.f));
            } else {
                float gv = r2[0], uv = r2[NM - 1];
                if (cur.has0) gv += bias0;
                if (cur.has1) uv += bias1;
                a.hidden[(size_t)p * a.I + er] = act_fn(a.act, gv, uv);
            }
        }
    };
    auto zero = [&]() {
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int vv = 0; vv < 4; vv++) acc[m][0][vv] = 0.f;
    };
    auto step = [&](u32x4 (&v)[NM][CH]) {
        const int nx = it + 1;
        const bool has_nx = nx < it_end;
        const bool new_ex = has_nx && nx / nslab != cur.ai;
        if (new_ex) {
            nxt = expert(nx / nslab);
            fetch_pairs(nxt, nxrows, nwts);
        }
        bar_lds();   /* the previous item is done with LDS */
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int c = 0; c < CH; c++)
                *(u32x4 *)((uint8_t *)lds + m * sstride + (uint32_t)(tid + NT * c) * 16u) = v[m][c];
        bar_lds();
        zero();
        mma_batch<NM, MT>(lds, sstride, rb, xb, b0w, min(b1w, b0w + XB), 1, lane, acc);
        for (int bb = b0w + XB; bb < b1w; bb += XB) {   /* rows wider than NWAVE * XB blocks */
            load_batch(xb, xs, bb, min(b1w, bb + XB), 1, xrow, g);
            mma_batch<NM, MT>(lds, sstride, rb, xb, bb, min(b1w, bb + XB), 1, lane, acc);
        }
        finish(0);
        /* further passes over the resident slab for an expert with more than
         * 16 pairs */
        for (int t0 = 16 * MT, k = 1; t0 < cur.ne; t0 += 16 * MT, k++) {
            bar_lds();   /* red is rewritten by this pass */
            int r = 0;
            float wk = 0.f;
#pragma unroll
            for (int q = 1; q < NPRE; q++)
                if (k == q) {
                    r = xrows[q];
                    wk = wts[q];
                }
            xrow[0] = k < NPRE ? (t0 + c16 < cur.ne ? r : -1) : pair_row(cur, t0 + c16);
            if (DOWN) wt = k < NPRE ? wk : pair_w(cur, t0 + (el & 15));
            zero();
            for (int bb = b0w; bb < b1w; bb += XB) {
                load_batch(xb, xs, bb, min(b1w, bb + XB), 1, xrow, g);
                mma_batch<NM, MT>(lds, sstride, rb, xb, bb, min(b1w, bb + XB), 1, lane, acc);
            }
            finish(t0);
            /* a wait the compiler sees: the pass's own loads (issued after
             * the next slabs, which they waited for already) are not left
             * pending where the compiler merges paths */
            wait_copies();
        }
        /* the next item's q8 operands (unless this item's first-pass ones
         * serve it: same expert, one pass, one batch), biases, pair weights */
        if (has_nx) {
            const bool keep = !new_ex && cur.ne <= 16 * MT && b1w - b0w <= XB;
            if (new_ex) {
                /* the new expert's pair loads (issued after the next slabs,
                 * so this waits for those too) */
                wait_copies();
                cur = nxt;
#pragma unroll
                for (int q = 0; q < NPRE; q++) {
                    xrows[q] = nxrows[q];
                    wts[q] = nwts[q];
                }
            }
            xrow[0] = c16 < cur.ne ? xrows[0] : -1;
            if (!keep) load_batch<MT>(xb, xs, b0w, min(b1w, b0w + XB), 1, xrow, g);
            er = ep_row(nx);
            bias0 = __uint_as_float(ld4(cur.bias[0], (uint32_t)er * 4u));
            bias1 = __uint_as_float(ld4(cur.bias[1], (uint32_t)er * 4u));
            wt = wts[0];
        }
        /* then the slabs two items ahead, into the registers just stored */
        __builtin_amdgcn_sched_barrier(0);
        issue(v, it + 2);
        it = nx;
    };
    while (it < it_end) {
        step(vA);
        if (it >= it_end) break;
        step(vB);
    }
}

/* Tiles of 16 pairs per pass.  One: an expert with more than 16 pairs runs
 * further passes over its resident slab. */
constexpr int MX_TILES = 1;

/* the device must allow the LDS to one workgroup, and the slab must fit the
 * staging registers */
bool grouped_lds_ok(int D, int I) {
    static int max_lds = -1;
    if (max_lds < 0) {
        int dev = 0;
        max_lds = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
            max_lds = 0;
    }
    return mx_lds_bytes(2, MX_TILES, D) <= (size_t)max_lds && mx_lds_bytes(1, MX_TILES, I) <= (size_t)max_lds &&
           (uint32_t)(D / 32) * MXB * 16 <= MAX_SLAB && (uint32_t)(I / 32) * MXB * 16 <= MAX_SLAB;
}

/* persistent grid: the workgroups that can be resident at once */
template <class K>
static unsigned mx_grid(K kern, size_t lds, int nitems) {
    int dev = 0, cus = 0, per = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, NT, lds) != hipSuccess || per < 1) per = 1;
    return (unsigned)std::max(1, std::min(std::max(cus, 1) * per, nitems));
}

template <int NM, bool DOWN>
static void launch_mx(const MoeArgs &a, int cols, int nitems, hipStream_t st) {
    if (nitems == 0) return;
    const size_t lds = mx_lds_bytes(NM, MX_TILES, cols);
    if (mx_chunks((uint32_t)(cols / 32) * MXB) == 3) {
        auto k = k_moe_mx<NM, MX_TILES, 3, DOWN>;
        hipLaunchKernelGGL(k, dim3(mx_grid(k, lds, nitems)), dim3(NT), lds, st, a);
    } else {
        auto k = k_moe_mx<NM, MX_TILES, CHUNKS, DOWN>;
        hipLaunchKernelGGL(k, dim3(mx_grid(k, lds, nitems)), dim3(NT), lds, st, a);
    }
}

namespace {

/* ---- persistent phases over rows of up to 90 blocks ----
 *
 * One workgroup a compute unit walks its list of items (ring_items: active
 * expert, pass of up to 16 pairs, item rows), the slabs streaming through a
 * ring of three LDS slots two items ahead of the item computed.  An item is
 * 48 KiB, two halves of 16 rows: the gate and the up rows (phase A), or 32
 * down rows (phase B).  Eight compute waves: wave c takes half c / 4 and a
 * quarter of its rows' blocks, with the fp8 halves of the run's pairs for
 * those blocks in registers (six groups of four blocks, 96 registers, loaded
 * once a run); they also finish the previous item, one barrier an item.  Two
 * copy waves issue the direct-to-LDS copies, one half each, and nothing else,
 * so they wait for their own with exact counts.
 *
 * Against k_moe_mx above (slabs through registers, two barriers and the
 * reduction between an item and the next loads) the compute unit always has
 * one to two whole items in flight, phase B moves 48 KiB a step instead of
 * 24, and a further pass of an expert re-reads its slab from the caches
 * instead of waiting for that pass's operands on every item.  gpt-oss layer
 * (top-4 of 128), whole call, 5 / 9 / 16 / 64 / 256 rows: 77.7 / 93.0 / 131 /
 * 282 / 636 us there, 74.4 / 71.9 / 103 / 184 / 376 here.
 *
 * Bound: a compute unit's share of HBM (an item's 48 KiB: 2 us); 71 experts'
 * 939 MB move at 5.6 TB/s in the two phases' ~167 us of the 64-row call. */
constexpr int MR_SLAB = 24 * 1024;               /* LDS bytes of a half: 16 rows of up to 90 blocks */
constexpr int MR_BLOCKS = MR_SLAB / (16 * MXB);  /* 90 */
constexpr int MR_LC = MR_SLAB / 1024;            /* copies of 1 KiB a half */
constexpr int MR_SLOTS = 3;
constexpr int MR_CW = 8, MR_YW = 2;              /* compute and copy waves */
constexpr int MR_NT = 64 * (MR_CW + MR_YW);
constexpr int MR_G = 6;                          /* groups of GB blocks a compute wave holds */
constexpr int MR_B = 2;                          /* groups whose codes are read together */
static_assert((MR_SLOTS - 2) * MR_LC <= 63, "a vmcnt count");
static_assert(4 * MR_G * GB >= MR_BLOCKS, "four waves cover a row");
static_assert(16 * MXB * MR_BLOCKS + (GB - 1) * MXB + 4 <= MR_SLAB, "the last group's reads stay in the half");

/* a compute lane's operands of one run: pair c16's fp8 halves of its wave's groups */
struct MrX {
    v8i hi[MR_G], lo[MR_G];
    float d[MR_G];   /* q8 scale of each group */
};

template <bool DOWN>
__global__ __launch_bounds__(MR_NT) void k_moe_mx_ring(MoeArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t ring[MR_SLOTS][2][MR_SLAB];
    __shared__ __attribute__((aligned(16))) v4f red[2][MR_CW][64];   /* by item parity */
    constexpr int IR = DOWN ? MX_RING_DOWN : MX_RING_UP;
    const int rows = DOWN ? a.D : a.I, nblk = (DOWN ? a.I : a.D) / 32;
    const uint32_t rb = (uint32_t)nblk * MXB, mbytes = (uint32_t)rows * rb;
    const int *items = DOWN ? a.rb_items : a.rg_items, *offs = DOWN ? a.rb_off : a.rg_off;
    const int *rend = DOWN ? a.rb_rend : a.rg_rend, *runs = DOWN ? a.rb_runs : a.rg_runs;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4,
              c16 = lane & 15;
    const int wg = ring_wg();
    const int i0 = ldc(offs, wg), n = ldc(offs, wg + 1) - i0;
    if (n <= 0) return;   /* uniform */
    /* item j of the list (j < n): expert index, item rows, pass */
    auto item = [&](int j) { return ldc(items, (size_t)(i0 + j)); };

    /* The two roles run loops of their own, meeting at one barrier an item.
     * Between the barriers of items i and i + 1 the compute waves finish item
     * i - 1 (reading red[(i - 1) % 2]) and compute item i (reading slot
     * i % MR_SLOTS, writing red[i % 2]) while the copy waves copy item i + 2
     * into item i - 1's slot. */
    if (w >= MR_CW) {
        const int m = w - MR_CW;
        struct Info {   /* an item's matrix and first byte; its scalar loads go out an item ahead */
            uint64_t base;
            int s;
        };
        auto info = [&](int it) __attribute__((always_inline)) {
            const ExpDesc *e = &a.ed[it >> 16];
            Info f;
            f.base = DOWN ? ldc(&e->down, 0) : m ? ldc(&e->up, 0) : ldc(&e->gate, 0);
            f.s = (it >> 8) & 255;
            return f;
        };
        const uint32_t slab = 16u * rb;
        auto copies = [&](int j, const Info &f) __attribute__((always_inline)) {
            const u32x4 desc = buf_desc((const void *)(uintptr_t)f.base, mbytes);
            const uint32_t first = (uint32_t)(DOWN ? 2 * f.s + m : f.s) * slab;
            uint8_t *dst = &ring[j % MR_SLOTS][m][0];
#pragma unroll
            for (int k = 0; k < MR_LC; k++) {
                const uint32_t i = 1024u * k + 16u * (uint32_t)lane;
                copy_lanes_nt(desc, i < slab ? first + i : OOB, lds_addr(dst + 1024 * k));
            }
        };
        for (int j = 0; j < MR_SLOTS - 1 && j < n; j++) copies(j, info(item(j)));
        Info fc = info(item(min(MR_SLOTS - 1, n - 1)));   /* item i + MR_SLOTS - 1 */
        int code = item(min(MR_SLOTS, n - 1));             /* item i + MR_SLOTS */
        for (int i = 0; i < n; i++) {
            /* item i's copies have landed, item i + 1's may be in flight */
            if (i + 1 < n) wait_copies_but<(MR_SLOTS - 2) * MR_LC>();
            else wait_copies_but<0>();
            asm volatile("s_barrier" ::: "memory");
            if (i + MR_SLOTS - 1 < n) copies(i + MR_SLOTS - 1, fc);
            fc = info(code);
            code = item(min(i + MR_SLOTS + 1, n - 1));
        }
        asm volatile("s_barrier" ::: "memory");
        wait_copies();   /* no copy outlives the workgroup */
        return;
    }

    /* the wave's half and its blocks [b0, b0 + GB ng), whole groups of a row */
    const int m = w >> 2, cw = ((nblk + 3) / 4 + GB - 1) / GB * GB, b0 = cw * (w & 3);
    const int ng = max(0, min(cw, nblk - b0) + GB - 1) / GB;
    const Q8Rows &q = DOWN ? a.hq : a.xq;
    const int qrows = DOWN ? a.P : a.k;
    const Buf sp = make_buf(DOWN ? a.hp : a.xp, (uint32_t)((size_t)qrows * nblk * 64));
    const Buf qd = make_buf(q.d, (uint32_t)((size_t)qrows * q.nb * 4));
    const Buf pw = make_buf(a.p_w, (uint32_t)a.P * 4u);
    auto load_x = [&](const int *rc, MrX &x) __attribute__((always_inline)) {
        const bool pv = c16 < ldc(rc, 1);
        uint32_t prow = 0u;
        if (DOWN) {
            prow = (uint32_t)(ldc(rc, 0) + c16);
        } else {
            uint32_t rj[16];
#pragma unroll
            for (int j = 0; j < 16; j++) rj[j] = (uint32_t)ldc(rc, 2 + j);
#pragma unroll
            for (int j = 0; j < 16; j++) prow = c16 == j ? rj[j] : prow;
        }
        const uint32_t base = prow * (uint32_t)nblk * 64u + 16u * (g & 1), dbase = prow * (uint32_t)q.nb;
#pragma unroll
        for (int k = 0; k < MR_G; k++) {
            const int bq = b0 + GB * k, ba = bq + (g >> 1), bb = ba + 2;   /* blocks of bytes 0..15 and 16..31 */
            const bool in = pv && k < ng;
            const uint32_t oa = in && ba < nblk ? base + (uint32_t)ba * 64u : OOB;
            const uint32_t ob = in && bb < nblk ? base + (uint32_t)bb * 64u : OOB;
            const u32x4 h0 = ld16(sp, oa), h1 = ld16(sp, ob);
            const u32x4 l0 = ld16(sp, oa + 32u), l1 = ld16(sp, ob + 32u);   /* OOB + 32 is past the buffer too */
            x.hi[k] = v8i{(int)h0.x, (int)h0.y, (int)h0.z, (int)h0.w, (int)h1.x, (int)h1.y, (int)h1.z, (int)h1.w};
            x.lo[k] = v8i{(int)l0.x, (int)l0.y, (int)l0.z, (int)l0.w, (int)l1.x, (int)l1.y, (int)l1.z, (int)l1.w};
            x.d[k] = __uint_as_float(ld4(qd, in ? (dbase + (uint32_t)(bq >> 3)) * 4u : OOB));
        }
        /* taken as the values of an empty asm statement: the compiler waits
         * for the loads there and not at their uses */
#pragma unroll
        for (int k = 0; k < MR_G; k++) asm volatile("" : "+v"(x.hi[k]), "+v"(x.lo[k]), "+v"(x.d[k]));
    };
    /* item j's slab against x: the wave's quarter of the rows' sums to red.
     * A group's blocks lie 17 dwords after the one's before, so a lane's codes
     * start at one byte of a dword in all of them. */
    const uint32_t e0 = (uint32_t)c16 * rb + (uint32_t)(b0 + g) * MXB;   /* the first group's e byte */
    const uint32_t sh = (e0 + 1u) & 3u;
    auto compute = [&](int j, const MrX &x) __attribute__((always_inline)) {
        const uint8_t *sb = &ring[j % MR_SLOTS][m][0];
        const uint32_t *dw = (const uint32_t *)(sb + ((e0 + 1u) & ~3u));
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < MR_G; k0 += MR_B) {
            uint32_t c[MR_B][5], e[MR_B];
#pragma unroll
            for (int i = 0; i < MR_B; i++) {
                if (k0 + i >= ng) break;   /* uniform */
#pragma unroll
                for (int t = 0; t < 5; t++) c[i][t] = dw[17 * (k0 + i) + t];
                e[i] = sb[e0 + 68u * (k0 + i)];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MR_B; i++) {
                const int k = k0 + i;
                if (k >= ng) break;   /* uniform */
                v8i av;
#pragma unroll
                for (int t = 0; t < 4; t++) av[t] = (int)__builtin_amdgcn_alignbyte(c[i][t + 1], c[i][t], sh);
                av[4] = av[5] = av[6] = av[7] = 0;
                /* past the row: the next row's block, or the slab's end, under a finite scale and zero operands */
                const int es = b0 + GB * k + g < nblk ? (int)e[i] : 0;
                const v4f z = {0.f, 0.f, 0.f, 0.f};
                v4f r = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, x.hi[k], z, FMT_FP4, FMT_FP8, 0, es, 0,
                                                                        SCALE_16);
                r = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, x.lo[k], r, FMT_FP4, FMT_FP8, 0, es, 0, SCALE_1);
#pragma unroll
                for (int v = 0; v < 4; v++) acc[v] += x.d[k] * r[v];
            }
        }
        red[j & 1][w][lane] = v4f{acc[0], acc[1], acc[2], acc[3]};
    };
    /* finishing item j, a lane one (pair, row) result: pair 4 (w % 4) + g and
     * row c16 (of half w / 4 in phase B; waves 0 to 3 in phase A), whose sums
     * sit in lane 16 (c16 / 4) + pair, register c16 % 4 */
    struct Done {   /* the item to finish: its first pair, pairs from there, first row of the wave's half, biases, pair weight */
        int pf, nv, r;
        float b0, b1, wt;
    };
    auto finish = [&](int j, const Done &f) __attribute__((always_inline)) {
        if (!DOWN && w >= 4) return;           /* uniform */
        if (4 * (w & 3) >= f.nv) return;       /* uniform */
        int ln = lane;
        asm volatile("" : "+v"(ln));   /* what follows of it is computed here, not kept in registers */
        const int jj = 4 * (w & 3) + (ln >> 4), c = ln & 15;
        const float *p = (const float *)&red[j & 1][DOWN ? 4 * m : 0][16 * (c >> 2) + jj] + (c & 3);
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int ww = 0; ww < 4; ww++) {
            s0 += p[256 * ww];
            if (!DOWN) s1 += p[256 * (4 + ww)];
        }
        const int r = f.r + c;
        if (jj >= f.nv || r >= rows) return;
        if (DOWN) a.part[(size_t)(f.pf + jj) * a.D + r] = f.wt * (s0 + f.b0);
        else a.hidden[(size_t)(f.pf + jj) * a.I + r] = act_fn(a.act, s0 + f.b0, s1 + f.b1);
    };

    MrX cur;
    Done done = {0, 0, 0, 0.f, 0.f, 0.f};
    int run = ldc(DOWN ? a.rb_run0 : a.rg_run0, wg);   /* the run of item 0; the runs follow in order */
    int s = (item(0) >> 8) & 255;
    const uint64_t *bp0 = DOWN ? a.dbias : a.gbias, *bp1 = DOWN ? nullptr : a.ubias;
    for (int i = 0; i < n; run++, s = 0) {
        const int *rc = runs + (size_t)RING_REC * run;
        load_x(rc, cur);
        const int re = min(ldc(rend, (size_t)(i0 + i)), i0 + n) - i0;   /* the run's end */
        const int pf = ldc(rc, 0), nv = ldc(rc, 1), e = ldc(rc, 2 + RING_P);
        const uint64_t q0 = bp0 ? ldc(bp0, e) : 0, q1 = bp1 ? ldc(bp1, e) : 0;
        const Buf bb0 = make_buf((const void *)(uintptr_t)q0, q0 ? (uint32_t)rows * 4u : 0u);   /* empty buffers read zero */
        const Buf bb1 = make_buf((const void *)(uintptr_t)q1, q1 ? (uint32_t)rows * 4u : 0u);
        const int jj = 4 * (w & 3) + g;
        const float wt = DOWN ? __uint_as_float(ld4(pw, jj < nv ? (uint32_t)(pf + jj) * 4u : OOB)) : 0.f;
        for (; i < re; i++, s++) {
            bar_lds();   /* item i's slab has landed, item i - 1's sums are in LDS */
            finish(i - 1, done);   /* nothing before the first item: no pairs */
            done.pf = pf;
            done.nv = nv;
            done.r = IR * s + (DOWN ? 16 * m : 0);
            if (bp0) done.b0 = __uint_as_float(ld4(bb0, (uint32_t)(done.r + c16) * 4u));
            if (bp1) done.b1 = __uint_as_float(ld4(bb1, (uint32_t)(done.r + c16) * 4u));
            done.wt = wt;
            compute(i, cur);
        }
    }
    bar_lds();   /* item n - 1's sums are in LDS */
    finish(n - 1, done);
}

/* the operands' offsets and OOB must not meet */
bool mx_ring_fits(const Q8Rows &q, int qrows, int nblk) {
    return (uint64_t)qrows * nblk * 64 < OOB && (uint64_t)qrows * q.nb * 4 < OOB;
}

}  // namespace

bool mx_ring_shape(int rows, int cols, int item_rows) {
    return cols / 32 <= MR_BLOCKS && (rows + item_rows - 1) / item_rows <= 256;   /* an item holds its rows in 8 bits */
}

void launch_moe_a_mx(const MoeArgs &a, hipStream_t st) {
    if (a.rg_items && a.rg_mx && mx_ring_fits(a.xq, a.k, a.D / 32)) {
        hipLaunchKernelGGL(k_moe_mx_ring<false>, dim3(a.rg_n), dim3(MR_NT), 0, st, a);
        return;
    }
    launch_mx<2, false>(a, a.D, a.n_act_a * ((a.I + 15) / 16), st);
}

void launch_moe_b_mx(const MoeArgs &a, hipStream_t st) {
    if (a.rb_items && a.rb_mx && mx_ring_fits(a.hq, a.P, a.I / 32)) {
        hipLaunchKernelGGL(k_moe_mx_ring<true>, dim3(a.rb_n), dim3(MR_NT), 0, st, a);
        return;
    }
    launch_mx<1, true>(a, a.I, a.n_act_b * ((a.D + 15) / 16), st);
}

}  // namespace tg
