// gemm_kq.hip — prompt-batch matmul of K-quant weights × Q8_K activations on CDNA4
// int8 MFMA: Q4_K and Q5_K (one kernel) and Q6_K.  Q4_K is described first:
// the batched counterpart of the Q4_K block dot (the x86 prefill tiles
// of kernels/mod.rs:238-296 cover Q4_K; kernels/avx2.rs dot_q4_k 78-107).
//
// Per 256-value superblock b, for activation row t and weight row r:
//   y += (f16(d_r)·d_t)·Σ_j sc_j·Σ_{32} q4·q8 − (f16(dmin_r)·d_t)·Σ_j m_j·(bsum_2j + bsum_2j+1)
// * the eight 32-value sub-block dots are v_mfma_i32_32x32x32_i8 (exact);
// * Σ_j sc_j·I_j is an exact int32 sum (|.| < 2^25);
// * Σ_j m_j·bs_j (< 2^21, exact in f32) and the scale products d·d_t, dmin·d_t are
//   v_mfma_f32_32x32x2_f32 rank-1 / rank-2 products;
// so the superblock's two integer sums equal the reference's exactly and only the
// f32 accumulation over superblocks differs in order.
//
// Workgroup tile: 64 weight rows × 64 tokens, 4 waves as 2 × 2 (32 rows × 32
// tokens each).  A stage is half a superblock (4 sub-blocks, 128 values): the
// activation codes, the weight nibbles and the half's 6-bit scales go to LDS, with
// the second half also what the superblock's end reads (activation scale and 32-value
// sums, d, dmin and mins); the next stage's global loads are in flight meanwhile.
// The scales and mins are unpacked four to a dword and the min term's operands made
// once per workgroup: one at a time, in every stage and wave, they were a third of the
// kernel's vector instructions (421 tokens, gate/up 2 × 8192 × 3072 in Q5_K: 128 us, now
// 91 us; Q6_K down of 3072 × 8192: 79 us, now 64 us).
// Operand lane layout as in gemm.hip: lane l supplies row l mod 32 and values
// 16·(l/32)..+16; tokens are permuted onto the A rows so that lane l's 16
// results are the 16 consecutive tokens 16·(l/32) + v.
//
// Q5_K weights (quant/reference.rs:321-350) differ in the code alone: the fifth bits
// come from the superblock's 32 qh bytes.  The stage store joins nibble and bit into
// one byte per code (two ALU operations per four codes, once per workgroup), so the
// multiply loop reads its B operand without the nibble shifts of Q4_K, for 64 more LDS
// bytes per row.  Bound like Q4_K by the int32 scale multiply-adds between the MFMAs.
// A 421-token prompt through two layers of hidden 3072 (Q5_K, V and one down
// projection Q6_K) takes 778 µs, against 7439 µs with its Q5_K weights in the batched
// GEMV, which reads and unpacks every weight once per 4 tokens.
//
// Q6_K weights × Q8_K activations (kernels/avx2.rs dot_q6_k 109-151): per
// superblock y += (f16(d_r)·d_t)·Σ_k sc_k·Σ_{16} (q6−32)·q8.  The codes are
// unpacked once per stage into int8 q6−32 in LDS (four at a time); each
// 16-value sub-block dot is one v_mfma_i32_32x32x16_i8 (exact), Σ_k sc_k·D_k
// accumulates in int32 with 24-bit multiply-adds (|.| < 2^27), and the
// superblock's float product is the rank-1 f32 MFMA of d_t and d_r.  The gated form
// stages gate and up rows beside each other (two weight tiles per activation tile).
#include "../common.hpp"
#include "../device.hpp"
#include "../kernels.hpp"
#include "../gemv_units.hpp"
#include "../gemm_split.hpp"

#include <type_traits>

namespace rie {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef _Float16 half8k __attribute__((ext_vector_type(8)));

struct KqP {
    const uint8_t *w[3];
    size_t rb[3];
    int rows[3];
    float *out[3];
    int ld[3];
    int epi[3];
    int nseg;
    int rg_end[3];  // cumulative 64-row groups at the end of each segment
    int n_rg, n_tg;
    int glu;        // 0 none; 1 silu / 2 gelu-tanh: seg 0 gate, seg 1 up, out[0] = h
    const int8_t *qs;
    const float *d;
    const int16_t *bsums;
    int n_tok, K;
    int grouped;     // expert groups: one matrix per expert (grp), token tiles from its table
    GroupTiles grp;
    int ks;  // K splits of a tile (64-token tiles, not grouped), in whole superblocks
    GemmWs ws;
    size_t plane;  // floats per plane of a split in planes (plane_count), 0: split_sum
};

constexpr int KQ_BM = 64, KQ_BN = 64;
static_assert(KQ_BN == GROUP_BN, "grouped tiles are built for this token tile");
// Q4_K tiles of BN = 32 tokens (groupings of Q4_K experts, a few dozen rows each)
// are 128 weight rows tall: the four waves stand along the rows
template <int BN> constexpr int kq_bm() { return BN == 64 ? 64 : 128; }

// A workgroup's token rows: tokens [r0, r_end) of the batch, or gathered rows
// [r0, r_end) of expert e (e < 0: a tile past the grouping's count, nothing to
// do).  Returned by value: the reference-parameter form kept it in scratch memory.
struct TileRows {
    int r0, r_end, e;
};
template <int BN = KQ_BN>
__device__ __forceinline__ TileRows tile_rows(const KqP &p, int tg) {
    if (!p.grouped) return TileRows{tg * BN, p.n_tok, 0};
    if (tg >= *p.grp.n_tiles) return TileRows{0, 0, -1};
    const int e = p.grp.tile_e[tg], r0 = p.grp.tile_r0[tg];
    return TileRows{r0, min(p.grp.off[e + 1], r0 + BN), e};
}
__device__ __forceinline__ int act_row(const KqP &p, int r) { return p.grouped && p.grp.amap ? p.grp.amap[r] : r; }
__device__ __forceinline__ int out_row(const KqP &p, int r) { return p.grouped && p.grp.omap ? p.grp.omap[r] : r; }
constexpr int KA_ST = 128 + 16;  // activation bytes per token in LDS (one half superblock, padded)
// weight code bytes per row in LDS (one half superblock, padded): Q4_K keeps its nibble
// pairs, Q5_K one byte per code
template <int TY> constexpr int kw_st() { return (TY == T_Q5_K ? 128 : 64) + 16; }
template <int TY> constexpr int kq_block() { return TY == T_Q5_K ? 176 : 144; }  // superblock bytes
template <int TY> constexpr int kq_qs() { return TY == T_Q5_K ? 48 : 16; }       // offset of its nibbles

// One half superblock; the sub-block scales stay 6-bit bytes, four to a dword.
template <int TY, bool GLU, int BN = KQ_BN>
struct __align__(16) KqStage {
    static constexpr int NW = GLU ? 2 : 1, BM = kq_bm<BN>();
    int8_t a[BN * KA_ST];
    uint8_t wq[NW][BM * kw_st<TY>()];
    uint32_t wsc[NW][BM];          // scales of the half's 4 sub-blocks
};

// What the end of a superblock reads: written with its second half, read in that half.
// Operands of the min term (see below), made once per workgroup: 8 halves for sub-blocks
// 0..3 and 8 for 4..7 of each token and row.
template <bool GLU, int BN = KQ_BN>
struct __align__(16) KqEnd {
    static constexpr int NW = GLU ? 2 : 1, BM = kq_bm<BN>();
    uint4 ab[BN * 2];              // base-64 digits of the tokens' 32-value sums
    uint4 bb[NW][BM * 2];          // m, 64·m
    float da[BN];
    float wd[NW][BM], wdm[NW][BM];
};

template <int TY, bool GLU, int BN = KQ_BN>
struct KqRegs {
    static constexpr int NA = BN == 64 ? 2 : 1, NQ = (BN == 32 && GLU) ? 4 : 2;
    v4i a[NA];        // 32 (BN 64) or 16 (BN 32) activation bytes of the thread's token
    float da;
    v4i bs;           // 8 of the token's 16 bsums (int16)
    v4i wq[NQ];       // 32 nibble bytes of the thread's row (64, both units, in the 32-token gated form)
    v4i qh[TY == T_Q5_K ? 2 : 1];  // Q5_K: the superblock's 32 bytes of fifth bits
    v4i hdr;          // d, dmin, scales[12]
};

// stage loads for half hs of superblock sb
// tokA: the activation row of the thread's token (tid/4, or tid/8 for BN 32); tokD: of
// token tid % BN (tid < 2·BN); woff: the expert's byte offset in a grouped launch
template <int TY, bool GLU, int BN, int hs>
__device__ __forceinline__ void kq_load(const KqP &p, int sg, int row0, int tokA, int tokD, size_t woff, int sb, int tid,
                                        KqRegs<TY, GLU, BN> &R) {
    static_assert(TY == T_Q4_K || BN == 64, "32-token tiles serve Q4_K");
    const int K = p.K, nsb = K >> 8;
    if constexpr (BN == 64) {
        const v4i *src = (const v4i *)(p.qs + (size_t)tokA * K + 256 * sb + 128 * hs + 32 * (tid & 3));
        R.a[0] = src[0];
        R.a[1] = src[1];
    } else {
        R.a[0] = *(const v4i *)(p.qs + (size_t)tokA * K + 256 * sb + 128 * hs + 16 * (tid & 7));
    }
    if (hs == 1 && tid < 2 * BN) {
        R.da = p.d[(size_t)tokD * nsb + sb];
        R.bs = *(const v4i *)(p.bsums + (size_t)tokD * (K >> 4) + 16 * sb + 8 * (tid / BN));
    }
    if constexpr (BN == 32 && GLU) {  // thread → (matrix, row): both units of the half
        const int nw = tid >> 7;
        const int row = min(row0 + (tid & 127), p.rows[0] - 1);
        const uint8_t *blk = p.w[nw] + woff + (size_t)row * p.rb[nw] + 144 * (size_t)sb;
        const v4i *q = (const v4i *)(blk + 16 + 64 * hs);
#pragma unroll
        for (int i = 0; i < 4; i++) R.wq[i] = wload(q + i);
        R.hdr = wload((const v4i *)blk);
    } else if (GLU || BN == 32 || tid < 128) {  // thread → (matrix, row, unit)
        const int nw = (GLU && BN == 64) ? (tid >> 7) : 0, idx = BN == 64 ? (tid & 127) : tid, u = idx & 1;
        const int s = GLU ? nw : sg;
        const int row = min(row0 + (idx >> 1), p.rows[GLU ? 0 : sg] - 1);
        const uint8_t *blk = p.w[s] + woff + (size_t)row * p.rb[s] + kq_block<TY>() * (size_t)sb;
        const v4i *q = (const v4i *)(blk + kq_qs<TY>() + 64 * hs + 32 * u);
        R.wq[0] = wload(q);
        R.wq[1] = wload(q + 1);
        if constexpr (TY == T_Q5_K) {
            R.qh[0] = wload((const v4i *)(blk + 16));
            R.qh[1] = wload((const v4i *)(blk + 32));
        }
        R.hdr = wload((const v4i *)blk);
    }
}

typedef _Float16 half2k __attribute__((ext_vector_type(2)));

// hs: the half that R holds
template <int TY, bool GLU, int BN, int hs>
__device__ __forceinline__ void kq_store(KqStage<TY, GLU, BN> &S, KqEnd<GLU, BN> &E, int tid, const KqRegs<TY, GLU, BN> &R) {
    if constexpr (BN == 64) {
        v4i *dst = (v4i *)(S.a + (tid >> 2) * KA_ST + 32 * (tid & 3));
        dst[0] = R.a[0];
        dst[1] = R.a[1];
    } else {
        *(v4i *)(S.a + (tid >> 3) * KA_ST + 16 * (tid & 7)) = R.a[0];
    }
    if (hs == 1 && tid < 2 * BN) {
        if (tid < BN) E.da[tid] = R.da;
        uint32_t q[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {  // bsum_2j + bsum_2j+1 = the two int16 halves of dword j
            const int bs = (int)(int16_t)(R.bs[j] & 0xffff) + (R.bs[j] >> 16);
            const half2k d = {(_Float16)(int16_t)(bs & 63), (_Float16)(int16_t)(bs >> 6)};
            q[j] = __builtin_bit_cast(uint32_t, d);
        }
        E.ab[2 * (tid % BN) + tid / BN] = make_uint4(q[0], q[1], q[2], q[3]);
    }
    if (GLU || BN == 32 || tid < 128) {
        int nw, row, u;
        if constexpr (BN == 32 && GLU) {
            nw = tid >> 7;
            row = tid & 127;
            u = 0;
            v4i *dst = (v4i *)(S.wq[nw] + row * kw_st<TY>());
#pragma unroll
            for (int i = 0; i < 4; i++) dst[i] = R.wq[i];
        } else {
            nw = (GLU && BN == 64) ? (tid >> 7) : 0;
            const int idx = BN == 64 ? (tid & 127) : tid;
            row = idx >> 1;
            u = idx & 1;
            if constexpr (TY == T_Q5_K) {
                // the unit's two sub-blocks as bytes: nibble + 16·(bit 2(2hs + u) of qh, and
                // the next bit for the high nibbles): quant/reference.rs:321-350
                const int b0 = 4 * hs + 2 * u;
                v4i lo[2], hi[2];
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const uint32_t q = (uint32_t)R.wq[i][c], b = (uint32_t)R.qh[i][c] >> b0;
                        lo[i][c] = (int)((q & 0x0F0F0F0Fu) | ((b & 0x01010101u) << 4));
                        hi[i][c] = (int)(((q >> 4) & 0x0F0F0F0Fu) | ((b & 0x02020202u) << 3));
                    }
                v4i *dst = (v4i *)(S.wq[nw] + row * kw_st<TY>() + 64 * u);
                dst[0] = lo[0];
                dst[1] = lo[1];
                dst[2] = hi[0];
                dst[3] = hi[1];
            } else {
                v4i *dst = (v4i *)(S.wq[nw] + row * kw_st<TY>() + 32 * u);
                dst[0] = R.wq[0];
                dst[1] = R.wq[1];
            }
        }
        // get_scale_min_k4 (quant/reference.rs:8-16), four sub-blocks at a time
        const uint32_t h0 = (uint32_t)R.hdr[0], h1 = (uint32_t)R.hdr[1], h2 = (uint32_t)R.hdr[2], h3 = (uint32_t)R.hdr[3];
        if (u == 0) S.wsc[nw][row] = hs == 0 ? h1 & 0x3F3F3F3Fu : (h3 & 0x0F0F0F0Fu) | ((h1 >> 2) & 0x30303030u);
        if (hs == 1) {
            constexpr bool BOTH = BN == 32 && GLU;  // one thread for the row's two units
#pragma unroll
            for (int k = 0; k < (BOTH ? 2 : 1); k++) {
                const int uu = BOTH ? k : u;
                const uint32_t mn = uu == 0 ? h2 & 0x3F3F3F3Fu : ((h3 >> 4) & 0x0F0F0F0Fu) | ((h2 >> 2) & 0x30303030u);
                uint32_t q[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {  // 0x6400 | m is the half 1024 + m
                    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, mn, 0x04000400u | (uint32_t)j | (uint32_t)j << 16);
                    const half2k v = (__builtin_bit_cast(half2k, b) - half2k{1024, 1024}) * half2k{1, 64};
                    q[j] = __builtin_bit_cast(uint32_t, v);
                }
                E.bb[nw][2 * row + uu] = make_uint4(q[0], q[1], q[2], q[3]);
            }
            if (u == 0) {
                E.wd[nw][row] = h2f(h0 & 0xffff);
                E.wdm[nw][row] = h2f(h0 >> 16);
            }
        }
    }
}

// c + a·b for |a|, |b| < 2^23 on the full-rate 24-bit multiplier (v_mul_i32_i24,
// folded into v_mad_i32_i24 where the compiler can); a 32-bit product would be the
// quarter-rate v_mul_lo_u32.  Plain code, not inline asm: b is an MFMA result, and
// the compiler inserts the wait states between an MFMA and a VALU read of its
// result only for instructions it generates itself.
__device__ __forceinline__ int mad24(int a, int b, int c) { return c + __mul24(a, b); }

// Keeps the 16 sums where they are computed: the compiler otherwise moves a product's
// multiply-adds past the stage's barrier, to their next use, and splits them into
// products and three-operand sums.
__device__ __forceinline__ void pin16(int (&s)[16]) {
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]), "+v"(s[6]), "+v"(s[7]), "+v"(s[8]),
                 "+v"(s[9]), "+v"(s[10]), "+v"(s[11]), "+v"(s[12]), "+v"(s[13]), "+v"(s[14]), "+v"(s[15]));
}

template <int TY, bool GLU, int BN = KQ_BN>
__global__ __launch_bounds__(256, TY == T_Q5_K && !GLU ? 3 : 1) void gemm_q45k_kernel(KqP p) {
    constexpr bool FINE = TY == T_Q5_K && !GLU;
    constexpr int NW = GLU ? 2 : 1, BM = kq_bm<BN>(), WC = BN / 32;  // waves along the tokens
    __shared__ KqStage<TY, GLU, BN> st[2];
    __shared__ KqEnd<GLU, BN> en;
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    const int wr = wv / WC, wc = wv % WC;
    constexpr bool KSPLIT = BN == 64;
    const GemmTile gt = gemm_tile(blockIdx.x, p.n_rg, p.n_tg, KSPLIT ? p.ks : 1, p.grouped);
    const int rg = gt.rg, tg = gt.tg, ksi = gt.ks;
    if (rg < 0) return;  // whole workgroup: uniform
    const int sg = (!GLU && p.nseg > 1 && rg >= p.rg_end[0]) ? ((p.nseg > 2 && rg >= p.rg_end[1]) ? 2 : 1) : 0;
    const int row0 = (rg - (sg ? p.rg_end[sg - 1] : 0)) * BM;
    const TileRows tr = tile_rows<BN>(p, tg);
    if (tr.e < 0) return;  // whole workgroup: uniform
    const size_t woff = p.grouped ? (size_t)tr.e * p.grp.wstride : 0;
    const int tokA = act_row(p, min(tr.r0 + (tid >> (BN == 64 ? 2 : 3)), tr.r_end - 1));
    const int tokD = act_row(p, min(tr.r0 + (tid & (BN - 1)), tr.r_end - 1));
    const int h = l >> 5, m = l & 31;
    const int tok_m = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    const int wrow = wr * 32 + m;   // this lane's weight row (B operand / result column)
    const int arow = wc * 32 + tok_m;  // this lane's token row of the A operands
    const v16i zi = {0};
    const v16f zf = {0};
    const v32f zf32 = {0};

    float acc[NW][16];
    int s1[NW][16];
#pragma unroll
    for (int a = 0; a < NW; a++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[a][v] = 0.0f;
    float tot[FINE ? 16 : 1] = {};
    // this workgroup's superblocks [sb0, sb1) (its K split)
    const int nsb = p.K >> 8;
    const int sb0 = KSPLIT ? ksi * nsb / p.ks : 0, sb1 = KSPLIT ? (ksi + 1) * nsb / p.ks : nsb;
    KqRegs<TY, GLU, BN> R;
    kq_load<TY, GLU, BN, 0>(p, sg, row0, tokA, tokD, woff, sb0, tid, R);
    kq_store<TY, GLU, BN, 0>(st[0], en, tid, R);
    __syncthreads();
    auto half = [&](int sb, auto hc) {
        constexpr int hs = decltype(hc)::value;
        const bool more = hs == 0 || sb + 1 < sb1;
        if (more) kq_load<TY, GLU, BN, 1 - hs>(p, sg, row0, tokA, tokD, woff, sb + hs, tid, R);
        const KqStage<TY, GLU, BN> &S = st[hs];
        uint32_t scw[NW];
#pragma unroll
        for (int a = 0; a < NW; a++) scw[a] = S.wsc[a][wrow];
        // all operands of the half, then its 4·NW products with the MFMA of product q + 1
        // issued ahead of the multiply-adds of q; the fences keep it so (left alone, the
        // scheduler issues every MFMA first, at 250 to 490 registers)
        constexpr int NQ = TY == T_Q5_K ? 4 : 2;
        v4i av[4], wq[NW][NQ];
#pragma unroll
        for (int j = 0; j < 4; j++) av[j] = *(const v4i *)(S.a + arow * KA_ST + 32 * j + 16 * h);
#pragma unroll
        for (int a = 0; a < NW; a++)
#pragma unroll
            for (int j = 0; j < NQ; j++) wq[a][j] = *(const v4i *)(S.wq[a] + wrow * kw_st<TY>() + 32 * j + 16 * h);
        v16i I[2];
        auto issue = [&](int q) {
            const int j = q / NW, a = q % NW;
            v4i bw;
            if constexpr (TY == T_Q5_K) bw = wq[a][j];
            else
#pragma unroll
                for (int i = 0; i < 4; i++) bw[i] = (int)(((uint32_t)wq[a][j >> 1][i] >> (4 * (j & 1))) & 0x0F0F0F0Fu);
            I[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[j], bw, zi, 0, 0, 0);
        };
        issue(0);
#pragma unroll
        for (int q = 0; q < 4 * NW; q++) {
            if (q + 1 < 4 * NW) issue(q + 1);
            __builtin_amdgcn_sched_barrier(0);
            const int j = q / NW, a = q % NW;
            const int sc = (int)(scw[a] >> (8 * j) & 0xff);  // sc < 64, |I| < 2^17
#pragma unroll
            for (int v = 0; v < 16; v++) s1[a][v] = hs == 0 && j == 0 ? __mul24(sc, I[q & 1][v]) : mad24(sc, I[q & 1][v], s1[a][v]);
            pin16(s1[a]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (hs == 1) {  // end of the superblock: the min term and the two scale products
            const half8k ab = __builtin_bit_cast(half8k, en.ab[2 * arow + h]);
#pragma unroll
            for (int a = 0; a < NW; a++) {
                // Σ_j m_j·bs_j exactly on one f16 MFMA: k-slots 2j, 2j + 1 hold the base-64
                // digits of the block sum (bs = 64·hi + lo, |bs| ≤ 32·127) against m_j and
                // 64·m_j; every product and partial sum is an integer below 2^24.  Lane half h
                // supplies sub-blocks 4h..4h+3.
                const half8k bb = __builtin_bit_cast(half8k, en.bb[a][2 * wrow + h]);
                const v16f s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(ab, bb, zf, 0, 0, 0);
                // d·d_a and dmin·d_a in one two-block outer product (block 0: lanes 0-31, d;
                // block 1: lanes 32-63, dmin)
                const v32f pp = __builtin_amdgcn_mfma_f32_32x32x1f32(en.da[arow], h == 0 ? en.wd[a][wrow] : en.wdm[a][wrow], zf32, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    // Q5_K: two rounding steps less (gate/up 2 × 8192 × 3072, 421 tokens: 91
                    // against 95 µs); Q4_K keeps the roundings its prompts always had, since
                    // others move near-tied expert choices
                    if constexpr (TY == T_Q5_K) acc[a][v] = fmaf(pp[v], (float)s1[a][v], fmaf(-pp[16 + v], s2[v], acc[a][v]));
                    else acc[a][v] += pp[v] * (float)s1[a][v] - pp[16 + v] * s2[v];
                }
            }
        }
        if (more) kq_store<TY, GLU, BN, 1 - hs>(st[1 - hs], en, tid, R);
        __syncthreads();
    };
    for (int sb = sb0; sb < sb1; sb++) {
        half(sb, std::integral_constant<int, 0>{});
        half(sb, std::integral_constant<int, 1>{});
        // Q5_K down projections: sums of 8 superblocks, then of those (K 14336 in one chain
        // has 1.3 to 2.1 times the error against float64 of the batched GEMV, which ran them before)
        if (FINE && ((sb - sb0) % 8 == 7 || sb + 1 == sb1)) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                tot[FINE ? v : 0] += acc[0][v];
                acc[0][v] = sb + 1 == sb1 ? tot[FINE ? v : 0] : 0.0f;
            }
        }
    }
    // ---- epilogue: lane holds weight row row0 + wrow for tokens t0 + wc·32 + 16h + v ----
    if constexpr (KSPLIT) {
        if (p.ks > 1 && !p.plane && !split_sum(reinterpret_cast<float(&)[NW * 16]>(acc), p.ws.part, (uint32_t)(p.ws.cap * 4), p.ws.cnt,
                                   rg * p.n_tg + tg, ksi, p.ks))
            return;
    }
    const int rows = p.rows[sg];
    const int row = row0 + wrow;
    if (row >= rows) return;
    const bool part = p.plane && ksi;
    float *out = part ? p.ws.part + (size_t)(ksi - 1) * p.plane : p.out[sg];
    const int ld = p.ld[sg];
    const int epi = part ? EPI_STORE : p.epi[sg];
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int r = tr.r0 + wc * 32 + 16 * h + v;
        if (r < tr.r_end) {
            float y = acc[0][v];
            if constexpr (GLU) y = (p.glu == 2 ? gelu_tanh_f(acc[0][v]) : silu_f(acc[0][v])) * acc[NW - 1][v];
            float *o = out + (size_t)out_row(p, r) * ld + row;
            if (epi == EPI_ADD) *o += y;
            else *o = y;
        }
    }
}

// ---- Q6_K ----------------------------------------------------------------
constexpr int K6_ST = 128 + 16;  // weight code bytes per row in LDS (one half superblock, padded)

// Codes lie in 8-byte groups in the order 0, 2, 1, 3 of each 32 values, so that a lane
// half's groups of two 16-value sub-blocks are one 16-byte read.
template <bool GLU>
struct __align__(16) K6Stage {
    static constexpr int NW = GLU ? 2 : 1;
    int8_t a[KQ_BN * KA_ST];
    int8_t wq[NW][KQ_BM * K6_ST];  // q6 − 32 of the half
    uint2 wsc[NW][KQ_BM];          // the half's 8 signed sub-block scales
};
template <bool GLU>
struct K6End {  // scales of the superblock: written with its second half, read in that half
    float da[KQ_BN];
    float wd[GLU ? 2 : 1][KQ_BM];
};

struct __attribute__((packed, aligned(2))) K6B8 {
    uint32_t w[2];
};
struct K6W {  // one weight row's part of a half superblock: 8 bytes each from a 2-byte boundary
    K6B8 lo, hi, qh, sc;
    uint32_t d;
};

template <bool GLU>
struct K6Regs {
    v4i a[2];
    float da;
    K6W w[GLU ? 2 : 1];
};

// thread → (row tid/4, part tid%4): values l + 32i of the half, l in 8·part..+8, i = 0..3
template <bool GLU, int hs>
__device__ __forceinline__ void k6_load(const KqP &p, int sg, int row0, int tokA, int tokD, size_t woff, int sb, int tid, K6Regs<GLU> &R) {
    const int K = p.K, nsb = K >> 8;
    {
        const v4i *src = (const v4i *)(p.qs + (size_t)tokA * K + 256 * sb + 128 * hs + 32 * (tid & 3));
        R.a[0] = src[0];
        R.a[1] = src[1];
    }
    if (hs == 1 && tid < KQ_BN) R.da = p.d[(size_t)tokD * nsb + sb];
    const int row = min(row0 + (tid >> 2), p.rows[GLU ? 0 : sg] - 1), part = tid & 3;
#pragma unroll
    for (int a = 0; a < (GLU ? 2 : 1); a++) {
        const int s = GLU ? a : sg;
        K6W &w = R.w[a];
        const uint8_t *blk = p.w[s] + woff + (size_t)row * p.rb[s] + 210 * (size_t)sb;
        w.lo = *(const K6B8 *)(blk + 64 * hs + 8 * part);
        w.hi = *(const K6B8 *)(blk + 64 * hs + 32 + 8 * part);
        w.qh = *(const K6B8 *)(blk + 128 + 32 * hs + 8 * part);
        if (part == 0) {
            w.sc = *(const K6B8 *)(blk + 192 + 8 * hs);
            if (hs == 1) w.d = *(const uint16_t *)(blk + 208);
        }
    }
}

template <bool GLU, int hs>
__device__ __forceinline__ void k6_store(K6Stage<GLU> &S, K6End<GLU> &E, int tid, const K6Regs<GLU> &R) {
    {
        v4i *dst = (v4i *)(S.a + (tid >> 2) * KA_ST + 32 * (tid & 3));
        dst[0] = v4i{R.a[0][0], R.a[0][1], R.a[1][0], R.a[1][1]};
        dst[1] = v4i{R.a[0][2], R.a[0][3], R.a[1][2], R.a[1][3]};
    }
    if (hs == 1 && tid < KQ_BN) E.da[tid] = R.da;
    const int row = tid >> 2, part = tid & 3;
#pragma unroll
    for (int a = 0; a < (GLU ? 2 : 1); a++) {
        const K6W &R6 = R.w[a];
        // value l + 32i: low nibble of ql[l] (i = 0), ql[l + 32] (i = 1), high nibbles (i = 2, 3);
        // bits 2i, 2i+1 of qh[l] on top (quant/reference.rs:190-212).  Four codes per dword:
        // (q | 0x80) − 32, then bit 7 flipped back, is the int8 q − 32 without cross-byte borrows.
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t *src = (i & 1) ? R6.hi.w : R6.lo.w;
            const int sl = 4 * (i >> 1), sq = 2 * i;
            uint32_t w[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint32_t q = ((src[k] >> sl) & 0x0F0F0F0Fu) | (((R6.qh.w[k] >> sq) & 0x03030303u) << 4);
                w[k] = ((q | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
            }
            *(uint2 *)(S.wq[a] + row * K6_ST + 32 * i + 16 * (part & 1) + 8 * (part >> 1)) = make_uint2(w[0], w[1]);
        }
        if (part == 0) {
            S.wsc[a][row] = make_uint2(R6.sc.w[0], R6.sc.w[1]);
            if (hs == 1) E.wd[a][row] = h2f(R6.d);
        }
    }
}

template <bool GLU>
__global__ __launch_bounds__(256) void gemm_q6k_kernel(KqP p) {
    constexpr int NW = GLU ? 2 : 1;
    __shared__ K6Stage<GLU> st[2];
    __shared__ K6End<GLU> en;
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    const int wr = wv >> 1, wc = wv & 1;
    const GemmTile gt = gemm_tile(blockIdx.x, p.n_rg, p.n_tg, p.ks, p.grouped);
    const int rg = gt.rg, tg = gt.tg, ksi = gt.ks;
    if (rg < 0) return;  // whole workgroup: uniform
    const int sg = (!GLU && p.nseg > 1 && rg >= p.rg_end[0]) ? ((p.nseg > 2 && rg >= p.rg_end[1]) ? 2 : 1) : 0;
    const int row0 = (rg - (sg ? p.rg_end[sg - 1] : 0)) * KQ_BM;
    const TileRows tr = tile_rows(p, tg);
    if (tr.e < 0) return;  // whole workgroup: uniform
    const size_t woff = p.grouped ? (size_t)tr.e * p.grp.wstride : 0;
    const int tokA = act_row(p, min(tr.r0 + (tid >> 2), tr.r_end - 1));
    const int tokD = act_row(p, min(tr.r0 + (tid & 63), tr.r_end - 1));
    const int h = l >> 5, m = l & 31;
    const int tok_m = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    const int wrow = wr * 32 + m;
    const int arow = wc * 32 + tok_m;
    const v16i zi = {0};
    const v16f zf = {0};
    float acc[NW][16];
    int s1[NW][16];
#pragma unroll
    for (int a = 0; a < NW; a++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[a][v] = 0.0f;
    // this workgroup's superblocks [sb0, sb1) (its K split)
    const int nsb = p.K >> 8;
    const int sb0 = ksi * nsb / p.ks, sb1 = (ksi + 1) * nsb / p.ks;
    K6Regs<GLU> R;
    k6_load<GLU, 0>(p, sg, row0, tokA, tokD, woff, sb0, tid, R);
    k6_store<GLU, 0>(st[0], en, tid, R);
    __syncthreads();
    auto half = [&](int sb, auto hc) {
        constexpr int hs = decltype(hc)::value;
        const bool more = hs == 0 || sb + 1 < sb1;
        if (more) k6_load<GLU, 1 - hs>(p, sg, row0, tokA, tokD, woff, sb + hs, tid, R);
        const K6Stage<GLU> &S = st[hs];
        // operands of the half, then its 8·NW products, as in gemm_q45k_kernel
        v4i av[4], bw[NW][4];
        uint2 scw[NW];
#pragma unroll
        for (int k = 0; k < 4; k++) av[k] = *(const v4i *)(S.a + arow * KA_ST + 32 * k + 16 * h);
#pragma unroll
        for (int a = 0; a < NW; a++) {
            scw[a] = S.wsc[a][wrow];
#pragma unroll
            for (int k = 0; k < 4; k++) bw[a][k] = *(const v4i *)(S.wq[a] + wrow * K6_ST + 32 * k + 16 * h);
        }
        auto sub8 = [](const v4i &v, int k) { return (long)(((uint64_t)(uint32_t)v[2 * k + 1] << 32) | (uint32_t)v[2 * k]); };
        v16i D[2];
        auto issue = [&](int q) {
            const int k = q / NW, a = q % NW;  // 16-value sub-block k of the half
            D[q & 1] = __builtin_amdgcn_mfma_i32_32x32x16_i8(sub8(av[k >> 1], k & 1), sub8(bw[a][k >> 1], k & 1), zi, 0, 0, 0);
        };
        issue(0);
#pragma unroll
        for (int q = 0; q < 8 * NW; q++) {
            if (q + 1 < 8 * NW) issue(q + 1);
            __builtin_amdgcn_sched_barrier(0);
            const int k = q / NW, a = q % NW;
            const int sc = (int)(int8_t)((k < 4 ? scw[a].x : scw[a].y) >> (8 * (k & 3)));
#pragma unroll
            for (int v = 0; v < 16; v++) s1[a][v] = hs == 0 && k == 0 ? __mul24(sc, D[q & 1][v]) : mad24(sc, D[q & 1][v], s1[a][v]);
            pin16(s1[a]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (hs == 1) {  // end of the superblock: (d_r·d_t)·Σ sc·D
#pragma unroll
            for (int a = 0; a < NW; a++) {
                const v16f p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(h == 0 ? en.da[arow] : 0.0f, h == 0 ? en.wd[a][wrow] : 0.0f, zf, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; v++) acc[a][v] = fmaf(p1[v], (float)s1[a][v], acc[a][v]);
            }
        }
        if (more) k6_store<GLU, 1 - hs>(st[1 - hs], en, tid, R);
        __syncthreads();
    };
    for (int sb = sb0; sb < sb1; sb++) {
        half(sb, std::integral_constant<int, 0>{});
        half(sb, std::integral_constant<int, 1>{});
    }
    if (p.ks > 1 && !p.plane && !split_sum(reinterpret_cast<float(&)[NW * 16]>(acc), p.ws.part, (uint32_t)(p.ws.cap * 4), p.ws.cnt,
                               rg * p.n_tg + tg, ksi, p.ks))
        return;
    const int rows = p.rows[sg];
    const int row = row0 + wrow;
    if (row >= rows) return;
    const bool part = p.plane && ksi;
    float *out = part ? p.ws.part + (size_t)(ksi - 1) * p.plane : p.out[sg];
    const int ld = p.ld[sg];
    const int epi = part ? EPI_STORE : p.epi[sg];
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int r = tr.r0 + wc * 32 + 16 * h + v;
        if (r < tr.r_end) {
            float y = acc[0][v];
            if constexpr (GLU) y = (p.glu == 2 ? gelu_tanh_f(acc[0][v]) : silu_f(acc[0][v])) * acc[NW - 1][v];
            float *o = out + (size_t)out_row(p, r) * ld + row;
            if (epi == EPI_ADD) *o += y;
            else *o = y;
        }
    }
}

void kq_groups(KqP &p, int nseg, const GroupTiles *grp, int bm = KQ_BM) {
    int acc = 0;
    for (int i = 0; i < 3; i++) {
        if (i < nseg) acc += (p.rows[i] + bm - 1) / bm;
        p.rg_end[i] = acc;
    }
    p.n_rg = acc;
    p.n_tg = (p.n_tok + KQ_BN - 1) / KQ_BN;
    if (grp) {
        p.grouped = 1;
        p.grp = *grp;
        p.n_tg = grp->max_tiles;
    }
}

// Launches of few tiles split K into parts of at least two superblocks, added up in the
// launch; one ungated segment of under 512 tiles into parts of at least four, in planes.
template <int TY, bool GLU, int BN = KQ_BN>
void kq_launch(KqP p, hipStream_t st, const GemmWs &ws = {}) {
    p.ks = p.grouped || BN != 64 ? 1 : split_count(p.n_rg * p.n_tg, p.K >> 8, 2, GLU ? 32 : 16, ws);
    p.ws = ws;
    if (p.ks == 1 && !GLU && BN == 64 && !p.grouped && p.nseg == 1 && p.n_tok > 64) {
        const size_t plane = (size_t)p.n_tok * p.ld[0];
        p.ks = plane_count(p.n_rg * p.n_tg, p.K >> 8, 4, plane, ws);
        p.plane = p.ks > 1 ? plane : 0;
    }
    const dim3 grid(gemm_grid(p.n_rg, p.n_tg, p.ks, p.grouped));
    if constexpr (TY == T_Q6_K) hipLaunchKernelGGL((gemm_q6k_kernel<GLU>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((gemm_q45k_kernel<TY, GLU, BN>), grid, dim3(256), 0, st, p);
    if (p.plane) launch_gemm_add_parts(p.out[0], ws.part, p.plane, p.ks - 1, p.rows[0], p.ld[0], p.n_tok, st);
}

}  // namespace

bool gemm_kq_supported(int ty, size_t K) { return (ty == T_Q4_K || ty == T_Q5_K || ty == T_Q6_K) && K % 256 == 0 && K > 0; }

bool launch_gemm_kq(const GemvSeg *segs, int nseg, const ActQ8 &act, int n_tok, int K, hipStream_t st, const GroupTiles *grp,
                    const GemmWs &ws) {
    if (nseg < 1 || nseg > 3 || n_tok < 1 || !act.qs || !act.d || (grp && (nseg != 1 || grp->max_tiles < 1))) return false;
    const int ty = segs[0].w.ty;
    if (ty != T_Q6_K && !act.bsums) return false;
    KqP p{};
    for (int i = 0; i < nseg; i++) {
        const GemvSeg &s = segs[i];
        if (s.w.ty != ty || !gemm_kq_supported(s.w.ty, K) || s.w.cols != (size_t)K || !s.w.data || !s.out) return false;
        p.w[i] = s.w.data;
        p.rb[i] = s.w.rb();
        p.rows[i] = (int)s.w.rows;
        p.out[i] = s.out;
        p.ld[i] = s.ld;
        p.epi[i] = s.epi;
    }
    p.nseg = nseg;
    p.n_tok = n_tok;
    p.K = K;
    p.qs = act.qs;
    p.d = act.d;
    p.bsums = act.bsums;
    if (grp && grp->bn != KQ_BN && (grp->bn != 32 || ty != T_Q4_K)) return false;
    const bool t32 = grp && grp->bn == 32;  // 32-token tiles of a Q4_K expert grouping
    kq_groups(p, nseg, grp, t32 ? kq_bm<32>() : KQ_BM);
    if (ty == T_Q6_K) kq_launch<T_Q6_K, false>(p, st, ws);
    else if (ty == T_Q5_K) kq_launch<T_Q5_K, false>(p, st, ws);
    else if (t32) kq_launch<T_Q4_K, false, 32>(p, st);
    else kq_launch<T_Q4_K, false>(p, st, ws);
    return true;
}

bool launch_gemm_kq_glu(const DevWeight &gate, const DevWeight &up, const ActQ8 &act, int n_tok, int K, float *h, int ld, int gelu,
                        hipStream_t st, const GroupTiles *grp, const GemmWs &ws) {
    if (grp && grp->max_tiles < 1) return false;
    if (n_tok < 1 || !act.qs || !act.d || (gate.ty != T_Q6_K && !act.bsums) || gate.ty != up.ty || !gemm_kq_supported(gate.ty, K) ||
        gate.cols != (size_t)K || up.cols != (size_t)K || gate.rows != up.rows || !gate.data || !up.data || !h)
        return false;
    KqP p{};
    p.w[0] = gate.data;
    p.w[1] = up.data;
    p.rb[0] = gate.rb();
    p.rb[1] = up.rb();
    p.rows[0] = p.rows[1] = (int)gate.rows;
    p.out[0] = h;
    p.ld[0] = ld;
    p.epi[0] = EPI_STORE;
    p.nseg = 1;
    p.glu = gelu ? 2 : 1;
    p.n_tok = n_tok;
    p.K = K;
    p.qs = act.qs;
    p.d = act.d;
    p.bsums = act.bsums;
    if (grp && grp->bn != KQ_BN && (grp->bn != 32 || gate.ty != T_Q4_K)) return false;
    const bool t32 = grp && grp->bn == 32;  // 32-token tiles of a Q4_K expert grouping
    kq_groups(p, 1, grp, t32 ? kq_bm<32>() : KQ_BM);
    if (gate.ty == T_Q6_K) kq_launch<T_Q6_K, true>(p, st, ws);
    else if (gate.ty == T_Q5_K) kq_launch<T_Q5_K, true>(p, st, ws);
    else if (t32) kq_launch<T_Q4_K, true, 32>(p, st);
    else kq_launch<T_Q4_K, true>(p, st, ws);
    return true;
}

}  // namespace rie
