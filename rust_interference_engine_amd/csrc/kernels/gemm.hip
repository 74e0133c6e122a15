// gemm.hip — prompt-batch matmul on CDNA4 int8 MFMA (Q4_0 / Q5_0 / Q8_0 weights ×
// Q8_0 activations), the batched counterpart of vec_dot / vec_dot_x4
// (crates/rie-core/src/kernels/mod.rs:136-284, kernels/matmul.rs:119-241).
//
// One wavefront computes 32 weight rows × 32·NT tokens.  Per 32-value block b:
//   I[t][r]  = Σ_k a_q[t][k]·(w_q[r][k] − 8)      v_mfma_i32_32x32x32_i8, exact
//   S[t][r]  = d_a[t][b]·d_w[r][b]                v_mfma_f32_32x32x1f32 (outer product;
//                                                  two blocks' S per instruction)
//   acc      = fma((float)I, S, acc)              VALU
// (Q4_0 codes enter the MFMA as 16·(w_q − 8) and d_w as d_w/16, Q5_0 codes as
// 8·(w_q − 16) and d_w/8: the same I·S)
// so each block contributes (d_w·d_a)·isum exactly as the reference's block dot
// does; only the order of the f32 sum over blocks differs.  Weights stay in
// their ggml layout: a thread loads a block (two of a gated pair) per stage and
// writes its codes to LDS as int8, for Q4_0 with the nibbles unpacked to 16·(q − 8)
// and the 1/16 on the block scale (once per workgroup, not per wave).
//
// Operand lane layout (checked by the parity tests): lane l supplies row
// (l mod 32) and values 16·(l/32)..+16 of the block, for A (tokens) and B
// (weights) alike; the 32×32 result holds column l mod 32 (weight row) and rows
// 8·(v/4) + 4·(l/32) + v mod 4 (v = 0..15).  Tokens are permuted onto A's rows
// so that lane l's 16 results are the 16 consecutive tokens 16·(l/32) + v.
#include "../common.hpp"
#include "../device.hpp"
#include "../kernels.hpp"
#include "../gemm_split.hpp"

#include <algorithm>
#include <type_traits>

namespace rie {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));


struct GemmP {
    const uint8_t *w[3];
    size_t rb[3];
    int rows[3];
    float *out[3];
    int ld[3];
    int epi[3];
    int nseg;
    int rg_end[3];  // cumulative row groups (64 rows) at the end of each segment
    int n_rg;       // row groups in total
    int n_tg;       // token groups
    int glu;        // 0 none; 1 silu / 2 gelu-tanh: seg 0 gate, seg 1 up, out[0] = h
    const int8_t *qs;
    const float *d;
    int n_tok, K;
    int grouped;    // expert groups: one matrix per expert (grp), 64-token tiles from its table
    GroupTiles grp;
    int ks;  // K splits of a tile (not grouped), added up in ws by the last of them
    GemmWs ws;
    size_t plane;  // floats per plane of a split in planes (plane_count), 0: split_sum
};

// A workgroup's token rows: tokens [r0, r_end) of the batch, or gathered rows
// [r0, r_end) of expert e (e < 0: a tile past the grouping's count).  Returned by
// value: the reference-parameter form kept the struct in scratch memory.
struct GTileRows {
    int r0, r_end, e;
};
__device__ __forceinline__ GTileRows gtile_rows(const GemmP &p, int tg, int bn) {
    if (!p.grouped) return GTileRows{tg * bn, p.n_tok, 0};
    if (tg >= *p.grp.n_tiles) return GTileRows{0, 0, -1};
    const int e = p.grp.tile_e[tg], r0 = p.grp.tile_r0[tg];
    return GTileRows{r0, min(p.grp.off[e + 1], r0 + bn), e};
}
__device__ __forceinline__ int gact_row(const GemmP &p, int r) { return p.grouped && p.grp.amap ? p.grp.amap[r] : r; }
__device__ __forceinline__ int gout_row(const GemmP &p, int r) { return p.grouped && p.grp.omap ? p.grp.omap[r] : r; }

template <int TY> constexpr int block_dwords() { return TY == T_Q8_0 ? 8 : 4; }  // of codes

// Weight unit: blocks b and b+1 of one row (36, 44 or 68 bytes from a dword boundary),
// for the gated pair, whose 256 threads have two blocks each.
template <int TY> constexpr int unit_dwords() { return 2 * block_dwords<TY>() + (TY == T_Q5_0 ? 3 : 1); }
template <int TY>
struct WUnit {
    uint32_t w[unit_dwords<TY>()];
};

template <int TY>
__device__ __forceinline__ void load_wunit(const uint8_t *row, int b, WUnit<TY> &u) {
    const uint32_t *p = (const uint32_t *)(row + (size_t)b * (2 * unit_dwords<TY>()));
#pragma unroll
    for (int i = 0; i < unit_dwords<TY>(); i++) u.w[i] = wload(p + i);
}

// One block's bytes, for the other launches, whose 256 threads have one block each: in
// units, half of the threads held two and the staging was two of the four waves' work
// (512 tokens, Q8_0, Q/K/V 6144 × 4096: 84 us, wo 4096 × 4096: 81 us; now 64 and 50 us;
// the gated pair by blocks 291 us against 237 us by units).  Blocks start at any even
// address.  Q4_0 in 128-token tiles keeps units (down 4096 × 14336: 115 against 118 us).
struct __attribute__((packed, aligned(2))) Bytes16 {
    uint32_t w[4];
};
struct __attribute__((packed, aligned(2))) Bytes4 {
    uint32_t w;
};
template <int TY>
struct WBlk {
    Bytes16 q[block_dwords<TY>() / 4];
    uint32_t qh;  // Q5_0
    uint32_t d;
};

template <int TY>
__device__ __forceinline__ void load_wblk(const uint8_t *row, int b, WBlk<TY> &u) {
    constexpr int HD = TY == T_Q5_0 ? 6 : 2, BB = HD + 4 * block_dwords<TY>();
    const uint8_t *p = row + (size_t)b * BB;
    u.d = *(const uint16_t *)p;
    if constexpr (TY == T_Q5_0) u.qh = ((const Bytes4 *)(p + 2))->w;
#pragma unroll
    for (int i = 0; i < block_dwords<TY>() / 4; i++) u.q[i] = *(const Bytes16 *)(p + HD + 16 * i);
}

// ---- LDS-tiled kernel ---------------------------------------------------------
// Workgroup tile: 64 weight rows × 128 tokens, 4 waves as 2 (rows) × 2 (tokens),
// each wave 32 rows × 64 tokens.  Per stage of KC = 4 blocks (128 values of K)
// the workgroup stages the activation codes and scales and the weight codes
// (nibbles kept packed, 16 B/block for Q4_0) and scales in LDS; the next
// stage's global loads are in flight while the current stage is multiplied.
constexpr int G_BM = 64, G_KC = 4;  // G_KC: 32-value blocks per LDS stage
constexpr int G_AST = G_KC * 32 + 16;  // activation row stride in LDS (bytes, padded)

template <int TY>
struct GemmLds {
    static constexpr int QB = 32;                       // weight codes per block in LDS: int8 (Q4_0 unpacked as 16·(q − 8))
    static constexpr int WST = G_KC * QB + 16;          // weight row stride (bytes, padded)
};

// BN tokens per workgroup tile: 128 (two 32-token tiles per wave) or 64 (one)
template <int TY, bool GLU, int BN>
constexpr bool by_units() { return GLU || (TY == T_Q4_0 && BN == 128); }

template <int TY, bool GLU, int BN>
struct __align__(16) GemmStage {
    static constexpr int NW = GLU ? 2 : 1;
    int8_t a[BN * G_AST];
    float da[BN * G_KC];
    uint8_t wq[NW][G_BM * GemmLds<TY>::WST];
    float dw[NW][G_BM * G_KC];
};

// registers holding one stage's global loads before they are written to LDS
template <int TY, bool GLU, int BN>
struct StageRegs {
    static constexpr int NW = GLU ? 2 : 1;
    v4i a[BN / 32];  // the thread's part of its token's 128-byte chunk
    float4 da;
    std::conditional_t<by_units<TY, GLU, BN>(), WUnit<TY>, WBlk<TY>> w;
};

// tokA: the activation row of the thread's token (tid / (256/BN)); tokD: of token tid
// (tid < BN); woff: the expert's byte offset in a grouped launch
// TAIL: K is an odd multiple of 64, so the last stage holds two blocks.  Its other two
// repeat the row's last ones (in bounds) with both scales 0 (the weights' at the store: an
// infinite one would make the row NaN).  (As a run-time check in every launch this took a
// 512-token Q8_0 prompt from 1353 to 1478 us.)
template <int TY, bool GLU, int BN, bool TAIL>
__device__ __forceinline__ void stage_load(const GemmP &p, int sg, int row0, int tokA, int tokD, size_t woff, int b0, int tid,
                                           StageRegs<TY, GLU, BN> &R) {
    const int K = p.K, nb = K >> 5;
    const bool tail = TAIL && b0 + G_KC > nb;  // workgroup-uniform
    {   // activation codes: thread → (token, part of its 128-byte chunk)
        constexpr int TPT = 256 / BN, NV = 128 / TPT / 16;  // threads per token, 16-byte loads per thread
        const int k = 32 * b0 + 16 * NV * (tid % TPT);
        const v4i *src = (const v4i *)(p.qs + (size_t)tokA * K + (tail ? min(k, K - 16 * NV) : k));
#pragma unroll
        for (int i = 0; i < NV; i++) R.a[i] = src[i];
    }
    if (!TAIL && tid < BN) R.da = *(const float4 *)(p.d + (size_t)tokD * nb + b0);
    if (TAIL && tid < BN) {
        const float *d = p.d + (size_t)tokD * nb + b0;
        const float2 d01 = *(const float2 *)d;
        const float2 d23 = *(const float2 *)(tail ? d : d + 2);
        R.da = make_float4(d01.x, d01.y, tail ? 0.0f : d23.x, tail ? 0.0f : d23.y);
    }
    if constexpr (by_units<TY, GLU, BN>()) {  // weights: thread → (matrix, row, unit)
        const int idx = tid & 127, sm = GLU ? (tid >> 7) : sg;
        const int row = min(row0 + (idx >> 1), p.rows[GLU ? 0 : sg] - 1);
        if (GLU || tid < 128) load_wunit<TY>(p.w[sm] + woff + (size_t)row * p.rb[sm], b0 + (tail ? 0 : 2 * (idx & 1)), R.w);
    } else {  // thread → (row, block)
        const int row = min(row0 + (tid >> 2), p.rows[sg] - 1), b = b0 + (tid & 3);
        load_wblk<TY>(p.w[sg] + woff + (size_t)row * p.rb[sg], tail ? min(b, nb - 1) : b, R.w);
    }
}

// a block's codes as int8 to LDS, and its scale
template <int TY>
__device__ __forceinline__ void put_block(const uint32_t (&q)[block_dwords<TY>()], uint32_t qh, uint32_t d, uint8_t *wq, float *dw) {
    if constexpr (TY == T_Q4_0) {
        // nibbles → int8 16·(q − 8) once per workgroup: bytes 0..15 of a block are
        // values 0..15 (low nibbles), bytes 16..31 values 16..31 (high nibbles).
        // q ^ 8 is q − 8 as a 4-bit two's complement number, so with every nibble
        // flipped by one XOR, a nibble moved into (or left in) the high half of its
        // byte, low half zero, is the int8 16·(q − 8): 4 instructions per 8 codes.
        // The block's product is then 16·I exactly (|16·I| < 2²⁴) and its weight
        // scale carries the 1/16 (a power of two: d_a·d_w/16 and the fma with 16·I
        // round exactly as d_a·d_w and I do).
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t f = q[k] ^ 0x88888888u;
            lo[k] = (f << 4) & 0xF0F0F0F0u;
            hi[k] = f & 0xF0F0F0F0u;
        }
        *(uint4 *)wq = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        *(uint4 *)(wq + 16) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        *dw = h2f(d) * 0.0625f;
    } else if constexpr (TY == T_Q5_0) {
        // a nibble with its fifth bit (bit j of qh for value j) put above it is the
        // 5-bit code q; q ^ 16 is q − 16 as a two's complement number, and moved to
        // the top of its byte the int8 8·(q − 16)
        auto code = [](uint32_t nib, uint32_t bits) {  // 4 nibbles in bytes, their fifth bits in bits 0..3
            const uint32_t e = (bits << 4 | bits << 11 | bits << 18 | bits << 25) & 0x10101010u;
            return ((nib & 0x0F0F0F0Fu) | (e ^ 0x10101010u)) << 3;
        };
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            lo[k] = code(q[k], (qh >> (4 * k)) & 15u);
            hi[k] = code(q[k] >> 4, (qh >> (16 + 4 * k)) & 15u);
        }
        *(uint4 *)wq = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        *(uint4 *)(wq + 16) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        *dw = h2f(d) * 0.125f;
    } else {
#pragma unroll
        for (int k = 0; k < 2; k++) *(uint4 *)(wq + 16 * k) = make_uint4(q[4 * k], q[4 * k + 1], q[4 * k + 2], q[4 * k + 3]);
        *dw = h2f(d);
    }
}

// tail: R holds a last stage of two blocks
template <int TY, bool GLU, int BN, bool TAIL>
__device__ __forceinline__ void stage_store(GemmStage<TY, GLU, BN> &S, int tid, const StageRegs<TY, GLU, BN> &R, bool tail) {
    {
        constexpr int TPT = 256 / BN, NV = 128 / TPT / 16;
        v4i *dst = (v4i *)(S.a + (tid / TPT) * G_AST + 16 * NV * (tid % TPT));
#pragma unroll
        for (int i = 0; i < NV; i++) dst[i] = R.a[i];
    }
    if (tid < BN) *(float4 *)(S.da + tid * G_KC) = R.da;
    constexpr int QB = GemmLds<TY>::QB, WST = GemmLds<TY>::WST, ND = block_dwords<TY>();
    uint32_t q[ND];
    if constexpr (by_units<TY, GLU, BN>()) {
        if (!GLU && tid >= 128) return;
        const int nw = GLU ? (tid >> 7) : 0, row = (tid & 127) >> 1, u = tid & 1;
        const uint32_t *w = R.w.w, keep = TAIL && tail && u ? 0u : ~0u;
        constexpr int C0 = TY == T_Q5_0 ? 1 : 0;  // the dword whose upper half starts block 0's codes
#pragma unroll
        for (int b = 0; b < 2; b++) {
            // block 0's codes start 2 bytes into a dword, block 1's at one
#pragma unroll
            for (int i = 0; i < ND; i++) q[i] = b ? w[unit_dwords<TY>() - ND + i] : __builtin_amdgcn_alignbyte(w[C0 + i + 1], w[C0 + i], 2);
            const uint32_t qh = TY == T_Q5_0 ? (b ? w[6] : __builtin_amdgcn_alignbyte(w[1], w[0], 2)) : 0u;
            put_block<TY>(q, qh, (b ? w[C0 + ND] >> 16 : w[0] & 0xffff) & keep, S.wq[nw] + row * WST + (2 * u + b) * QB, S.dw[nw] + row * G_KC + 2 * u + b);
        }
    } else {
#pragma unroll
        for (int i = 0; i < ND; i++) q[i] = R.w.q[i / 4].w[i % 4];
        put_block<TY>(q, R.w.qh, TAIL && tail && (tid & 2) ? 0u : R.w.d, S.wq[0] + (tid >> 2) * WST + (tid & 3) * QB, S.dw[0] + (tid >> 2) * G_KC + (tid & 3));
    }
}

// Sums in three levels: a stage's four blocks, 8 stages, all of them.  For the launches
// that ran in the batched GEMV before, whose sums are trees: one chain over the K / 32
// blocks has up to 3 times its error against float64 (Q5_0, K 896 / 4096 / 14336, in 1e-7:
// GEMV 0.67 / 0.78 / 0.87, one chain 1.00 / 2.05 / 2.71, three levels 0.72 / 0.84 / 0.95).
// Two waves per SIMD (three spill: 68 against 50 us for 512 tokens, 4096 x 4096); the
// gated and 128-token forms hold one register set of loads (two spill: gate/up 2 x 14336 x
// 4096 321 against 253 us, down 186 against 135 us; in one chain 239 and 127 us).
template <int TY, bool TAIL>
constexpr bool fine_sums() { return TY == T_Q5_0 || TAIL; }

template <int TY, bool GLU, int NT, bool TAIL>
__global__ __launch_bounds__(256, (!GLU && NT == 1 && !fine_sums<TY, TAIL>()) ? 3 : 2) void gemm_kernel(GemmP p) {  // one-tile non-gated: three waves per SIMD
    constexpr bool FINE = fine_sums<TY, TAIL>(), ONE = FINE && (GLU || NT == 2);
    constexpr int NW = GLU ? 2 : 1;
    constexpr int BN = 64 * NT;  // tokens per workgroup tile: NT 32-token tiles per wave, 2 waves along tokens
    constexpr int QB = GemmLds<TY>::QB, WST = GemmLds<TY>::WST;
    __shared__ GemmStage<TY, GLU, BN> st[2];
    const int tid = threadIdx.x;
    const int wv = tid >> 6, l = tid & 63;
    const int wr = wv >> 1, wc = wv & 1;
    const GemmTile gt = gemm_tile(blockIdx.x, p.n_rg, p.n_tg, p.ks, p.grouped);
    const int rg = gt.rg, tg = gt.tg, ksi = gt.ks;
    if (rg < 0) return;  // whole workgroup: uniform
    const int sg = (!GLU && p.nseg > 1 && rg >= p.rg_end[0]) ? ((p.nseg > 2 && rg >= p.rg_end[1]) ? 2 : 1) : 0;
    const int row0 = (rg - (sg ? p.rg_end[sg - 1] : 0)) * G_BM;
    const GTileRows tr = gtile_rows(p, tg, BN);
    if (tr.e < 0) return;  // whole workgroup: uniform
    const size_t woff = p.grouped ? (size_t)tr.e * p.grp.wstride : 0;
    const int tokA = gact_row(p, min(tr.r0 + tid / (256 / BN), tr.r_end - 1));
    const int tokD = gact_row(p, min(tr.r0 + tid % BN, tr.r_end - 1));
    const int h = l >> 5, m = l & 31;
    const int tok_m = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    const int wrow = wr * 32 + m;  // this lane's weight row in the tile (B operand / result column)
    int arow[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) arow[t] = wc * 32 * NT + 32 * t + tok_m;

    float acc[NW][NT][16];
#pragma unroll
    for (int a = 0; a < NW; a++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[a][t][v] = 0.0f;
    float tot[FINE ? NW : 1][NT][16] = {}, part4[16];  // FINE: sums of 8 stages' acc, of one stage
    const v16i zi = {0};
    const v32f zf32 = {0};

    // Stage ring: LDS holds stages s (being multiplied) and s + 1; two register sets
    // hold the global loads of stages s + 1 and s + 2, so a stage's loads are issued
    // two stages before their LDS store.  Load indices past the last stage repeat the
    // last stage and the step count is even, so every load is unconditional and the
    // compiler's wait for a register set counts exactly the loads issued after it.
    // this workgroup's stages: [k0, k0 + n_stages) of the K / 128, rounded up (its K split)
    const int all_stages = (p.K + 32 * G_KC - 1) / (32 * G_KC);
    const int k0 = ksi * all_stages / p.ks;
    const int n_stages = (ksi + 1) * all_stages / p.ks - k0;
    const int last_stage = n_stages - 1;
    StageRegs<TY, GLU, BN> ra, rb;
    stage_load<TY, GLU, BN, TAIL>(p, sg, row0, tokA, tokD, woff, k0 * G_KC, tid, ra);
    auto tail_at = [&](int s) { return TAIL && 32 * G_KC * (k0 + s + 1) > p.K; };
    stage_store<TY, GLU, BN, TAIL>(st[0], tid, ra, tail_at(0));
    stage_load<TY, GLU, BN, TAIL>(p, sg, row0, tokA, tokD, woff, (k0 + min(1, last_stage)) * G_KC, tid, rb);
    __syncthreads();
    // Per stage: all operands of the stage's KC blocks from LDS, then the
    // P = KC·NT·NW tile products in a software pipeline: the MFMAs of product
    // q+1 are issued before the VALU epilogue of product q.
    constexpr int P = G_KC * NT * NW;
    // rl: receives stage s + 2; rs: holds stage s + 1, stored to LDS after stage s (ONE: one
    // register set, which is stored and then loaded again before stage s)
    auto body = [&](int s, StageRegs<TY, GLU, BN> &rl, const StageRegs<TY, GLU, BN> &rs) {
        if (ONE && s + 1 < n_stages) stage_store<TY, GLU, BN, TAIL>(st[(s + 1) & 1], tid, rs, tail_at(s + 1));
        stage_load<TY, GLU, BN, TAIL>(p, sg, row0, tokA, tokD, woff, (k0 + min(s + 2, last_stage)) * G_KC, tid, rl);
        if (s < n_stages) {  // workgroup-uniform; the idle step of an odd stage count skips it
            const GemmStage<TY, GLU, BN> &S = st[s & 1];
            v4i bw[G_KC][NW], av[G_KC][NT];
#pragma unroll
            for (int j = 0; j < G_KC; j++) {
#pragma unroll
                for (int a = 0; a < NW; a++) {
                    const uint4 q = *(const uint4 *)(S.wq[a] + wrow * WST + j * QB + 16 * h);
                    bw[j][a] = v4i{(int)q.x, (int)q.y, (int)q.z, (int)q.w};
                }
#pragma unroll
                for (int t = 0; t < NT; t++) av[j][t] = *(const v4i *)(S.a + arow[t] * G_AST + 32 * j + 16 * h);
            }
            // scale operands of the product pairs (2i, 2i + 1): lane half h supplies
            // product 2i + h's, for the two-block outer product v_mfma_f32_32x32x1f32
            // (block h's 32×32 result in registers 16h..16h+15, laid out as a single
            // block's); one such MFMA per two products halves the scale-MFMA cycles
            // product q: block j of tile (t, a); FINE: a tile's blocks one after the other
            auto blk = [](int q) { return FINE ? q % G_KC : q / (NT * NW); };
            auto tok = [](int q) { return FINE ? q / G_KC / NW : (q / NW) % NT; };
            auto mat = [](int q) { return FINE ? q / G_KC % NW : q % NW; };
            float sa[P / 2], sb[P / 2];
#pragma unroll
            for (int i = 0; i < P / 2; i++) {
                const int qh = 2 * i + h;
                const int jh = blk(qh), th = tok(qh), ah = mat(qh);
                const int arh = wc * 32 * NT + 32 * th + tok_m;
                sa[i] = S.da[arh * G_KC + jh];
                sb[i] = S.dw[ah][wrow * G_KC + jh];
            }
            v16i Iq[2];
            v32f Sp[2];
            // The MFMAs of product q take an (empty asm) dependency on the finished
            // accumulators of product q-2: at most two result pairs are live, and the
            // MFMAs of q overlap the VALU epilogue of q-1.
            auto issue = [&](int q) {
                const int j = blk(q), t = tok(q), a = mat(q);
                v4i aop = av[j][t];
                if (q >= 2) {
                    const float *d = FINE && blk(q - 2) != G_KC - 1 ? part4 : acc[mat(q - 2)][tok(q - 2)];
                    asm volatile("" : "+v"(aop) : "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "v"(d[4]), "v"(d[5]), "v"(d[6]), "v"(d[7]),
                                 "v"(d[8]), "v"(d[9]), "v"(d[10]), "v"(d[11]), "v"(d[12]), "v"(d[13]), "v"(d[14]), "v"(d[15]));
                }
                Iq[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(aop, bw[j][a], zi, 0, 0, 0);
                if ((q & 1) == 0) Sp[(q >> 1) & 1] = __builtin_amdgcn_mfma_f32_32x32x1f32(sa[q >> 1], sb[q >> 1], zf32, 0, 0, 0);
            };
            issue(0);
#pragma unroll
            for (int q = 0; q < P; q++) {
                if (q + 1 < P) issue(q + 1);
                // scheduling fences: the epilogue of q stays between the MFMAs of q + 1 and
                // those of q + 2, so it runs while the matrix core works on q + 1 (left to
                // itself the scheduler moves each epilogue right behind its own MFMAs and
                // fills the latency with s_nop)
                __builtin_amdgcn_sched_barrier(0);
                const int t = tok(q), a = mat(q);
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float I = (float)Iq[q & 1][v], S = Sp[(q >> 1) & 1][16 * (q & 1) + v];
                    if constexpr (!FINE) acc[a][t][v] = fmaf(I, S, acc[a][t][v]);
                    else part4[v] = blk(q) == 0 ? I * S : fmaf(I, S, part4[v]);
                    if (FINE && blk(q) == G_KC - 1) acc[a][t][v] += part4[v];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!ONE && s + 1 < n_stages) stage_store<TY, GLU, BN, TAIL>(st[(s + 1) & 1], tid, rs, tail_at(s + 1));
        __syncthreads();
    };
    for (int s = 0; s < n_stages; s += 2) {
        if constexpr (ONE) {
            body(s, rb, rb);
            body(s + 1, rb, rb);
        } else {
            body(s, ra, rb);
            body(s + 1, rb, ra);
        }
        if (FINE && ((s & 6) == 6 || s + 2 >= n_stages)) {
#pragma unroll
            for (int a = 0; a < NW; a++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        tot[FINE ? a : 0][t][v] += acc[a][t][v];
                        acc[a][t][v] = s + 2 >= n_stages ? tot[FINE ? a : 0][t][v] : 0.0f;
                    }
        }
    }
    // ---- epilogue: lane holds weight row row0 + wrow for tokens t0 + wc·64 + 32t + 16h + v ----
    if (p.ks > 1 && !p.plane && !split_sum(reinterpret_cast<float(&)[NW * NT * 16]>(acc), p.ws.part, (uint32_t)(p.ws.cap * 4), p.ws.cnt,
                               rg * p.n_tg + tg, ksi, p.ks))
        return;
    const int rows = p.rows[sg];
    const int row = row0 + wrow;
    if (row >= rows) return;
    const int ld = p.ld[sg];
    const bool part = p.plane && ksi;
    float *out = part ? p.ws.part + (size_t)(ksi - 1) * p.plane : p.out[sg];
    const int epi = part ? EPI_STORE : p.epi[sg];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int r = tr.r0 + wc * 32 * NT + 32 * t + 16 * h + v;
            if (r < tr.r_end) {
                float y = acc[0][t][v];
                if constexpr (GLU) y = (p.glu == 2 ? gelu_tanh_f(acc[0][t][v]) : silu_f(acc[0][t][v])) * acc[NW - 1][t][v];
                float *o = out + (size_t)gout_row(p, r) * ld + row;
                if (epi == EPI_ADD) *o += y;
                else *o = y;
            }
        }
}

bool gemm_supported(int ty, size_t K) {
    return ((ty == T_Q4_0 || ty == T_Q5_0 || ty == T_Q8_0) && K % 64 == 0 && K > 0) || gemm_kq_supported(ty, K);
}

// out[t·ld + r] += part[0][…] + … + part[n_part−1][…] for r < rows, in split order
__global__ __launch_bounds__(256) void gemm_add_parts_kernel(float *__restrict__ out, const float *__restrict__ part, size_t stride,
                                                             int n_part, int rows, int ld) {
    const int r = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (r >= rows) return;
    const size_t i = (size_t)t * ld + r;
    float v = out[i];
    for (int k = 0; k < n_part; k++) v += part[(size_t)k * stride + i];
    out[i] = v;
}

void launch_gemm_add_parts(float *out, const float *part, size_t stride, int n_part, int rows, int ld, int n_tok, hipStream_t st) {
    hipLaunchKernelGGL(gemm_add_parts_kernel, dim3((rows + 255) / 256, n_tok), dim3(256), 0, st, out, part, stride, n_part, rows, ld);
}

// 128-token tiles where that leaves two workgroups per CU (256 CUs), or where K is long
// (≥ 48 stages of 128, one segment) and splits of ≥ 16 stages in planes leave one per CU;
// otherwise 64-token tiles (one 32-token tile per wave), as always for the gated pair,
// which split K as split_count allows while each split keeps 4 stages.
template <int TY, bool GLU>
static void launch_t(GemmP p, hipStream_t st, const GroupTiles *grp, const GemmWs &ws) {
    const int tiles128 = p.n_rg * ((p.n_tok + 127) / 128);
    const int n_st = (p.K + 32 * G_KC - 1) / (32 * G_KC);
    int nt = 1;
    p.ks = 1;
    p.ws = ws;
    if (!GLU && !grp && p.n_tok > 64) {  // GLU: two register sets of 128-token stages do not fit
        const size_t plane = (size_t)p.n_tok * p.ld[0];
        const int ks = p.nseg == 1 && n_st >= 48 ? plane_count(tiles128, n_st, 16, plane, ws) : 1;
        if (tiles128 >= 512 || (ks > 1 && tiles128 * ks >= 256)) {
            nt = 2;
            p.ks = ks;
            p.plane = ks > 1 ? plane : 0;
        }
    }
    p.n_tg = (p.n_tok + 64 * nt - 1) / (64 * nt);
    if (grp) {  // 64-token tiles from the grouping's table
        static_assert(GROUP_BN == 64, "grouped tiles are one 32-token tile per wave");
        p.grouped = 1;
        p.grp = *grp;
        p.n_tg = grp->max_tiles;
    } else if (nt == 1) {
        p.ks = split_count(p.n_rg * p.n_tg, n_st, 4, GLU ? 32 : 16, ws);
    }
    const dim3 grid(gemm_grid(p.n_rg, p.n_tg, p.ks, p.grouped));
    const bool tail = p.K % (32 * G_KC) != 0;
    if constexpr (!GLU) {
        if (nt == 2 && tail) hipLaunchKernelGGL((gemm_kernel<TY, GLU, 2, true>), grid, dim3(256), 0, st, p);
        else if (nt == 2) hipLaunchKernelGGL((gemm_kernel<TY, GLU, 2, false>), grid, dim3(256), 0, st, p);
        else if (tail) hipLaunchKernelGGL((gemm_kernel<TY, GLU, 1, true>), grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL((gemm_kernel<TY, GLU, 1, false>), grid, dim3(256), 0, st, p);
        if (p.plane) launch_gemm_add_parts(p.out[0], ws.part, p.plane, p.ks - 1, p.rows[0], p.ld[0], p.n_tok, st);
        return;
    }
    if (tail) hipLaunchKernelGGL((gemm_kernel<TY, GLU, 1, true>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((gemm_kernel<TY, GLU, 1, false>), grid, dim3(256), 0, st, p);
}

static bool operands_ok(const ActQ8 &act) { return act.qs && act.d; }

static void set_groups(GemmP &p, int nseg) {
    int acc = 0;
    for (int i = 0; i < 3; i++) {
        if (i < nseg) acc += (p.rows[i] + G_BM - 1) / G_BM;
        p.rg_end[i] = acc;
    }
    p.n_rg = acc;
}

bool launch_gemm(const GemvSeg *segs, int nseg, const ActQ8 &act, int n_tok, int K, hipStream_t st, const GroupTiles *grp,
                 const GemmWs &ws) {
    if (nseg < 1 || nseg > 3 || n_tok < 1 || !operands_ok(act) || (grp && (nseg != 1 || grp->max_tiles < 1))) return false;
    const int ty = segs[0].w.ty;
    if (gemm_kq_supported(ty, K)) return launch_gemm_kq(segs, nseg, act, n_tok, K, st, grp, ws);
    if (grp && grp->bn != GROUP_BN) return false;  // this kernel's grouped tiles are 64 tokens
    GemmP p{};
    for (int i = 0; i < nseg; i++) {
        const GemvSeg &s = segs[i];
        if (s.w.ty != ty || !gemm_supported(s.w.ty, K) || s.w.cols != (size_t)K || !s.w.data || !s.out) return false;
        p.w[i] = s.w.data;
        p.rb[i] = s.w.rb();
        p.rows[i] = (int)s.w.rows;
        p.out[i] = s.out;
        p.ld[i] = s.ld;
        p.epi[i] = s.epi;
    }
    p.nseg = nseg;
    set_groups(p, nseg);
    p.glu = 0;
    p.qs = act.qs;
    p.d = act.d;
    p.n_tok = n_tok;
    p.K = K;
    if (ty == T_Q4_0) launch_t<T_Q4_0, false>(p, st, grp, ws);
    else if (ty == T_Q5_0) launch_t<T_Q5_0, false>(p, st, grp, ws);
    else launch_t<T_Q8_0, false>(p, st, grp, ws);
    return true;
}

bool launch_gemm_glu(const DevWeight &gate, const DevWeight &up, const ActQ8 &act, int n_tok, int K, float *h, int ld, int gelu,
                     hipStream_t st, const GroupTiles *grp, const GemmWs &ws) {
    if (grp && grp->max_tiles < 1) return false;
    if (gemm_kq_supported(gate.ty, K)) return launch_gemm_kq_glu(gate, up, act, n_tok, K, h, ld, gelu, st, grp, ws);
    if (grp && grp->bn != GROUP_BN) return false;  // this kernel's grouped tiles are 64 tokens
    if (n_tok < 1 || !operands_ok(act) || gate.ty != up.ty || !gemm_supported(gate.ty, K) || gate.cols != (size_t)K ||
        up.cols != (size_t)K || gate.rows != up.rows || !gate.data || !up.data || !h)
        return false;
    GemmP p{};
    p.w[0] = gate.data;
    p.w[1] = up.data;
    p.rb[0] = gate.rb();
    p.rb[1] = up.rb();
    p.rows[0] = p.rows[1] = (int)gate.rows;
    p.out[0] = h;
    p.ld[0] = ld;
    p.epi[0] = EPI_STORE;
    p.nseg = 1;
    set_groups(p, 1);
    p.glu = gelu ? 2 : 1;
    p.qs = act.qs;
    p.d = act.d;
    p.n_tok = n_tok;
    p.K = K;
    if (gate.ty == T_Q4_0) launch_t<T_Q4_0, true>(p, st, grp, ws);
    else if (gate.ty == T_Q5_0) launch_t<T_Q5_0, true>(p, st, grp, ws);
    else launch_t<T_Q8_0, true>(p, st, grp, ws);
    return true;
}

}  // namespace rie
