// gemm_float.hip — prompt-batch matmul of unquantized weights (BF16 / F16 × f32
// activations, matmul.rs:119-241 with vec_dot_f16 / vec_dot_bf16) on the 16-bit
// matrix cores of CDNA4, without giving up the f32 activations.
//
// An f32 activation is held as a sum of 16-bit parts, so a weight (exact in its
// own 16-bit type) times an activation is a sum of products that are exact in the
// f32 accumulator:
//   BF16 weights: x = x0 + x1 + x2, three bf16 of 8 bits each, cut off, not rounded
//                 (exact; bf16 has the exponents of f32, so nothing over- or underflows)
//   F16 weights:  2^e·x = x0 + x1 + x2, three f16, with e chosen for each row so that
//                 its largest finite value lies in [2^14, 2^15) (exact down to 2^-39 of
//                 that value, so a value below 2^-15 of it keeps fewer than 24 bits);
//                 the epilogue multiplies by 2^-e
// The parts are made once per batch (split_rows_kernel, which also takes the
// RMSNorm in front of a projection), not per tile.
//
// Sums: an MFMA chain over all of K would round K/16·parts times at full magnitude,
// and the matrix core rounds its sums down (measured: a mean error of -0.6 of the root
// mean square at K 2560).  A chain covers one stage of 32 values, small parts first;
// every other stage runs on negated weights and is subtracted, which cancels the shift;
// stages add up in a second accumulator, and 8 or 16 of those in a third.  Relative error
// (2-norm, in 1e-7, with the residual row's addition) at K 1024 / 2560 / 4864 / 9728:
// 0.77 / 0.89 / 0.99 / 1.04 against 0.93 / 1.01 / 1.12 / 1.25 in the batched GEMV.
//
// Bound: three MFMAs per product, ~830 TFLOP/s of useful rate, or the weight bytes for
// short prompts; measured 180 TFLOP/s (203 tokens, gate/up 2 × 9728 × 2560: 110 us),
// held by LDS operand reads and by the waits between a stage's reads and its MFMAs.  The
// prompt through two layers of hidden 2560: 6.20 ms in the batched GEMV, which reads the
// weights once per 4 tokens, 0.76 ms here.
#include "../common.hpp"
#include "../device.hpp"
#include "../kernels.hpp"
#include "../norm_quant.hpp"

#include <algorithm>

namespace rie {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 fh16x8 __attribute__((ext_vector_type(8)));
typedef float facc __attribute__((ext_vector_type(16)));

namespace {

constexpr int F_PARTS = 3;

// ---- activations ----------------------------------------------------------------

// One workgroup per row: y = RMSNorm(x)·w (or x), f32 to xn (optional) and its parts.
// The norm's sum runs in rmsnorm_kernel's order (or the reference's), so xn is the
// same row.  E and ldx are multiples of 4 (gemm_float_supported: of 32).
template <int TY>
__global__ __launch_bounds__(256) void split_rows_kernel(const float *__restrict__ x, int ldx, const float *__restrict__ w, float eps,
                                                         int E, float *__restrict__ xn, ActSplit act, int ref_order) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float *xr = x + (size_t)row * ldx;
    float scale = 1.0f;
    if (w && ref_order) {
        scale = rms_scale_ref_wg(xr, E, eps, red);
    } else if (w) {
        float ss = 0.0f;
        for (int i0 = 0; i0 < E; i0 += 2048) {  // 8 loads in flight
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = i0 + 256 * k + tid < E ? xr[i0 + 256 * k + tid] : 0.0f;
#pragma unroll
            for (int k = 0; k < 8; k++) ss = fmaf(v[k], v[k], ss);
        }
        ss = wave_sum(ss, 64);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
        __syncthreads();
        scale = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)E + eps);
    }
    auto values = [&](int i) {
        float4 v = *(const float4 *)(xr + i);
        if (w) {
            const float4 g = *(const float4 *)(w + i);
            v = make_float4(v.x * scale * g.x, v.y * scale * g.y, v.z * scale * g.z, v.w * scale * g.w);
        }
        return v;
    };
    float up = 1.0f;  // 2^e
    if constexpr (TY == T_F16) {
        float amax = 0.0f;
        for (int i = 4 * tid; i < E; i += 1024) {
            const float4 v = values(i);
            for (const float y : {v.x, v.y, v.z, v.w})
                if (fabsf(y) < INFINITY) amax = fmaxf(amax, fabsf(y));  // false for NaN too
        }
        amax = wave_max(amax, 64);
        __syncthreads();  // red may still be read above
        if ((tid & 63) == 0) red[tid >> 6] = amax;
        __syncthreads();
        amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        if (amax > 0.0f) {
            const int e = min(max(14 - ilogbf(amax), -113), 126);  // 2^e and 2^-e are normal numbers
            up = __uint_as_float((uint32_t)(127 + e) << 23);
            if (tid == 0) act.scale[row] = __uint_as_float((uint32_t)(127 - e) << 23);
        } else if (tid == 0) {
            act.scale[row] = 1.0f;
        }
    }
    const size_t o = (size_t)row * E;
    for (int i = 4 * tid; i < E; i += 1024) {
        const float4 v = values(i);
        if (xn) *(float4 *)(xn + o + i) = v;
        uint16_t q[3][4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float y = k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w;
            const bool fin = fabsf(y) < INFINITY;
            if constexpr (TY == T_BF16) {
                const uint32_t b = __float_as_uint(y), b0 = b & 0xFFFF0000u;
                const float r1 = y - __uint_as_float(b0);
                const uint32_t b1 = __float_as_uint(r1) & 0xFFFF0000u;
                const float r2 = r1 - __uint_as_float(b1);
                q[0][k] = fin || !(b & 0x7FFFFFu) ? (uint16_t)(b >> 16) : (uint16_t)0x7FC0;
                q[1][k] = fin ? (uint16_t)(b1 >> 16) : (uint16_t)0;
                q[2][k] = fin ? (uint16_t)(__float_as_uint(r2) >> 16) : (uint16_t)0;
            } else {
                // 11 bits each, cut off, so that no conversion rounds
                const float ys = y * up;
                const float x0 = fin ? __uint_as_float(__float_as_uint(ys) & 0xFFFFE000u) : ys, r1 = ys - x0;
                const float x1 = __uint_as_float(__float_as_uint(r1) & 0xFFFFE000u);
                q[0][k] = f2h(x0);
                q[1][k] = fin ? f2h(x1) : (uint16_t)0;
                q[2][k] = fin ? f2h(r1 - x1) : (uint16_t)0;
            }
        }
#pragma unroll
        for (int k = 0; k < F_PARTS; k++)
            *(uint2 *)(act.p[k] + o + i) = make_uint2(q[k][0] | (uint32_t)q[k][1] << 16, q[k][2] | (uint32_t)q[k][3] << 16);
    }
}

// ---- GEMM -----------------------------------------------------------------------

// Workgroup tile: 128 weight rows × 64 tokens; 4 waves as 2 (rows) × 2 (tokens), each
// 64 rows × 32 tokens (128-token tiles, two per wave, leave no registers for the sums:
// 203 tokens, gate/up 2 × 9728 × 2560: 125 against 110 us).  The gated pair's tile is
// 64 gate and 64 up rows.
// Stages of 32 values of K in two LDS buffers, the next stage's loads in registers.
// The row stride of 80 bytes puts 16 rows' 16-byte operands on all 64 banks.
constexpr int F_BM = 128, F_BN = 64, F_BK = 32, F_ST = F_BK * 2 + 16;

struct FGemmP {
    const uint8_t *w[3];
    size_t rb[3];
    int rows[3];
    float *out[3];
    int ld[3];
    int epi[3];
    int rt_end[3];  // cumulative row tiles at the end of each segment
    int nseg, n_rt, n_tt;
    int glu;        // 0 none; 1 silu / 2 gelu-tanh: matrix 0 gate, 1 up, out[0] = h
    ActSplit act;
    int n_tok, K;
    // K split: split i stores its partial sums to part + i·part_stride ([n_tok][part_ld],
    // the segments' rows side by side); a second launch adds them up
    int ks;
    float *part;
    size_t part_stride;
    int part_ld;
    int mid;        // stages per middle sum (a power of two, about the square root of their number)
};

template <int TY>
__device__ __forceinline__ facc fmma(u32x4 a, u32x4 b, facc c) {
    if constexpr (TY == T_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(fh16x8, a), __builtin_bit_cast(fh16x8, b), c, 0, 0, 0);
}

// Σ_k x[k]·w[k] in plain f32, for an output that came out as NaN: an infinite weight
// times a part that is zero or of the other sign is NaN where the sum is not
template <int TY>
__device__ float plain_dot(const ActSplit &act, size_t arow, const uint16_t *w, int k_lo, int k_hi, float scale) {
    float s = 0.0f;
    for (int k = k_lo; k < k_hi; k++) {
        float x, wv;
        if constexpr (TY == T_BF16) {
            x = (__uint_as_float((uint32_t)act.p[2][arow + k] << 16) + __uint_as_float((uint32_t)act.p[1][arow + k] << 16)) +
                __uint_as_float((uint32_t)act.p[0][arow + k] << 16);
            wv = __uint_as_float((uint32_t)w[k] << 16);
        } else {
            x = (h2f(act.p[2][arow + k]) + h2f(act.p[1][arow + k]) + h2f(act.p[0][arow + k])) * scale;
            wv = h2f(w[k]);
        }
        s = fmaf(x, wv, s);
    }
    return s;
}

template <int TY, bool GLU>
__global__ __launch_bounds__(256, 3) void gemm_float_kernel(FGemmP p) {
    constexpr int P = F_PARTS, BN = F_BN;
    constexpr int NA = P * BN * (F_BK / 8) / 256, NWL = F_BM * (F_BK / 8) / 256;  // 16-byte loads per thread and stage
    struct __align__(16) Stage {
        uint8_t a[P][BN * F_ST];
        uint8_t w[F_BM * F_ST];
    };
    __shared__ Stage st[2];
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, h = l >> 5, m = l & 31;
    const int wr = wv >> 1, wc = wv & 1;
    const GemmTile gt = gemm_tile(blockIdx.x, p.n_rt, p.n_tt, p.ks, false);
    const int rt = gt.rg, tt = gt.tg, ksi = gt.ks;
    if (rt < 0) return;  // whole workgroup
    const int sg = (!GLU && p.nseg > 1 && rt >= p.rt_end[0]) ? ((p.nseg > 2 && rt >= p.rt_end[1]) ? 2 : 1) : 0;
    const int row0 = (rt - (sg ? p.rt_end[sg - 1] : 0)) * (GLU ? F_BM / 2 : F_BM);
    const int rows = p.rows[sg], t0 = tt * BN, K = p.K;
    const int all_st = K / F_BK;
    const int s_lo = ksi * all_st / p.ks, n_st = (ksi + 1) * all_st / p.ks - s_lo;

    // this thread's 16-byte pieces of a stage (rows and tokens past the end repeat the last)
    const uint16_t *asrc[NA];
    const uint8_t *wsrc[NWL];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int c = tid + 256 * i, part = c / (BN * 4), r = c / 4 % BN;
        asrc[i] = p.act.p[part] + (size_t)min(t0 + r, p.n_tok - 1) * K + s_lo * F_BK + (c & 3) * 8;
    }
#pragma unroll
    for (int i = 0; i < NWL; i++) {
        const int c = tid + 256 * i, r = c >> 2;
        const int mat = GLU ? r / (F_BM / 2) : sg, wrow = min(row0 + (GLU ? r % (F_BM / 2) : r), rows - 1);
        wsrc[i] = p.w[mat] + (size_t)wrow * p.rb[mat] + (size_t)(s_lo * F_BK + (c & 3) * 8) * 2;
    }
    struct Regs {
        u32x4 a[NA], w[NWL];
    };
    auto fetch = [&](int s, Regs &R) {
#pragma unroll
        for (int i = 0; i < NA; i++) R.a[i] = *(const u32x4 *)(asrc[i] + s * F_BK);
#pragma unroll
        for (int i = 0; i < NWL; i++) R.w[i] = ld_w16(wsrc[i] + s * F_BK * 2);
    };
    auto stage = [&](Stage &S, const Regs &R, uint32_t neg) {
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int c = tid + 256 * i;
            *(u32x4 *)(S.a[c / (BN * 4)] + (c / 4 % BN) * F_ST + (c & 3) * 16) = R.a[i];
        }
#pragma unroll
        for (int i = 0; i < NWL; i++) {
            const int c = tid + 256 * i;
            *(u32x4 *)(S.w + (c >> 2) * F_ST + (c & 3) * 16) = R.w[i] ^ neg;
        }
    };
    facc tot[2] = {}, mid[2] = {};
    const int wrow_l[2] = {GLU ? wr * 32 + m : wr * 64 + m, GLU ? 64 + wr * 32 + m : wr * 64 + 32 + m};

    // One register set: with a second one, its loads issued two stages ahead, a stage's
    // LDS operands no longer fit beside it (203 tokens: 45 against 42 us a projection)
    Regs R;
    const int last = n_st - 1;
    fetch(0, R);
    stage(st[0], R, 0u);
    fetch(min(1, last), R);
    lds_barrier();
    for (int s = 0; s < n_st; s++) {
        const Stage &S = st[s & 1];
        if (s < last) stage(st[(s + 1) & 1], R, (s & 1) ? 0u : 0x80008000u);
        fetch(min(s + 2, last), R);
        facc acc[2] = {};
        u32x4 bw[2][2], av[2][P];
#pragma unroll
        for (int k = 0; k < 2; k++) {
#pragma unroll
            for (int r = 0; r < 2; r++) bw[k][r] = *(const u32x4 *)(S.w + wrow_l[r] * F_ST + 32 * k + 16 * h);
#pragma unroll
            for (int q = 0; q < P; q++) av[k][q] = *(const u32x4 *)(S.a[q] + (wc * 32 + m) * F_ST + 32 * k + 16 * h);
        }
#pragma unroll
        for (int q = P - 1; q >= 0; q--)  // the small parts first
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int r = 0; r < 2; r++) acc[r] = fmma<TY>(av[k][q], bw[k][r], acc[r]);
#pragma unroll
        for (int r = 0; r < 2; r++) mid[r] = (s & 1) ? mid[r] - acc[r] : mid[r] + acc[r];
        if ((s & (p.mid - 1)) == p.mid - 1 || s == last) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                tot[r] += mid[r];
                mid[r] = facc{};
            }
        }
        lds_barrier();
    }

    // ---- epilogue: the lane holds weight row wrow_l[r] of tokens 8·(v/4) + 4h + v%4 of each tile ----
    const int ld = p.ks > 1 ? p.part_ld : p.ld[sg];
    int col0 = 0;  // first column of the segment in a partial row
    if (p.ks > 1)
        for (int i = 0; i < sg; i++) col0 += p.rows[i];
    float *out = p.ks > 1 ? p.part + (size_t)ksi * p.part_stride + col0 : p.out[sg];
    const int k_lo = s_lo * F_BK, k_hi = (s_lo + n_st) * F_BK;
    auto finish = [&](int row, int t, float g, float up) {
        float y = g;
        if constexpr (GLU) y = (p.glu == 2 ? gelu_tanh_f(g) : silu_f(g)) * up;
        float *o = out + (size_t)t * ld + row;
        if (p.ks == 1 && p.epi[sg] == EPI_ADD) *o += y;
        else *o = y;
    };
    uint32_t redo = 0;
#pragma unroll
    for (int r = 0; r < (GLU ? 1 : 2); r++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int row = row0 + wrow_l[r], t = t0 + wc * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
            if (row >= rows || t >= p.n_tok) continue;
            const float sc = TY == T_F16 ? p.act.scale[t] : 1.0f;
            const float g = tot[r][v] * sc, up = GLU ? tot[1][v] * sc : 0.0f;
            if (g != g || up != up) redo |= 1u << (r * 16 + v);
            else finish(row, t, g, up);
        }
    while (redo) {
        const int i = __builtin_ctz(redo), v = i & 15;
        redo &= redo - 1;
        const int row = row0 + (i >> 4 ? wrow_l[1] : wrow_l[0]), t = t0 + wc * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
        const float sc = TY == T_F16 ? p.act.scale[t] : 1.0f;
        float y[2] = {0.0f, 0.0f};
        for (int a = 0; a < (GLU ? 2 : 1); a++) {
            const int mat = GLU ? a : sg;
            y[a] = plain_dot<TY>(p.act, (size_t)t * K, (const uint16_t *)(p.w[mat] + (size_t)row * p.rb[mat]), k_lo, k_hi, sc);
        }
        finish(row, t, y[0], y[1]);
    }
}

// out rows (= or +=) the sum of a K split's partials in split order
__global__ __launch_bounds__(256) void gemm_float_sum_kernel(FGemmP p) {
    const int c = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (c >= p.part_ld) return;
    float v = 0.0f;
    for (int k = 0; k < p.ks; k++) v += p.part[(size_t)k * p.part_stride + (size_t)t * p.part_ld + c];
    int sg = 0, r = c;
    while (r >= p.rows[sg]) r -= p.rows[sg++];
    float *o = p.out[sg] + (size_t)t * p.ld[sg] + r;
    *o = p.epi[sg] == EPI_ADD ? *o + v : v;
}

template <int TY, bool GLU>
void launch_ty(const FGemmP &p, hipStream_t st) {
    const dim3 grid(gemm_grid(p.n_rt, p.n_tt, p.ks, false));
    hipLaunchKernelGGL((gemm_float_kernel<TY, GLU>), grid, dim3(256), 0, st, p);
    if (p.ks > 1) hipLaunchKernelGGL(gemm_float_sum_kernel, dim3((p.part_ld + 255) / 256, p.n_tok), dim3(256), 0, st, p);
}

// An ungated launch of fewer than 512 workgroups splits K in up to 8 parts of at least
// 128 values, while part holds the partial sums (parts of at least 512: 9 tokens through
// two layers of hidden 960 / 1536 / 3072 take 292 / 354 / 477 us against 221 / 298 / 441).
void launch_any(FGemmP p, int ty, hipStream_t st, float *part, size_t part_cap) {
    p.n_tt = (p.n_tok + F_BN - 1) / F_BN;
    p.ks = 1;
    if (!p.glu && part) {
        p.part_ld = p.rows[0] + p.rows[1] + p.rows[2];
        p.part_stride = (size_t)p.n_tok * p.part_ld;
        while (p.ks < 8 && p.n_rt * p.n_tt * p.ks < 512 && p.K / (2 * p.ks) >= 128 && (size_t)(2 * p.ks) * p.part_stride <= part_cap) p.ks *= 2;
        p.part = part;
    }
    p.mid = p.K / p.ks >= 4096 ? 16 : 8;
    if (ty == T_BF16) p.glu ? launch_ty<T_BF16, true>(p, st) : launch_ty<T_BF16, false>(p, st);
    else p.glu ? launch_ty<T_F16, true>(p, st) : launch_ty<T_F16, false>(p, st);
}

bool weight_ok(const DevWeight &w, int ty, int K) {
    return w.ty == ty && w.cols == (size_t)K && w.data && w.rows > 0 && ((uintptr_t)w.data & 15) == 0;
}

}  // namespace

bool gemm_float_supported(int ty, size_t K) { return (ty == T_BF16 || ty == T_F16) && K % F_BK == 0 && K > 0; }

void launch_split_rows(const float *x, int ldx, const float *w, float eps, int n_rows, int E, float *xn, int ty, const ActSplit &act,
                       hipStream_t st, bool ref_order) {
    const int ro = ref_order ? 1 : 0;
    if (ty == T_BF16) hipLaunchKernelGGL(split_rows_kernel<T_BF16>, dim3(n_rows), dim3(256), 0, st, x, ldx, w, eps, E, xn, act, ro);
    else hipLaunchKernelGGL(split_rows_kernel<T_F16>, dim3(n_rows), dim3(256), 0, st, x, ldx, w, eps, E, xn, act, ro);
}

bool launch_gemm_float(const GemvSeg *segs, int nseg, const ActSplit &act, int n_tok, int K, hipStream_t st, float *part, size_t part_cap) {
    if (nseg < 1 || nseg > 3 || n_tok < 1 || !act.p[0] || !gemm_float_supported(segs[0].w.ty, K)) return false;
    FGemmP p{};
    for (int i = 0; i < nseg; i++) {
        const GemvSeg &s = segs[i];
        if (!weight_ok(s.w, segs[0].w.ty, K) || !s.out) return false;
        p.w[i] = s.w.data;
        p.rb[i] = s.w.rb();
        p.rows[i] = (int)s.w.rows;
        p.out[i] = s.out;
        p.ld[i] = s.ld;
        p.epi[i] = s.epi;
        p.n_rt += (p.rows[i] + F_BM - 1) / F_BM;
        p.rt_end[i] = p.n_rt;
    }
    p.nseg = nseg;
    p.act = act;
    p.n_tok = n_tok;
    p.K = K;
    launch_any(p, segs[0].w.ty, st, part, part_cap);
    return true;
}

bool launch_gemm_float_glu(const DevWeight &gate, const DevWeight &up, const ActSplit &act, int n_tok, int K, float *h, int ld, int gelu,
                           hipStream_t st) {
    if (n_tok < 1 || !act.p[0] || !gemm_float_supported(gate.ty, K) || !weight_ok(gate, gate.ty, K) || !weight_ok(up, gate.ty, K) ||
        gate.rows != up.rows || !h)
        return false;
    FGemmP p{};
    const DevWeight *ws[2] = {&gate, &up};
    for (int i = 0; i < 2; i++) {
        p.w[i] = ws[i]->data;
        p.rb[i] = ws[i]->rb();
        p.rows[i] = (int)ws[i]->rows;
    }
    p.out[0] = h;
    p.ld[0] = ld;
    p.epi[0] = EPI_STORE;
    p.nseg = 1;
    p.n_rt = (p.rows[0] + F_BM / 2 - 1) / (F_BM / 2);
    p.rt_end[0] = p.n_rt;
    p.glu = gelu ? 2 : 1;
    p.act = act;
    p.n_tok = n_tok;
    p.K = K;
    launch_any(p, gate.ty, st, nullptr, 0);
    return true;
}

}  // namespace rie
