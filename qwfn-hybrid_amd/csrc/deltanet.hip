// The Gated DeltaNet recurrent update of a step, with its rollback snapshots
// written by the kernel itself: the ggml_gated_delta_net of
// graph_builder::deltanet (qwfn_graph.cpp:240-278) and the state copies of
// deltanet_write_state (:208-238) in one launch.
//
// Per value head h (key head h / (n_v / n_k)) the state S [dk][dv] (dv
// contiguous) evolves token by token (the gated delta rule):
//   S = S * exp(g);  m[c] = sum_r S[r][c] k[r];  S[r][c] += k[r] (v[c] - m[c]) beta
//   out[c] = sum_r S[r][c] q[r] scale
// Columns c are independent: a workgroup takes 32 columns of one head and
// splits the 128 rows into 16 slices of 8; lane l of wave w holds column
// 32 cb + (l & 31) of slice 2 w + (l >> 5), so every state load and store of a
// wave covers two whole 128-byte row pieces. A column stays in registers for
// the whole step and the state is read and written once. The sums over r
// are finished across the two halves of the wave (permlane32 swap) and then
// across the 8 waves through LDS, in a fixed order; one barrier a token (a
// token's output sums share the next token's barrier) and one at the end. The inputs of up to DN_TC
// tokens (k and q of the key head in LDS, v, the decay and beta in registers)
// are loaded together with the state. After token T-1-s the state is also
// stored to rollback slot s-1 (s = 1 .. n_snap): the state s tokens back.
#include "qwfn_common.h"
#include "qwfn_state.h"

#include <cmath>

namespace qwfn {
namespace {

constexpr int DN_D = 128;                  // key and value head size (ssm_d_state)
constexpr int DN_COLS = 32;                // state columns per workgroup: 128 bytes of each state row
constexpr int DN_TC = 4;                   // tokens whose inputs are loaded at once
constexpr int DN_SLICES = 16;              // row slices per column
constexpr int DN_WAVES = DN_SLICES / 2;    // two slices a wave
constexpr int DN_RPS = DN_D / DN_SLICES;   // rows per lane

struct dn_args {
    const float * q;  int64_t q_ts;        // [T] x [n_k][dk], token stride in floats
    const float * k;  int64_t k_ts;
    const float * v;  int64_t v_ts;        // [T] x [n_v][dv]
    const float * g;                       // [T][n_v] log decay
    const float * beta;                    // [T][n_v]
    float *       state;                   // [n_v][dk][dv], in place
    float *       out;                     // [T][n_v][dv]
    float *       snap;                    // slot s: snap + s * snap_stride floats, [n_v][dk][dv]
    int64_t       snap_stride;
    int32_t       n_snap;
    int32_t       T, n_k, n_v, rep;
    float         scale;
};

// x plus the value of the lane 32 away (the same column, the other slice)
__device__ __forceinline__ float sum_halves(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    unsigned p = r[0], q = r[1];
    asm volatile("" : "+v"(p), "+v"(q));
    return __builtin_bit_cast(float, p) + __builtin_bit_cast(float, q);
}

static_assert(DN_COLS == 32 && DN_WAVES * 64 == DN_COLS * DN_SLICES, "a wave: 32 columns x 2 slices");

// the waves' partial sums of column cl, in a fixed order (pairs, then pairs
// of pairs)
__device__ __forceinline__ float red_sum(const float (*red)[DN_COLS], int cl) {
    float x[DN_WAVES];
#pragma unroll
    for (int i = 0; i < DN_WAVES; i++) x[i] = red[i][cl];
#pragma unroll
    for (int n = DN_WAVES; n > 1; n >>= 1)
#pragma unroll
        for (int i = 0; i < n / 2; i++) x[i] = x[2 * i] + x[2 * i + 1];
    return x[0];
}

__global__ __launch_bounds__(DN_WAVES * 64) void k_gated_delta_net(dn_args a) {
    __shared__ float4 kq[DN_TC][2][DN_D / 4];   // [token][k, q][rows / 4]
    // the waves' partial sums, two buffers each by token parity: token t's
    // output sums are read after token t + 1's first barrier (or the last one)
    __shared__ float red_m[2][DN_WAVES][DN_COLS], red_o[2][DN_WAVES][DN_COLS];
    const int h = blockIdx.x / (DN_D / DN_COLS), cb = blockIdx.x % (DN_D / DN_COLS);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int cl = lane & 31;
    const int c = cb * DN_COLS + cl;
    const int r0 = DN_RPS * (2 * w + (lane >> 5));
    float * Sg = a.state + (size_t) h * DN_D * DN_D;
    float S[DN_RPS];
#pragma unroll
    for (int i = 0; i < DN_RPS; i++) S[i] = Sg[(size_t) (r0 + i) * DN_D + c];
    const int hk = h / a.rep;
    for (int t0 = 0; t0 < a.T; t0 += DN_TC) {
        const int nt = a.T - t0 < DN_TC ? a.T - t0 : DN_TC;
        if (t0 > 0) __syncthreads();   // every lane has read the previous tokens' k and q
        for (int u = (int) threadIdx.x; u < nt * 2 * (DN_D / 4); u += DN_WAVES * 64) {
            const int tt = u / (2 * (DN_D / 4)), kqs = (u / (DN_D / 4)) & 1, e4 = u % (DN_D / 4);
            const float * src = kqs ? a.q + (int64_t) (t0 + tt) * a.q_ts : a.k + (int64_t) (t0 + tt) * a.k_ts;
            kq[tt][kqs][e4] = *(const float4 *) (src + (int64_t) hk * DN_D + 4 * e4);
        }
        float vv[DN_TC], ee[DN_TC], bb[DN_TC];
#pragma unroll
        for (int tt = 0; tt < DN_TC; tt++) {
            vv[tt] = ee[tt] = bb[tt] = 0.f;
            if (tt < nt) {
                const int64_t t = t0 + tt;
                vv[tt] = a.v[t * a.v_ts + (int64_t) h * DN_D + c];
                ee[tt] = expf(a.g[t * a.n_v + h]);
                bb[tt] = a.beta[t * a.n_v + h];
            }
        }
        __syncthreads();
#pragma unroll
        for (int tt = 0; tt < DN_TC; tt++) {
            if (tt >= nt) break;
            const int t = t0 + tt;
            float kk[DN_RPS], qq[DN_RPS];
#pragma unroll
            for (int i = 0; i < DN_RPS / 4; i++) {
                const float4 k4 = kq[tt][0][r0 / 4 + i], q4 = kq[tt][1][r0 / 4 + i];
                kk[4 * i] = k4.x; kk[4 * i + 1] = k4.y; kk[4 * i + 2] = k4.z; kk[4 * i + 3] = k4.w;
                qq[4 * i] = q4.x; qq[4 * i + 1] = q4.y; qq[4 * i + 2] = q4.z; qq[4 * i + 3] = q4.w;
            }
            const float e = ee[tt], b = bb[tt], vc = vv[tt];
            float m = 0.f;
#pragma unroll
            for (int i = 0; i < DN_RPS; i++) {
                S[i] = S[i] * e;
                m = __fmaf_rn(S[i], kk[i], m);
            }
            m = sum_halves(m);
            if (lane < 32) red_m[t & 1][w][cl] = m;
            __syncthreads();
            if (t > 0 && w == 0 && lane < 32)
                a.out[((int64_t) (t - 1) * a.n_v + h) * DN_D + c] = red_sum(red_o[(t - 1) & 1], cl);
            m = red_sum(red_m[t & 1], cl);
            const float d = (vc - m) * b;
            float o = 0.f;
#pragma unroll
            for (int i = 0; i < DN_RPS; i++) {
                S[i] = __fmaf_rn(kk[i], d, S[i]);
                o = __fmaf_rn(S[i], qq[i] * a.scale, o);
            }
            o = sum_halves(o);
            if (lane < 32) red_o[t & 1][w][cl] = o;
            const int sb = a.T - 1 - t;
            if (sb >= 1 && sb <= a.n_snap) {
                float * sp = a.snap + (sb - 1) * a.snap_stride + (size_t) h * DN_D * DN_D;
#pragma unroll
                for (int i = 0; i < DN_RPS; i++) __builtin_nontemporal_store(S[i], &sp[(size_t) (r0 + i) * DN_D + c]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < DN_RPS; i++) __builtin_nontemporal_store(S[i], &Sg[(size_t) (r0 + i) * DN_D + c]);
    __syncthreads();
    if (w == 0 && lane < 32)
        a.out[((int64_t) (a.T - 1) * a.n_v + h) * DN_D + c] = red_sum(red_o[(a.T - 1) & 1], cl);
}

// ---------------------------------------------------------------- many tokens
//
// The same rule for chunks of 16 tokens, as matrix products on the f32 matrix
// cores (v_mfma_f32_16x16x4_f32): the chunkwise (WY) form of the gated delta rule. With e_t = exp(g_t), D_ij = e_{j+1} .. e_i
// (j <= i), c_i = e_0 .. e_i within the chunk and S0 the state before it:
//   d    = (I + A)^-1 b (v - c (K S0)),  A_ij = b_i D_ij (k_i . k_j) for j < i
//   out  = scale (c (Q S0) + (D o QK^T) d)        (D o QK^T: j <= i only)
//   S    = c_15 S0 + sum_j D_15,j k_j d_j^T
//
// A workgroup of 8 waves takes 32 columns of one head: wave w the 16 columns
// 16 (w & 1) .. and the 32 rows 32 (w >> 1) .. . Its part of the state stays
// in 8 registers in the accumulator layout of the MFMA (lane l: column l & 15,
// rows 4 (l >> 4) + r of each 16-row tile), which is also the B operand of
// K S0 and Q S0 when the rows of a tile are summed in the order r, l >> 4: no
// data moves between the products. The row quarters' partial sums meet in LDS,
// one barrier a chunk. k, q and v of a group of DC_CHUNKS chunks lie in LDS
// (the next group's are on the way into registers meanwhile), and what does not
// depend on the state, (I + A)^-1 and D o QK^T, is made for the whole group
// first, two waves a chunk; (I + A)^-1 by forward substitution, one column a
// lane. The decays enter as running products, never as quotients or
// exponentials of differences, so that a decay of 0 (g = -inf) stays exact.
//
// A column whose d turns non-finite at token i (a non-finite input, a state that
// overflowed, a d that overflows) is not finite from token i on in the
// recurrence; a product with the zeros of the triangular matrices would carry
// that into earlier tokens, so the right-hand sides and the solved d of such
// tokens enter the products as 0 and the column is set to NaN from i on.
//
// Rounding: with isotropic keys the error against float64 is the token form's or
// less (T 512 5.9e-7 for 6.2e-7); with keys and queries around one direction and
// beta near 1, c (Q S0) and (D o QK^T) d cancel and the outputs' is larger: mean
// cosine 0.74 2.8e-7 for 0.75e-7 at T 16, 3.3e-7 for 1.7e-7 at T 256 (the state's
// 2.1e-7 for 1.3e-7, 5.85e-7 for 5.9e-7). The matrices' sums, P and the output in
// double bring 1.8e-7 and 2.4e-7 for 3.5% of the time; not kept.
//
// What bounds it: the token-by-token kernel is a chain of T steps of 0.68 us (a
// barrier and two cross-wave sums each); here a group of 64 tokens takes 8.6 us,
// of it about 4 us of f32 matrix work a SIMD (304 MFMAs of 32 cycles), the rest
// the matrices' serial part (decays, inverse) and each chunk's exchange of
// partial sums. 48 heads, T 512: 348 -> 72 us (T 64: 44 -> 12). Measured on the
// way there: 4 waves a block (one a SIMD) 104 us; the operands loaded from L2
// in every chunk instead of LDS 86 us; the next group's matrices made between
// the current chunks' products 90 us (the extra registers and loads cost more
// than the overlap gave).
constexpr int DC_C      = 16;              // tokens of a chunk
constexpr int DC_CHUNKS = 4;               // chunks of a group
constexpr int DC_TOK    = DC_C * DC_CHUNKS;
constexpr int DC_KS     = DN_D + 4;        // row stride of k and q in LDS (floats): the operand reads meet no bank twice
constexpr int DC_VS     = DN_COLS + 4;     // of v
constexpr int DC_MS     = 20;              // of a 16x16 matrix
constexpr int DC_WAVES  = 8;               // two a SIMD: one wave alone issues at half rate
constexpr int DC_THREADS = DC_WAVES * 64;
constexpr int DC_QUARTERS = DC_WAVES / 2;  // row quarters of a head
constexpr int DC_TILES  = DN_D / 16 / DC_QUARTERS;   // 16-row tiles of a wave's 32 rows
constexpr int DC_LD4    = DC_TOK * DN_D / 4 / DC_THREADS;    // float4 of k (and of q) a thread brings in
constexpr int DC_LDV    = DC_TOK * DN_COLS / DC_THREADS;     // values of v
// Fewer tokens take the token-by-token kernel. At 48 heads in a HIP graph it takes 6.9 / 8.1 / 9.2 / 11.5 us
// at T 8 / 10 / 12 / 16, one chunk 7.1 .. 7.3 us; at T 9 and 10 the chunk's error against float64 is 1%
// larger (state 9.3e-8 against 9.2e-8), from 12 on no larger.
constexpr int DC_MIN_T  = 12;
static_assert(DC_WAVES == 2 * DC_CHUNKS, "the group's matrices: two waves a chunk");
static_assert(DC_TILES == 2, "the partial sums of a wave: two chains in each of two tiles");

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct dc_mats {
    float tinv[DC_C * DC_MS];   // A, then (I + A)^-1
    float p[DC_C * DC_MS];      // scale D o QK^T
    float c[DC_C], cs[DC_C], dend[DC_C];   // c_i, scale c_i, D_15,i
};

struct dc_lds {
    float   k[DC_TOK][DC_KS], q[DC_TOK][DC_KS], v[DC_TOK][DC_VS];
    float   e[DC_TOK], b[DC_TOK];                       // exp(g), beta; past the sequence 1 and 0
    dc_mats mats[DC_CHUNKS];
    f32x4   xm[2][DC_WAVES][64];                        // K S0 of a wave's rows: [chunk parity][wave][lane]
    f32x4   xo[DC_CHUNKS][DC_WAVES][64];                // Q S0: [chunk][wave][lane]
};
static_assert(sizeof(dc_lds) <= 160 * 1024, "LDS of a CU");

struct dc_regs {                // a thread's part of a group's inputs on their way to LDS
    f32x4 k[DC_LD4], q[DC_LD4];
    float v[DC_LDV], g, b;
};

__device__ __forceinline__ f32x4 mfma4(float x, float y, f32x4 z) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, z, 0, 0, 0);
}

// every wave's LDS accesses are done and visible to the block; loads from global memory stay in flight
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Part j of the inputs of the group at token t0; a token past the sequence reads the last one's (beta 0
// makes its d 0, and nothing else of it is used).
__device__ __forceinline__ void dc_load(const dn_args & a, const float * kh, const float * qh, const float * vh,
                                        const float * gh, const float * bh, int t0, int j, dc_regs & x) {
    const int u = (int) threadIdx.x + DC_THREADS * j;
    const int t = t0 + (u >> 5) < a.T ? t0 + (u >> 5) : a.T - 1;
    x.k[j] = *(const f32x4 *) (kh + t * a.k_ts);
    x.q[j] = *(const f32x4 *) (qh + t * a.q_ts);
    x.v[j] = vh[t * a.v_ts];
    if (j == 0) {
        const int64_t tg = t0 + ((int) threadIdx.x & (DC_TOK - 1)) < a.T ? t0 + ((int) threadIdx.x & (DC_TOK - 1)) : a.T - 1;
        x.g = gh[tg * a.n_v];
        x.b = bh[tg * a.n_v];
    }
}
static_assert(DC_LD4 == DC_CHUNKS && DC_LDV == DC_CHUNKS, "a part of the next group's loads in each step");
static_assert(DN_D / 4 == 32 && DN_COLS == 32, "a token's row of k, q and v: 32 lanes");

__device__ __forceinline__ void dc_store(const dn_args & a, int t0, const dc_regs & x, dc_lds & sm) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < DC_LD4; j++) {
        const int u = tid + DC_THREADS * j;
        *(f32x4 *) &sm.k[u >> 5][4 * (u & 31)] = x.k[j];
        *(f32x4 *) &sm.q[u >> 5][4 * (u & 31)] = x.q[j];
    }
#pragma unroll
    for (int j = 0; j < DC_LDV; j++) {
        const int u = tid + DC_THREADS * j;
        sm.v[u >> 5][u & 31] = x.v[j];
    }
    if (tid < DC_TOK) {
        const bool in = t0 + tid < a.T;
        sm.e[tid] = in ? expf(x.g) : 1.f;
        sm.b[tid] = in ? x.b : 0.f;
    }
}

// The matrices of chunk c of the group: A and its decays (what 0) or scale D o QK^T (what 1).
__device__ __forceinline__ void dc_matrices(int c, int what, int m, int g, float scale, dc_lds & sm) {
    dc_mats & o = sm.mats[c];
    const float (*k)[DC_KS] = sm.k + DC_C * c, (*l)[DC_KS] = what ? sm.q + DC_C * c : k;
    // two products a chain, then pairs: the error of a sum grows with its longest chain
    f32x4 x[DN_D / 8];
#pragma unroll
    for (int i = 0; i < DN_D / 16; i++) {
        const f32x4 kv = *(const f32x4 *) &k[m][16 * i + 4 * g], lv = *(const f32x4 *) &l[m][16 * i + 4 * g];
        x[2 * i] = x[2 * i + 1] = f32x4{};
#pragma unroll
        for (int r = 0; r < 4; r++) x[2 * i + (r >> 1)] = mfma4(lv[r], kv[r], x[2 * i + (r >> 1)]);
    }
#pragma unroll
    for (int n = DN_D / 8; n > 1; n >>= 1)
#pragma unroll
        for (int i = 0; i < n / 2; i++) x[i] = x[2 * i] + x[2 * i + 1];
    asm volatile("" : "+v"(m), "+v"(g));       // the lane masks are made here, not kept over the main loop
    f32x4 e[4];
#pragma unroll
    for (int i = 0; i < 4; i++) e[i] = *(const f32x4 *) &sm.e[DC_C * c + 4 * i];
    // lane (j = m, g): rows i = 4 g + r of column j; pr runs over D_sj, cr over c_s, with the
    // output's scale for D o QK^T (in double: up to 17 factors, rounded once)
    double pr = what ? scale : 1., cr = pr;
    float cm = 1.f, D[4];
#pragma unroll
    for (int s = 0; s < DC_C; s++) {
        const double es = e[s >> 2][s & 3];
        cr = cr * es;
        if (s > m) pr = pr * es;
        if (s == m) cm = (float) cr;
        if ((s >> 2) == g) D[s & 3] = (float) pr;
    }
    if (what == 0) {
        const f32x4 bi = *(const f32x4 *) &sm.b[DC_C * c + 4 * g];
        o.c[m] = cm;
        o.dend[m] = (float) pr;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 4 * g + r;
            float A = i > m && bi[r] != 0.f ? bi[r] * (D[r] * x[0][r]) : 0.f;
            if (!__builtin_isfinite(A)) {      // token i's d is not finite; the products stay finite
                A = 0.f;
                sm.b[DC_C * c + i] = __builtin_nanf("");
            }
            o.tinv[i * DC_MS + m] = A;
        }
    } else {
        o.cs[m] = cm;
#pragma unroll
        for (int r = 0; r < 4; r++) o.p[(4 * g + r) * DC_MS + m] = 4 * g + r >= m ? D[r] * x[0][r] : 0.f;
    }
}

// A -> (I + A)^-1 in place. B, the inverse of the two 8x8 diagonal blocks, by forward substitution (column
// m, its block's rows; T_i = [i == m] - sum_{j < i} A_ij T_j); then with A21 the block below them
// (B^-1 + A21)^-1 = B - B A21 B.
__device__ __forceinline__ void dc_invert(float * tinv, int m, int g) {
    asm volatile("" : "+v"(m), "+v"(g));
    constexpr int H = DC_C / 2;
    const int h0 = m & H;                      // the block's first row
    f32x4 row[H][2], low;                      // its rows of A; A21's row m (rows H .., columns 0 .. H - 1)
#pragma unroll
    for (int i = 0; i < H; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) row[i][j] = *(const f32x4 *) (tinv + (h0 + i) * DC_MS + h0 + 4 * j);
    low = *(const f32x4 *) (tinv + m * DC_MS + 4 * g);
    float t[H];
#pragma unroll
    for (int i = 0; i < H; i++) {
        float x = i == (m & (H - 1)) ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; j++) x = __fmaf_rn(-row[i][j >> 2][j & 3], t[j], x);
        t[i] = i < (m & (H - 1)) ? 0.f : x;
    }
#pragma unroll
    for (int i = 0; i < H; i++) {
        tinv[(h0 + i) * DC_MS + m] = t[i];
        tinv[((h0 ^ H) + i) * DC_MS + m] = 0.f;
    }
    const f32x4 bm = *(const f32x4 *) (tinv + m * DC_MS + 4 * g);
    f32x4 bc, y = {}, z = {};
#pragma unroll
    for (int r = 0; r < 4; r++) bc[r] = tinv[(4 * g + r) * DC_MS + m];
#pragma unroll
    for (int r = 0; r < 4; r++) y = mfma4(m >= H && g < 2 ? low[r] : 0.f, bc[r], y);
#pragma unroll
    for (int r = 0; r < 4; r++) z = mfma4(bm[r], y[r], z);
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (4 * g + r >= H && m < H) tinv[(4 * g + r) * DC_MS + m] = -z[r];
}

// The first token of the lane's column whose x (tokens 4 g + r) is not finite, or `first` if that is
// earlier; x is 0 from there on.
__device__ __forceinline__ int dc_cut(f32x4 & x, int first, int g) {
#pragma unroll
    for (int r = 3; r >= 0; r--)
        if (!__builtin_isfinite(x[r]) && 4 * g + r < first) first = 4 * g + r;
    for (int o = 16; o < 64; o <<= 1) {
        const int z = __shfl_xor(first, o);
        first = z < first ? z : first;
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (4 * g + r >= first) x[r] = 0.f;
    return first;
}

__global__ __launch_bounds__(DC_THREADS, 2) void k_gated_delta_chunks(dn_args a) {
    __shared__ dc_lds sm;
    // the blocks of a key head read the same k and q: consecutive heads on one XCD
    int blk = blockIdx.x;
    if (gridDim.x % 8 == 0) blk = (blk % 8) * (int) (gridDim.x / 8) + blk / 8;
    const int h = blk / (DN_D / DN_COLS), cb = blk % (DN_D / DN_COLS);
    const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), quarter = w >> 1, ct = w & 1;
    const int c0 = cb * DN_COLS + 16 * ct, row0 = 16 * DC_TILES * quarter;
    const int hk = h / a.rep;
    // the thread's columns of the group's loads
    const int l32 = (int) threadIdx.x & 31;
    const float * kh = a.k + (int64_t) hk * DN_D + 4 * l32, * qh = a.q + (int64_t) hk * DN_D + 4 * l32;
    const float * vh = a.v + (int64_t) h * DN_D + cb * DN_COLS + l32, * gh = a.g + h, * bh = a.beta + h;
    dc_regs x;
#pragma unroll
    for (int j = 0; j < DC_CHUNKS; j++) dc_load(a, kh, qh, vh, gh, bh, 0, j, x);
    float * Sg = a.state + (size_t) h * DN_D * DN_D + (size_t) (row0 + 4 * g) * DN_D + c0 + m;
    f32x4 S[DC_TILES];
#pragma unroll
    for (int i = 0; i < DC_TILES; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) S[i][r] = Sg[(size_t) (16 * i + r) * DN_D];
    float * ob = a.out + (int64_t) h * DN_D + c0 + m;
    const int64_t ots = (int64_t) a.n_v * DN_D;
    // the d of the chunk whose output is the wave's, and its first non-finite token in the column
    f32x4 Uf = {};
    int ff = DC_C;
    // out of chunk `quarter` of the group at token t0, one chunk and 16 columns a wave
    auto finish = [&](int t0) {
        const dc_mats & mt = sm.mats[quarter];
        const f32x4 (*xo)[64] = sm.xo[quarter];
        const f32x4 pr = *(const f32x4 *) (mt.p + m * DC_MS + 4 * g), cs = *(const f32x4 *) (mt.cs + 4 * g);
        f32x4 o = ((xo[ct][lane] + xo[ct + 2][lane]) + (xo[ct + 4][lane] + xo[ct + 6][lane])) * cs;
#pragma unroll
        for (int r = 0; r < 4; r++) o = mfma4(pr[r], Uf[r], o);
        const int t = t0 + DC_C * quarter + 4 * g;
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (t + r < a.T) ob[(t + r) * ots] = 4 * g + r < ff ? o[r] : __builtin_nanf("");
    };
    static_assert(DC_QUARTERS == DC_CHUNKS, "finish: one chunk of a group a quarter");
    // a chunk's operands in this wave: lane (m, g): token m, rows 16 i + 4 g + r of k and q
    f32x4 kx[DC_TILES], qx[DC_TILES];
    auto operands = [&](int c) {
#pragma unroll
        for (int i = 0; i < DC_TILES; i++) {
            kx[i] = *(const f32x4 *) &sm.k[DC_C * c + m][row0 + 16 * i + 4 * g];
            qx[i] = *(const f32x4 *) &sm.q[DC_C * c + m][row0 + 16 * i + 4 * g];
        }
    };
    // chunk c of the group at token t0; part c of the next group's loads
    auto step = [&](int t0, int c) {
        const dc_mats & mt = sm.mats[c];
        // two products a chain, then pairs: the error of a sum grows with its longest chain
        f32x4 kt[DC_TILES], Mt[2 * DC_TILES] = {}, Ot[2 * DC_TILES] = {};
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < DC_TILES; i++) Mt[2 * i + (r >> 1)] = mfma4(kx[i][r], S[i][r], Mt[2 * i + (r >> 1)]);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < DC_TILES; i++) kt[i][r] = sm.k[DC_C * c + 4 * g + r][row0 + 16 * i + m];
        f32x4 (*xm)[64] = sm.xm[c & 1];
        const f32x4 tr = *(const f32x4 *) (mt.tinv + m * DC_MS + 4 * g);
        const f32x4 cc = *(const f32x4 *) (mt.c + 4 * g), dd = *(const f32x4 *) (mt.dend + 4 * g);
        const f32x4 bb = *(const f32x4 *) &sm.b[DC_C * c + 4 * g];
        const float cend = mt.c[DC_C - 1];
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = sm.v[DC_C * c + 4 * g + r][16 * ct + m];
        xm[w][lane] = (Mt[0] + Mt[1]) + (Mt[2] + Mt[3]);
        lds_barrier();
        const f32x4 M0 = xm[ct][lane], M1 = xm[ct + 2][lane], M2 = xm[ct + 4][lane], M3 = xm[ct + 6][lane];
        // Q S0 runs under the exchange
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < DC_TILES; i++) Ot[2 * i + (r >> 1)] = mfma4(qx[i][r], S[i][r], Ot[2 * i + (r >> 1)]);
        const f32x4 M = (M0 + M1) + (M2 + M3);
        f32x4 R, U = {};
#pragma unroll
        for (int r = 0; r < 4; r++) R[r] = __fmaf_rn(-cc[r], M[r], v[r]) * bb[r];
#pragma unroll
        for (int r = 0; r < 4; r++) U = mfma4(tr[r], R[r], U);
        // T_ii = 1, so a token whose R is not finite has no finite U either: one test for both
        bool bad = false;
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= !__builtin_isfinite(U[r]);
        int first = DC_C;
        if (__builtin_expect(__ballot(bad) != 0, 0)) {
            first = dc_cut(R, first, g);
            U = f32x4{};
#pragma unroll
            for (int r = 0; r < 4; r++) U = mfma4(tr[r], R[r], U);
            first = dc_cut(U, first, g);
        }
        if (quarter == c) { Uf = U; ff = first; }
#pragma unroll
        for (int i = 0; i < DC_TILES; i++) S[i] = S[i] * cend;
        const f32x4 Ud = U * dd;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < DC_TILES; i++) S[i] = mfma4(kt[i][r], Ud[r], S[i]);
        // issued under the products of the update
        if (c < DC_CHUNKS - 1) operands(c + 1);
        dc_load(a, kh, qh, vh, gh, bh, t0 + DC_TOK, c, x);
        sm.xo[c][w][lane] = (Ot[0] + Ot[1]) + (Ot[2] + Ot[3]);
        if (first < DC_C) {
#pragma unroll
            for (int i = 0; i < DC_TILES; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) S[i][r] = __builtin_nanf("");
        }
    };
    for (int t0 = 0; t0 < a.T; t0 += DC_TOK) {
        const int nc = a.T - t0 < DC_TOK ? (a.T - t0 + DC_C - 1) / DC_C : DC_CHUNKS;
        dc_store(a, t0, x, sm);
        lds_barrier();
        // waves 0 .. 3 (one a SIMD) the inverses, waves 4 .. 7 D o QK^T
        if ((w & (DC_CHUNKS - 1)) < nc) {
            dc_matrices(w & (DC_CHUNKS - 1), w / DC_CHUNKS, m, g, a.scale, sm);
            if (w < DC_CHUNKS) dc_invert(sm.mats[w].tinv, m, g);
        }
        lds_barrier();
        operands(0);
#pragma unroll
        for (int c = 0; c < DC_CHUNKS; c++)
            if (c < nc) step(t0, c);
        lds_barrier();          // the partials of Q S0; every wave is done with the group's k, q and v
        if (quarter < nc) finish(t0);   // reads mats and xo, which are written after the next group's first barrier
    }
#pragma unroll
    for (int i = 0; i < DC_TILES; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) __builtin_nontemporal_store(S[i][r], &Sg[(size_t) (16 * i + r) * DN_D]);
}

}  // namespace
}  // namespace qwfn

using namespace qwfn;

extern "C" int qwfn_gated_delta_net(const float * q, int64_t q_token_stride, const float * k, int64_t k_token_stride,
                                    const float * v, int64_t v_token_stride, const float * g, const float * beta,
                                    int32_t T, int32_t n_k_heads, int32_t n_v_heads, int32_t head_dim, float scale,
                                    float * state, float * out, float * snap, size_t snap_stride_bytes, int32_t n_snap,
                                    void * stream) {
    return ::qwfn::abi_call("gated_delta_net", [&]() -> int {
        if (!q || !k || !v || !g || !beta || !state || !out) return set_error(QWFN_EINVAL, "gated_delta_net: NULL pointer");
        if (head_dim != DN_D) return set_error(QWFN_ENOTSUP, "gated_delta_net: head_dim must be 128");
        if (T < 1 || n_k_heads < 1 || n_v_heads < 1 || n_v_heads % n_k_heads)
            return set_error(QWFN_EINVAL, "gated_delta_net: T >= 1 and n_v_heads a multiple of n_k_heads");
        if (q_token_stride < (int64_t) n_k_heads * DN_D || k_token_stride < (int64_t) n_k_heads * DN_D ||
            v_token_stride < (int64_t) n_v_heads * DN_D)
            return set_error(QWFN_EINVAL, "gated_delta_net: token strides shorter than a token's heads");
        if (n_snap < 0 || n_snap > T - 1) return set_error(QWFN_EINVAL, "gated_delta_net: n_snap must lie in [0, T-1]");
        const size_t state_bytes = (size_t) n_v_heads * DN_D * DN_D * sizeof(float);
        if (n_snap > 0 && (!snap || snap_stride_bytes < state_bytes || snap_stride_bytes % 4))
            return set_error(QWFN_EINVAL, "gated_delta_net: snapshot slots must hold the state (stride a multiple of 4)");
        if (!is_aligned(q, 16) || !is_aligned(k, 16) || q_token_stride % 4 || k_token_stride % 4 || !is_aligned(v, 4) ||
            !is_aligned(g, 4) || !is_aligned(beta, 4) || !is_aligned(state, 4) || !is_aligned(out, 4) ||
            (snap && !is_aligned(snap, 4)))
            return set_error(QWFN_EALIGN, "gated_delta_net: q, k 16-byte aligned (token strides multiples of 4), the rest 4");
        dn_args a{};
        a.q = q; a.q_ts = q_token_stride; a.k = k; a.k_ts = k_token_stride; a.v = v; a.v_ts = v_token_stride;
        a.g = g; a.beta = beta; a.state = state; a.out = out;
        a.snap = snap; a.snap_stride = (int64_t) (snap_stride_bytes / sizeof(float)); a.n_snap = n_snap;
        a.T = T; a.n_k = n_k_heads; a.n_v = n_v_heads; a.rep = n_v_heads / n_k_heads; a.scale = scale;
        const unsigned blocks = (unsigned) n_v_heads * (DN_D / DN_COLS);
        // the tokens before the snapshots' and the last one's, in chunks
        const int32_t Tc = n_snap > 0 ? T - n_snap - 1 : T;
        if (Tc >= DC_MIN_T) {
            a.T = Tc;
            hipLaunchKernelGGL(k_gated_delta_chunks, dim3(blocks), dim3(DC_WAVES * 64), 0, as_stream(stream), a);
            if (int rc = hip_check(hipGetLastError(), "gated_delta_net launch")) return rc;
            if (Tc == T) return QWFN_OK;
            a.T = T - Tc;
            a.q += Tc * a.q_ts; a.k += Tc * a.k_ts; a.v += Tc * a.v_ts;
            a.g += (int64_t) Tc * n_v_heads; a.beta += (int64_t) Tc * n_v_heads; a.out += (int64_t) Tc * n_v_heads * DN_D;
        }
        hipLaunchKernelGGL(k_gated_delta_net, dim3(blocks), dim3(DN_WAVES * 64), 0, as_stream(stream), a);
        return hip_check(hipGetLastError(), "gated_delta_net launch");
    });
}
