// gdn_bwd_chunk.hip -- gradients of the Gated DeltaNet reference variant in chunk (WY/UT) form on the
// fp32 matrix cores.
//
// Same arithmetic as gdn_bwd.hip (the reference differentiates fast_recurrent_gated_deltanet,
// triune/kernels/fast_gla.py:781-836, with autograd).  Per 64-token chunk, with G the inclusive and
// Gp the exclusive cumulative log-decay, w = beta k, S the state entering the chunk and D the
// gradient reaching the state that leaves it:
//   Q0 = q e^G,  B0 = k e^Gp,  Wc = w e^(G_C - G)                      (every factor at most 1)
//   L[t][s] = k_t . e^(Gp_t - G_s) w_s (s < t),  A[t][s] = q_t . e^(G_t - G_s) w_s (s <= t)
//   U = (I + L)^-1 (V - B0 S),   S_next = e^G_C S + Wc^T U,   dU = A^T dO + Wc D,   dR = (I + L)^-T dU
//   D_prev = e^G_C D + Q0^T dO - B0^T dR,   dV = dR
//   dA = tril(dO U^T),  dL = -tril(dR U^T, -1)
//   dq = e^G (dO S^T) + [dA W],   dkB = -e^Gp (dR S^T) + [dL W],   dw = e^(G_C - G) (U D^T) + [dA^T Q + dL^T B]
//   dk = beta dw + dkB,   dbeta = sum_d k dw
//   dg_t = sum_{r >= t} (q dq - w dw)_r + sum_{r > t} (k dkB)_r + sum_c (D * S_next), 0 where g_t > 0
//        = sum_{r >= t} (q dq - w [.])_r + sum_{r > t} (k dkB)_r + sum_{s < t} w dw'_s + e^G_C sum_c (D * S),
//          dw' the part of dw through D
// where [.] are the in-chunk pair sums with their factors e^(G_t - G_s) (or Gp_t), formed as
// e^(G - m) e^(m - G) around the midpoint m = G_C / 2 of each key dim.
//
// S and D obey S_next = M S + N and D_prev = M^T D + K with M = e^G_C - Wc^T (I + L)^-1 B0,
// N = Wc^T (I + L)^-1 V, K = Q0^T dO - B0^T (I + L)^-T A^T dO, all known per chunk.  Three launches:
//   gdn_bwd_map_kernel   one workgroup per (b, h, chunk): L, (I + L)^-1's diagonal blocks, A, M, N, K
//   gdn_bwd_scan_kernel  one workgroup per (b, h, 16 columns, direction): S entering and D leaving
//                        every chunk, one D x D product per chunk
//   gdn_bwd_grad_kernel  one workgroup per (b, h, chunk): the gradients
// so only the scan is serial, and its step is one product.
//
// Products run on v_mfma_f32_16x16x4_f32: its operands are fp32 as they come out of the accumulators
// (nothing is rounded on the way), and a tile held in accumulator layout (lane 16 g4 + r16: rows
// 4 g4 + r of column r16) is a B operand as it stands when product r contracts rows 4 g4 + r.  With
// two bf16 parts per operand on v_mfma_f32_16x16x32_bf16 they were a fifth to a third faster (403 against
// 480 us at D = 64, 520 against 730 at D = 128, the shapes below) but carried 2^-17 into dg, which is
// a difference of sums: against 64 bits its error rose from the token-serial kernels' 2.087e-4 to
// 2.141e-4 (fp16, B = 2, T = 600, H = 4, D = 64, gate per key dim) and elements below 1 % of its rms
// lost up to eight bits (at 1e-3 to 1e-2 of it 1.6e-4 -> 4.4e-3 of their value).  In fp32 those are
// 2.087e-4 and 1.9e-4.  Solves with I + L are block substitutions with the inverses of the four diagonal
// blocks; dependent products issue back to back (32 cycles each), so the substitutions cost no more
// than products with an explicit inverse would.
//
// Measured, backward alone (bf16): B=4, H=6, T=8192, D=64, gate and beta per head 2884 us on the
// token-serial kernels, 480 here (map 165, scan 90, gradients 258); B=4, H=12, T=2048, D=128, gate per
// key dim 5834 and 727 (232, 229, 332).  The map and gradient kernels are bound by the fp32 matrix pipe
// and the chain of a chunk between its products: by counters the pipe is busy 58 and 49 % of the cycles
// at D = 64 (two workgroups per CU), 62 and 55 % at D = 128 (one), HBM moves 254 and 319 MB (1.5 and 1.2
// TB/s) and LDS is active in 15-20 %.  The scan is bound by the latency of its steps: pipe 41-42 %, 188
// and 371 MB (2.1 and 1.6 TB/s).
//
// A chunk in which some key dim decays by more than GB_SPAN nats takes its pair sums ([.], L and A) in
// two levels.  Between two 16-token tiles the decay from s to t is the rest of s's tile, the tiles
// between and t's tile up to t, all factors of at most 1.  Within a tile whose dims decay by at most
// GB_TILE the factors are e^(sum up to t) and e^-(sum up to s); a steeper tile (a reset, -inf) takes
// running products of its decays token by token.  The products with S and D use factors of at most 1
// everywhere.  With gates three times as steep, all chunks past GB_SPAN: B=4, H=12, T=8192, D=64 1019 us
// (ordinary gates 901, token-serial kernels 5036, all pair sums token by token 4320), T=1000 154 (122,
// 694, 674), B=1, H=4, T=200 50 (44, 123, 297); every tile past GB_TILE (B=4, H=6, T=8192) 771 (2881
// token-serial).
#include "chunk_common.h"

namespace triune {

namespace {

constexpr int GC = 64;            // tokens per chunk
constexpr float GB_SPAN = 128.f;  // factors within e^(+-64); a chunk of fewer tokens counts as steep pro rata
constexpr float GB_TILE = 64.f;   // the same for a tile of a steeper chunk, all on one side
constexpr float GB_GMIN = -104.f; // e^-104 is 0 in fp32: gates below it (-inf resets) act alike
constexpr int TSR = 20;           // row stride of a 16 x 16 tile in LDS (floats): rows and columns conflict-free
constexpr int TSZ = 16 * TSR;
constexpr int NTL = 10;           // lower-triangular 16 x 16 tiles of a 64 x 64 matrix

__host__ __device__ constexpr int tl(int i, int j) { return i * (i + 1) / 2 + j; }

// c + a b over 16 contracted indices: product r contracts index 4 g4 + r.
__device__ __forceinline__ f32x4 mma(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
    return c;
}

struct Lane {
    int w, g4, r16;
    __device__ __forceinline__ Lane() {
        const int l = threadIdx.x & 63;
        w = threadIdx.x >> 6;
        g4 = l >> 4;
        r16 = l & 15;
    }
};

// M, N, K, S and D in memory: 16 x 16 tiles, row tile major, each in accumulator order (lane's four
// rows of its column contiguous).  As an accumulator tile or B operand, and transposed.
__device__ __forceinline__ f32x4 mem_col(const float* m, int t, const Lane& L) {
    return *reinterpret_cast<const f32x4*>(m + t * 256 + (uint32_t)(L.g4 * 64 + L.r16 * 4));
}
__device__ __forceinline__ f32x4 mem_row(const float* m, int t, const Lane& L) {
    const float* q = m + t * 256;
    const uint32_t o = (uint32_t)((L.r16 >> 2) * 64 + L.g4 * 16 + (L.r16 & 3));
    return f32x4{q[o], q[o + 4u], q[o + 8u], q[o + 12u]};
}
__device__ __forceinline__ void mem_put(float* m, int t, const Lane& L, const f32x4& x) {
    *reinterpret_cast<f32x4*>(m + t * 256 + (uint32_t)(L.g4 * 64 + L.r16 * 4)) = x;
}

// Operand whose free index is the row of a row-major plane or tile (contracted index along the row).
__device__ __forceinline__ f32x4 row_frag(const float* p, int ld, const Lane& L) {
    return *reinterpret_cast<const f32x4*>(p + L.r16 * ld + 4 * L.g4);
}
// Operand whose free index is the column (contracted index down the rows).
__device__ __forceinline__ f32x4 col_frag(const float* p, int ld, const Lane& L) {
    const float* q = p + 4 * L.g4 * ld + L.r16;
    return f32x4{q[0], q[ld], q[2 * ld], q[3 * ld]};
}
__device__ __forceinline__ void put_tile(float* p, int ld, const Lane& L, const f32x4& x) {
#pragma unroll
    for (int r = 0; r < 4; ++r) p[(4 * L.g4 + r) * ld + L.r16] = x[r];
}
// Four consecutive 16-bit elements of an LDS row as an operand.
template <typename T>
__device__ __forceinline__ f32x4 row_frag16(const T* p, int ld, const Lane& L) {
    typedef T v4 __attribute__((ext_vector_type(4)));
    const v4 x = *reinterpret_cast<const v4*>(p + L.r16 * ld + 4 * L.g4);
    return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
}

// A chunk's rows of one 16-bit tensor: records end at the last valid row, so rows past it read as
// zero and are not written.  The range check covers the vector offset only: a partial chunk puts
// the row into it, a whole one into the scalar offset.  64 rows span less than 2^31 bytes.
struct Rows {
    __amdgpu_buffer_rsrc_t r;
    int st, lane;  // bytes
    bool whole;
};
template <typename T>
__device__ __forceinline__ Rows rows_at(const void* base, int64_t off, int64_t st, int width, int col, int nv,
                                        const Lane& L) {
    Rows x;
    x.st = (int)st * 2;
    x.lane = 4 * L.g4 * x.st + 2 * col;
    x.whole = nv == GC;
    x.r = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(reinterpret_cast<const T*>(base)) + off, (short)0,
                                            (nv - 1) * x.st + 2 * width, 0x00020000);
    return x;
}
template <typename T>
__device__ __forceinline__ float from16(uint32_t u) {
    if constexpr (std::is_same<T, __bf16>::value) return __uint_as_float(u << 16);
    else return (float)__builtin_bit_cast(_Float16, (uint16_t)u);
}
// x[i][r] = row 16 i + 4 g4 + r of the lane's column.
template <typename T>
__device__ __forceinline__ void load_rows(const Rows& a, f32x4 (&x)[4]) {
    uint32_t u[16];  // one per register: packed pairs would have to land before the next tensor's loads
    if (a.whole) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            u[e] = __builtin_amdgcn_raw_buffer_load_b16(a.r, a.lane, (16 * (e >> 2) + (e & 3)) * a.st, 0);
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            u[e] = __builtin_amdgcn_raw_buffer_load_b16(a.r, a.lane + (16 * (e >> 2) + (e & 3)) * a.st, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e >> 2][e & 3] = from16<T>(u[e]);
}
template <typename T>
__device__ __forceinline__ void store_rows(const Rows& a, const f32x4 (&x)[4]) {
    uint16_t u[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) u[e] = __builtin_bit_cast(uint16_t, (T)x[e >> 2][e & 3]);
    if (a.whole) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            __builtin_amdgcn_raw_buffer_store_b16(u[e], a.r, a.lane, (16 * (e >> 2) + (e & 3)) * a.st, 0);
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            __builtin_amdgcn_raw_buffer_store_b16(u[e], a.r, a.lane + (16 * (e >> 2) + (e & 3)) * a.st, 0, 0);
    }
}

// Sum over the four row groups, in every lane.
__device__ __forceinline__ float g4_sum(float x) { return xor_sum<32>(xor_sum<16>(x)); }

// Sums of the lane's column in accumulator layout over the 16 tokens of a tile, on top of run: inc[r]
// over tokens up to and with 4 g4 + r, exc[r] without it; the tile's total is returned.  REV: from
// the end.
template <bool REV>
__device__ __forceinline__ float scan16(const f32x4& x, float run, const Lane& L, f32x4& inc, f32x4& exc) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) s += x[r];
    const RowPair a = swap16(s);
    const RowPair b = swap32(a.lo + a.hi);
    float e = run;
    if constexpr (REV) {
        e += (L.g4 & 2) ? 0.f : b.hi;
        e += (L.g4 & 1) ? 0.f : a.hi;
    } else {
        e += (L.g4 & 2) ? b.lo : 0.f;
        e += (L.g4 & 1) ? a.lo : 0.f;
    }
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        const int r = REV ? 3 - rr : rr;
        exc[r] = e;
        e += x[r];
        inc[r] = e;
    }
    return b.lo + b.hi;
}
// The same over the chunk's four tiles: token 16 i + 4 g4 + r in [i][r].
template <bool REV>
__device__ __forceinline__ float token_scan(const f32x4 (&x)[4], const Lane& L, f32x4 (&inc)[4], f32x4 (&exc)[4]) {
    float run = 0.f;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
        const int i = REV ? 3 - ii : ii;
        run += scan16<REV>(x[i], run, L, inc[i], exc[i]);
    }
    return run;
}

// What both chunk kernels know of a chunk: its place, its gates' sums and its rows.
struct Chunk {
    int64_t b, h, c, id;  // id: (b H + h) NC + c
    int nv;
};
__device__ __forceinline__ Chunk chunk_of(const GdnChunkBwdParams& p) {
    // heads fastest: neighbouring workgroups read neighbouring rows
    const int64_t x = blockIdx.x;
    Chunk k;
    k.h = x % p.f.H;
    const int64_t y = x / p.f.H;
    k.c = y % p.nc;
    k.b = y / p.nc;
    k.id = (k.b * p.f.H + k.h) * p.nc + k.c;
    const int64_t left = p.f.T - k.c * GC;
    k.nv = left < GC ? (int)left : GC;
    return k;
}

// The gate as the recurrence takes it: min(g, 0), held at GB_GMIN.
__device__ __forceinline__ float gate_val(float g) { return fmaxf(fminf(g, 0.f), GB_GMIN); }

// Rows of the inputs: column col of head h (gate and beta per head: their one value per token).
template <typename T, int D>
__device__ __forceinline__ void load_in(const void* base, int64_t sb, int64_t st, int64_t sh, const Chunk& k, int col,
                                        const Lane& L, f32x4 (&x)[4]) {
    load_rows<T>(rows_at<T>(base, k.b * sb + k.c * GC * st + k.h * sh, st, D, col, k.nv, L), x);
}
template <typename T, int D>
__device__ __forceinline__ void load_gate(const GdnChunkBwdParams& p, const Chunk& k, int col, const Lane& L,
                                          f32x4 (&x)[4]) {
    const int64_t off = k.b * p.f.g_sb + k.c * GC * p.f.g_st + k.h * p.f.g_sh;
    load_rows<T>(rows_at<T>(p.f.g, off, p.f.g_st, p.g_head ? 1 : D, p.g_head ? 0 : col, k.nv, L), x);
    // a head gate that repeats one value over the tokens (stride 0) is in range past the last row too
    if (k.nv < GC) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (16 * (e >> 2) + 4 * L.g4 + (e & 3) >= k.nv) x[e >> 2][e & 3] = 0.f;
    }
}
template <typename T>
__device__ __forceinline__ void load_beta(const GdnChunkBwdParams& p, const Chunk& k, const Lane& L, f32x4 (&x)[4]) {
    if (p.f.beta_kind == BETA_HEAD) {
        load_in<T, 1>(p.f.beta, p.f.b_sb, p.f.b_st, p.f.b_sh, k, 0, L, x);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = f32x4{1.f, 1.f, 1.f, 1.f};
    }
}
template <typename T, int D>
__device__ __forceinline__ void load_dout(const GdnChunkBwdParams& p, const Chunk& k, int col, const Lane& L,
                                          f32x4 (&x)[4]) {
    if (p.dout) {
        load_in<T, D>(p.dout, p.do_sb, p.do_st, p.do_sh, k, col, L, x);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = zero4();
    }
}
// Rows of a contiguous [B, T, H, D] output.
template <typename T, int D>
__device__ __forceinline__ Rows out_rows(const GdnChunkBwdParams& p, void* o, const Chunk& k, int col, const Lane& L) {
    return rows_at<T>(o, ((k.b * p.f.T + k.c * GC) * p.f.H + k.h) * D, p.f.H * D, D, col, k.nv, L);
}

// X_i = T_ii (R_i - sum_{j<i} L_ij X_j), in place.  tiles: T_ii on the diagonal, -L_ij below it.
__device__ __forceinline__ void solve(const float* tiles, const Lane& L, f32x4 (&x)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f32x4 a = x[i];
#pragma unroll
        for (int j = 0; j < i; ++j) a = mma(row_frag(tiles + tl(i, j) * TSZ, TSR, L), x[j], a);
        x[i] = mma(row_frag(tiles + tl(i, i) * TSZ, TSR, L), a, zero4());
    }
}
// The same with the transpose: X_i = T_ii^T (Y_i - sum_{j>i} L_ji^T X_j).
__device__ __forceinline__ void solve_t(const float* tiles, const Lane& L, f32x4 (&x)[4]) {
#pragma unroll
    for (int i = 3; i >= 0; --i) {
        f32x4 a = x[i];
#pragma unroll
        for (int j = 3; j > i; --j) a = mma(col_frag(tiles + tl(j, i) * TSZ, TSR, L), x[j], a);
        x[i] = mma(col_frag(tiles + tl(i, i) * TSZ, TSR, L), a, zero4());
    }
}
// acc += Lt^T X for a lower-triangular Lt in tiles and a 64-row column block X.
__device__ __forceinline__ void mul_lower_t(const float* tiles, const f32x4 (&x)[4], const Lane& L, f32x4 (&acc)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = j; i < 4; ++i) acc[j] = mma(col_frag(tiles + tl(i, j) * TSZ, TSR, L), x[i], acc[j]);
}
// acc += Lt X.
__device__ __forceinline__ void mul_lower(const float* tiles, const f32x4 (&x)[4], const Lane& L, f32x4 (&acc)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) acc[i] = mma(row_frag(tiles + tl(i, j) * TSZ, TSR, L), x[j], acc[i]);
}

__device__ __forceinline__ void tile_ij(int n, int& i, int& j) {
    i = n >= 6 ? 3 : (n >= 3 ? 2 : (n >= 1 ? 1 : 0));
    j = n - tl(i, 0);
}

// x where the entry of tile (i, j) lies at least `from` below the diagonal, else 0 (from at most 2).
__device__ __forceinline__ f32x4 lower(const f32x4& x, int i, int j, int from, const Lane& L) {
    if (i - j > 1 || (i != j && from < 2)) return x;
    const int below = 16 * (i - j) + 4 * L.g4 - L.r16;
    f32x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = below + r >= from ? x[r] : 0.f;
    return y;
}
// The entries of tile (i, j) that lie `at` below the diagonal, to p[row].
__device__ __forceinline__ void put_diag(float* p, const f32x4& x, int i, int j, int at, const Lane& L) {
    const int u = L.r16 + at - 16 * (i - j);  // row of the lane's column
    if (u >= 0 && u >> 2 == L.g4) p[16 * i + u] = (u & 2) ? ((u & 1) ? x[3] : x[2]) : ((u & 1) ? x[1] : x[0]);
}

// The 2 NTL tiles between LDS (padded rows) and memory (1 KB each).  NT: threads.
template <bool OUT, int NT>
__device__ __forceinline__ void copy_tiles(float* tiles, float* mem) {
    for (int n = threadIdx.x; n < 2 * NTL * 64; n += NT) {
        f32x4* l = reinterpret_cast<f32x4*>(tiles + (n >> 6) * TSZ + ((n >> 2) & 15) * TSR + (n & 3) * 4);
        f32x4* m = reinterpret_cast<f32x4*>(mem) + n;
        if constexpr (OUT) *m = *l;
        else *l = *m;
    }
}

// ---------------------------------------------------------------------------------------
// Chunk maps
// ---------------------------------------------------------------------------------------
template <int D>
struct MapLay {
    static constexpr int NW = D / 16;
    static constexpr int LD = D + 4;  // rows 4 banks apart for row reads, 4 rows 16 banks apart for column reads
    static constexpr int PL = GC * LD;
    static constexpr int BYTES = (3 * PL + 2 * NTL * TSZ + GC + 7 * D) * 4;
};

// MFMA-bound: 416 products of 32 cycles per wave and chunk at D = 64 (2 workgroups per CU).
template <typename T, int D>
__global__ __launch_bounds__(4 * D, 2) void gdn_bwd_map_kernel(GdnChunkBwdParams p) {
    using Y = MapLay<D>;
    constexpr int NW = Y::NW, LD = Y::LD;
    __shared__ __attribute__((aligned(16))) char smem[Y::BYTES];
    float* P0 = reinterpret_cast<float*>(smem);  // Qt rows, then Q0
    float* P1 = P0 + Y::PL;                      // Bt rows, then B0
    float* P2 = P1 + Y::PL;                      // Wt rows, then Wc
    float* sL = P2 + Y::PL;                      // T_ii and -L_ij
    float* sA = sL + NTL * TSZ;                  // A
    float* sB = sA + NTL * TSZ;                  // beta (steep tiles)
    float* sC = sB + GC;                         // wide chunks: decays of tiles (see below)
    const Lane L;
    const int w = L.w, g4 = L.g4, r16 = L.r16, col = 16 * w + r16;
    const Chunk k = chunk_of(p);

    f32x4 q[4], kk[4], g[4], be[4], G[4], Gp[4];
    load_gate<T, D>(p, k, col, L, g);
    load_in<T, D>(p.f.q, p.f.q_sb, p.f.q_st, p.f.q_sh, k, col, L, q);
    load_in<T, D>(p.f.k, p.f.k_sb, p.f.k_st, p.f.k_sh, k, col, L, kk);
    load_beta<T>(p, k, L, be);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) g[i][r] = gate_val(g[i][r]);
    const float gc = token_scan<false>(g, L, G, Gp);
    const bool wide = __syncthreads_or(gc < -GB_SPAN / GC * k.nv);
    const float ec = fast_exp(gc);
    // V and dO fly until the products with them
    f32x4 v[4], dO[4];
    load_in<T, D>(p.f.v, p.f.v_sb, p.f.v_st, p.f.v_sh, k, col, L, v);
    load_dout<T, D>(p, k, col, L, dO);

    if (!wide) {
        const float m = 0.5f * gc, em = fast_exp(m);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int a = (16 * i + 4 * g4 + r) * LD + col;
                P0[a] = q[i][r] *= fast_exp(G[i][r] - m);
                P2[a] = g[i][r] = kk[i][r] * be[i][r] * fast_exp(m - G[i][r]);  // g holds the W rows from here on
                P1[a] = kk[i][r] *= fast_exp(Gp[i][r] - m);
            }
        lds_sync();
        for (int n = w; n < NTL; n += NW) {
            int i, j;
            tile_ij(n, i, j);
            f32x4 a = zero4();
#pragma unroll
            for (int kt = 0; kt < NW; ++kt)
                a = mma(row_frag(P1 + 16 * i * LD + 16 * kt, LD, L), row_frag(P2 + 16 * j * LD + 16 * kt, LD, L), a);
            put_tile(sL + n * TSZ, TSR, L, i == j ? lower(a, i, j, 1, L) : -a);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            q[i] *= em;
            kk[i] *= em;
            g[i] *= em;
        }
    } else {
        f32x4 inc[4], exc[4];
        float tot[4];
        bool steep[4], any = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            tot[i] = scan16<false>(g[i], 0.f, L, inc[i], exc[i]);
            steep[i] = __syncthreads_or(tot[i] < -GB_TILE);
            any |= steep[i];
        }
        if (any) {  // rows of q, k and the decays; a lane (two dims per lane at D = 128) per key dim
            for (int n = threadIdx.x; n < 2 * NTL * TSZ; n += 4 * D) sL[n] = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 16 * i + 4 * g4 + r;
                    P0[t * LD + col] = q[i][r];
                    P1[t * LD + col] = kk[i][r];
                    P2[t * LD + col] = fast_exp(g[i][r]);
                    if (w == 0 && r16 == 0) sB[t] = be[i][r];
                }
            lds_sync();
            const int lane = threadIdx.x & 63;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!steep[i]) continue;
                for (int s = w; s < 16; s += NW) {
                    const int rs = (16 * i + s) * LD + lane;
                    float run[D / 64], dot = 0.f;
#pragma unroll
                    for (int e = 0; e < D / 64; ++e) {
                        run[e] = sB[16 * i + s] * P1[rs + 64 * e];
                        dot += P0[rs + 64 * e] * run[e];
                    }
                    dot = g4_sum(dpp_sum16(dot));
                    if (lane == 0) sA[tl(i, i) * TSZ + s * (TSR + 1)] = dot;
                    for (int t = s + 1; t < 16; ++t) {
                        float l = 0.f, a = 0.f;
#pragma unroll
                        for (int e = 0; e < D / 64; ++e) {
                            const int o = (16 * i + t) * LD + lane + 64 * e;
                            l += P1[o] * run[e];
                            run[e] *= P2[o];
                            a += P0[o] * run[e];
                        }
                        l = g4_sum(dpp_sum16(l));
                        a = g4_sum(dpp_sum16(a));
                        if (lane == 0) {
                            sL[tl(i, i) * TSZ + t * TSR + s] = l;
                            sA[tl(i, i) * TSZ + t * TSR + s] = a;
                        }
                    }
                }
            }
            lds_sync();
        }
        // rows decayed within their tile: q and k from its start, w to its end
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int a = (16 * i + 4 * g4 + r) * LD + col;
                P0[a] = q[i][r] * fast_exp(inc[i][r]);
                P1[a] = kk[i][r] * fast_exp(exc[i][r]);
            }
            scan16<true>(g[i], 0.f, L, inc[i], exc[i]);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                P2[(16 * i + 4 * g4 + r) * LD + col] = kk[i][r] * be[i][r] * fast_exp(exc[i][r]);
        }
        if (g4 == 0) {  // what takes w's rows from their tile's end to the reference of the other row
#pragma unroll
            for (int i = 0; i < 4; ++i) sC[i * D + col] = steep[i] ? 0.f : fast_exp(-tot[i]);  // own tile: its start
            sC[4 * D + col] = fast_exp(tot[1]);  // tiles (2, 0)
            sC[5 * D + col] = fast_exp(tot[2]);  // (3, 1)
            sC[6 * D + col] = fast_exp(tot[1] + tot[2]);  // (3, 0)
        }
        token_scan<true>(g, L, inc, exc);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                q[i][r] *= fast_exp(G[i][r]);
                g[i][r] = kk[i][r] * be[i][r] * fast_exp(exc[i][r]);
                kk[i][r] *= fast_exp(Gp[i][r]);
            }
        lds_sync();
        for (int n = w; n < 2 * NTL; n += NW) {
            const bool isA = n >= NTL;
            int i, j;
            tile_ij(isA ? n - NTL : n, i, j);
            if (i == j && (i == 0 ? steep[0] : (i == 1 ? steep[1] : (i == 2 ? steep[2] : steep[3])))) continue;
            const float* pr = (isA ? P0 : P1) + 16 * i * LD;
            const float* pc = sC + (i == j ? i : (i - j == 3 ? 6 : 2 + i)) * D + 4 * g4;
            f32x4 a = zero4();
#pragma unroll
            for (int kt = 0; kt < NW; ++kt) {
                f32x4 b = row_frag(P2 + 16 * j * LD + 16 * kt, LD, L);
                if (i - j != 1) b *= *reinterpret_cast<const f32x4*>(pc + 16 * kt);
                a = mma(row_frag(pr + 16 * kt, LD, L), b, a);
            }
            put_tile(sL + n * TSZ, TSR, L, i == j ? lower(a, i, j, isA ? 0 : 1, L) : (isA ? a : -a));
        }
    }
    lds_sync();
    if (w == 0) {
        // T = (I + L_ii)^-1 of the four diagonal blocks, one column per lane: T[i] = 1[i = c] - sum L[i][k] T[k]
        float* t = sL + (g4 * (g4 + 3) / 2) * TSZ;
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float a = i == r16 ? 1.f : 0.f;
#pragma unroll
            for (int k4 = 0; k4 < i; k4 += 4) {
                const f32x4 l = *reinterpret_cast<const f32x4*>(t + i * TSR + k4);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k4 + e < i) a = fmaf(-l[e], x[k4 + e], a);
            }
            x[i] = a;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i * TSR + r16] = x[i];
    } else if (!wide) {
        for (int n = w - 1; n < NTL; n += NW - 1) {
            int i, j;
            tile_ij(n, i, j);
            f32x4 a = zero4();
#pragma unroll
            for (int kt = 0; kt < NW; ++kt)
                a = mma(row_frag(P0 + 16 * i * LD + 16 * kt, LD, L), row_frag(P2 + 16 * j * LD + 16 * kt, LD, L), a);
            put_tile(sA + n * TSZ, TSR, L, lower(a, i, j, 0, L));
        }
    }
    lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        put_tile(P0 + 16 * i * LD + 16 * w, LD, L, q[i]);
        put_tile(P1 + 16 * i * LD + 16 * w, LD, L, kk[i]);
        put_tile(P2 + 16 * i * LD + 16 * w, LD, L, g[i]);
    }
    copy_tiles<true, 4 * D>(sL, p.ws_t + k.id * (2 * NTL * 256));
    lds_sync();

    float* wm = p.ws_m + k.id * (D * D);
    float* wn = p.ws_s + k.id * (D * D);
    float* wk = p.ws_d + k.id * (D * D);
    solve(sL, L, kk);
    solve(sL, L, v);
    f32x4 z[4] = {zero4(), zero4(), zero4(), zero4()};  // -dR from A^T dO alone
    mul_lower_t(sA, dO, L, z);
    solve_t(sL, L, z);
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = -z[j];
#pragma unroll 1
    for (int rt = 0; rt < NW; ++rt) {
        f32x4 am = zero4(), an = zero4(), ak = zero4();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4 a = col_frag(P2 + 16 * i * LD + 16 * rt, LD, L);
            am = mma(a, kk[i], am);
            an = mma(a, v[i], an);
            ak = mma(col_frag(P0 + 16 * i * LD + 16 * rt, LD, L), dO[i], ak);
            ak = mma(col_frag(P1 + 16 * i * LD + 16 * rt, LD, L), z[i], ak);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) am[r] = ((rt == w && r16 == 4 * g4 + r) ? ec : 0.f) - am[r];
        mem_put(wm, rt * NW + w, L, am);
        mem_put(wn, rt * NW + w, L, an);
        mem_put(wk, rt * NW + w, L, ak);
    }
}

// ---------------------------------------------------------------------------------------
// Scan over the chunks: S_next = M S + N forwards, D_prev = M^T D + K backwards
// ---------------------------------------------------------------------------------------
// One workgroup per (b, h, direction, strip of 16 columns), one wave per 16-row tile.  A step is one
// chain: the strip's state crosses the waves through LDS (one barrier), then D / 4 MFMAs of 32 cycles
// in two chains.  The operands of the next PF chunks are in flight.  The strips of a (b, h) read the
// same maps, so its workgroups share an XCD (workgroup x runs on XCD x mod 8).
// Two column tiles per wave at D = 128, which halve what its waves read from L2, ran 2 % slower (235
// against 229 us at B = 4, H = 12, T = 2048), M stored a second time with its rows contiguous 10 %
// faster, all of which the map kernel's added stores took back.
template <int D, int PF, bool REV>
__device__ __forceinline__ void scan_walk(const GdnChunkBwdParams& p, float* sX, int64_t bh, int strip) {
    constexpr int NW = D / 16, XLD = D + 4;
    const Lane L;
    const int w = L.w;
    const int64_t DD = (int64_t)D * D, base = bh * p.nc;
    float* io = REV ? p.ws_d : p.ws_s;
    const int own = w * NW + strip;  // this wave's tile of the state
    const float* x0 = REV ? p.dsf : p.f.s0;
    const int64_t flat = bh * DD + (16 * w + 4 * L.g4) * D + 16 * strip + L.r16;
    f32x4 x = zero4();
    if (x0)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = x0[flat + r * D];
    f32x4 mf[PF][NW], yf[PF];
    auto slot = [&](int64_t n) { return base + (REV ? p.nc - 1 - n : n); };
    auto fetch = [&](int64_t n, f32x4(&m)[NW], f32x4& y) {
        const int64_t c = slot(n);
        const float* M = p.ws_m + c * DD;
#pragma unroll
        for (int kt = 0; kt < NW; ++kt) m[kt] = REV ? mem_col(M, kt * NW + w, L) : mem_row(M, w * NW + kt, L);
        y = mem_col(io + c * DD, own, L);
    };
    auto step = [&](int64_t n, const f32x4(&m)[NW], const f32x4& y) {
        mem_put(io + slot(n) * DD, own, L, x);
        float* X = sX + (n & 1) * 16 * XLD;
        *reinterpret_cast<f32x4*>(X + L.r16 * XLD + 16 * w + 4 * L.g4) = x;
        lds_sync();  // LDS only: the maps in flight need not land
        f32x4 a = y, b = zero4();
#pragma unroll
        for (int kt = 0; kt < NW; kt += 2) {
            a = mma(m[kt], row_frag(X + 16 * kt, XLD, L), a);
            b = mma(m[kt + 1], row_frag(X + 16 * (kt + 1), XLD, L), b);
        }
        x = a + b;
    };
    // every step of the main loop issues the same loads and stores, so its waits count exactly
    // (steps past the end fetch the last chunk again)
#pragma unroll
    for (int u = 0; u < PF; ++u) fetch(u < p.nc ? u : p.nc - 1, mf[u], yf[u]);
    int64_t n0 = 0;
    for (; n0 + PF <= p.nc; n0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            step(n0 + u, mf[u], yf[u]);
            const int64_t nx = n0 + u + PF;
            fetch(nx < p.nc ? nx : p.nc - 1, mf[u], yf[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < PF - 1; ++u) {
        if (n0 + u < p.nc) step(n0 + u, mf[u], yf[u]);
    }
    if (REV && p.ds0)
#pragma unroll
        for (int r = 0; r < 4; ++r) p.ds0[flat + r * D] = x[r];
}

template <int D>
__global__ __launch_bounds__(4 * D, 2) void gdn_bwd_scan_kernel(GdnChunkBwdParams p) {
    constexpr int NS = D / 16, PF = D == 128 ? 2 : 4;  // NS: strips
    __shared__ __attribute__((aligned(16))) float sX[2 * 16 * (D + 4)];
    const int64_t BH = p.f.B * p.f.H;
    const int64_t slot = blockIdx.x / 8;
    const int64_t bh = slot / (2 * NS) * 8 + blockIdx.x % 8;
    if (bh >= BH) return;
    const int s = (int)(slot % (2 * NS));
    if (s < NS) scan_walk<D, PF, false>(p, sX, bh, s);
    else scan_walk<D, PF, true>(p, sX, bh, s - NS);
}

// ---------------------------------------------------------------------------------------
// Gradients
// ---------------------------------------------------------------------------------------
template <int D>
struct GradLay {
    static constexpr int NW = D / 16;
    static constexpr int LD = D + 4;
    static constexpr int PL = GC * LD;
    static constexpr int LO = D + 8;  // 16-bit row stride of the dO plane
    static constexpr int BYTES = (2 * PL + 2 * NTL * TSZ + (2 * NW + 2) * GC + 4) * 4 + GC * LO * 2;
};

// The pair sums inside the steep tiles (bits of mask) for the lane's key dim and its tokens, from
// running products of the decays.  pq, pa, pk: the dim's column of q, decays and k in planes of 64
// rows, pbe: beta per token; the lanes of the wave that share the column have filled them.  The sums
// go to rows of D floats (oq, ob, ow: the dim's column).
template <typename T, int D>
__device__ __forceinline__ void steep_pairs(const float* pq, const float* pa, const T* pk, const float* pbe,
                                            const float* sdA, const float* sdL, int mask, const Lane& L, float* oq,
                                            float* ob, float* ow) {
    constexpr int LD = GradLay<D>::LD, LO = GradLay<D>::LO;
#pragma unroll 1
    for (int n = 0; n < 16; ++n) {
        const int i = n >> 2, t = 4 * L.g4 + (n & 3);
        if (!(mask >> i & 1)) continue;
        const float *q = pq + 16 * i * LD, *a = pa + 16 * i * LD, *be = pbe + 16 * i;
        const float *dA = sdA + tl(i, i) * TSZ, *dL = sdL + tl(i, i) * TSZ;
        const T* k = pk + 16 * i * LO;
        float rq = 1.f, rb = 1.f, sq = 0.f, sb = 0.f;  // decays over (s, t] and (s, t - 1]
#pragma unroll 4
        for (int e = 0; e < 16; ++e) {
            const int s = (t - e) & 15;
            const float w = t >= e ? be[s] * (float)k[s * LO] : 0.f, d = a[s * LD];
            sq = fmaf(dA[t * TSR + s] * w, rq, sq);
            sb = fmaf(dL[t * TSR + s] * w, rb, sb);
            rb = e ? rb * d : rb;
            rq *= d;
        }
        float rw = 1.f, sw = 0.f;
#pragma unroll 3
        for (int e = 1; e < 16; ++e) {
            const int s = (t + e) & 15;
            const float in = t + e < 16 ? rw : 0.f;
            sw = fmaf(dL[s * TSR + t] * (float)k[s * LO], in, sw);
            rw *= a[s * LD];
            sw = fmaf(dA[s * TSR + t] * q[s * LD], t + e < 16 ? rw : 0.f, sw);
        }
        const int o = (16 * i + t) * D;
        oq[o] = sq;
        ob[o] = sb;
        ow[o] = sw;
    }
}

// The gradients of one chunk (WIDE: some key dim decays by more than GB_SPAN).  The two forms part at
// the top of the kernel: one body with both branches spilled 300 registers.
template <typename T, int D, bool WIDE>
__device__ __forceinline__ void grad_chunk(const GdnChunkBwdParams& p, const Chunk& k, const Lane& L, char* smem,
                                           f32x4 (&q)[4], f32x4 (&kk)[4], f32x4 (&g)[4], const f32x4 (&be)[4],
                                           const f32x4 (&G)[4], const f32x4 (&Gp)[4], float gc, uint32_t pass) {
    using Y = GradLay<D>;
    constexpr int NW = Y::NW, LD = Y::LD, LO = Y::LO;
    float* P1 = reinterpret_cast<float*>(smem);  // B0 rows, then U
    float* P2 = P1 + Y::PL;                      // Wc rows, then dR
    float* sL = P2 + Y::PL;                      // T_ii and -L_ij, then dL (WIDE: below its subdiagonal)
    float* sA = sL + NTL * TSZ;                  // A, then dA below its diagonal
    float* red = sA + NTL * TSZ;                 // [2][NW][64] sums over each wave's key dims
    float* sD = red + 2 * NW * GC;               // dA's diagonal
    float* sE = sD + GC;                         // WIDE: dL's subdiagonal, (t, t - 1) at t
    T* sO = reinterpret_cast<T*>(sE + GC + 4);   // dO rows
    const int w = L.w, g4 = L.g4, r16 = L.r16, col = 16 * w + r16;
    f32x4 v[4], dO[4];
    load_in<T, D>(p.f.v, p.f.v_sb, p.f.v_st, p.f.v_sh, k, col, L, v);
    load_dout<T, D>(p, k, col, L, dO);
    const float m = 0.5f * gc;
    f32x4 ew[4];  // e^(G_C - G)
    if constexpr (WIDE) {
        f32x4 S[4], Se[4];
        token_scan<true>(g, L, S, Se);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) ew[i][r] = fast_exp(Se[i][r]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) ew[i][r] = fast_exp(gc - G[i][r]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 16 * i + 4 * g4 + r;
            P1[t * LD + col] = kk[i][r] * fast_exp(Gp[i][r]);
            P2[t * LD + col] = kk[i][r] * be[i][r] * ew[i][r];
            sO[t * LO + col] = (T)dO[i][r];
        }
    if (WIDE && threadIdx.x == 0) sE[0] = sE[GC] = 0.f;
    copy_tiles<false, 4 * D>(sL, p.ws_t + k.id * (2 * NTL * 256));
    lds_sync();

    const float* S = p.ws_s + k.id * (D * D);
    const float* Dn = p.ws_d + k.id * (D * D);
    // value columns [16 w, 16 w + 16): U in v, dR in z
    f32x4 z[4] = {zero4(), zero4(), zero4(), zero4()};
    mul_lower_t(sA, dO, L, z);
#pragma unroll 2
    for (int kt = 0; kt < NW; ++kt) {
        const f32x4 s = -mem_col(S, kt * NW + w, L), d = mem_col(Dn, kt * NW + w, L);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = mma(row_frag(P1 + 16 * i * LD + 16 * kt, LD, L), s, v[i]);
            z[i] = mma(row_frag(P2 + 16 * i * LD + 16 * kt, LD, L), d, z[i]);
        }
    }
    solve(sL, L, v);
    solve_t(sL, L, z);
    store_rows<T>(out_rows<T, D>(p, p.dv, k, col, L), z);
    lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        put_tile(P1 + 16 * i * LD + 16 * w, LD, L, v[i]);
        put_tile(P2 + 16 * i * LD + 16 * w, LD, L, z[i]);
    }
    lds_sync();
    for (int n = w; n < 2 * NTL; n += NW) {
        const bool isA = n < NTL;
        int i, j;
        tile_ij(isA ? n : n - NTL, i, j);
        f32x4 a = zero4();
        if (isA) {
#pragma unroll
            for (int kt = 0; kt < NW; ++kt)
                a = mma(row_frag16(sO + 16 * i * LO + 16 * kt, LO, L), row_frag(P1 + 16 * j * LD + 16 * kt, LD, L), a);
            put_tile(sA + n * TSZ, TSR, L, lower(a, i, j, 1, L));
            if (i == j) put_diag(sD, a, i, j, 0, L);
        } else {
#pragma unroll
            for (int kt = 0; kt < NW; ++kt)
                a = mma(row_frag(P2 + 16 * i * LD + 16 * kt, LD, L), row_frag(P1 + 16 * j * LD + 16 * kt, LD, L), a);
            a = -a;
            if (WIDE && i - j < 2) put_diag(sE, a, i, j, 1, L);
            put_tile(sL + (n - NTL) * TSZ, TSR, L, lower(a, i, j, WIDE ? 2 : 1, L));
        }
    }
    lds_sync();

    // key dims [16 w, 16 w + 16): products with the states first
    f32x4 aq[4], ab[4], aw[4];
    float es = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) aq[i] = ab[i] = aw[i] = zero4();
#pragma unroll 2
    for (int kt = 0; kt < NW; ++kt) {
        const f32x4 s = mem_row(S, w * NW + kt, L), d = mem_row(Dn, w * NW + kt, L);
#pragma unroll
        for (int r = 0; r < 4; ++r) es = fmaf(s[r], d[r], es);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            aq[i] = mma(row_frag16(sO + 16 * i * LO + 16 * kt, LO, L), s, aq[i]);
            ab[i] = mma(row_frag(P2 + 16 * i * LD + 16 * kt, LD, L), s, ab[i]);
            aw[i] = mma(row_frag(P1 + 16 * i * LD + 16 * kt, LD, L), d, aw[i]);
        }
    }
    es = g4_sum(es) * fast_exp(gc);  // sum over the value columns of D * e^G_C S
    f32x4 ad[4];                     // WIDE: dw through D, which joins dw at the end
    float wd = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            aq[i][r] *= fast_exp(G[i][r]);
            ab[i][r] *= -fast_exp(Gp[i][r]);
            aw[i][r] *= ew[i][r];
            if constexpr (WIDE) {
                ad[i][r] = aw[i][r];
                aw[i][r] = 0.f;
            } else {
                wd = fmaf(kk[i][r] * be[i][r], aw[i][r], wd);
            }
        }
    if constexpr (!WIDE) es += g4_sum(wd);  // ... of D * S_next

    if constexpr (!WIDE) {
        f32x4 x[4], y[4], a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) x[i][r] = kk[i][r] * be[i][r] * fast_exp(m - G[i][r]);
            a[i] = b[i] = zero4();
        }
        mul_lower(sA, x, L, a);
        mul_lower(sL, x, L, b);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float fq = fast_exp(G[i][r] - m), fb = fast_exp(Gp[i][r] - m);
                aq[i][r] = fmaf(a[i][r], fq, aq[i][r]);
                ab[i][r] = fmaf(b[i][r], fb, ab[i][r]);
                x[i][r] = q[i][r] * fq;
                y[i][r] = kk[i][r] * fb;
            }
            a[i] = zero4();
        }
        mul_lower_t(sA, x, L, a);
        mul_lower_t(sL, y, L, a);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) aw[j][r] = fmaf(a[j][r], fast_exp(m - G[j][r]), aw[j][r]);
    } else {
        __syncthreads();  // every wave is past its reads of U, dR and dO
        // a lane's rows wait in its own places of the planes
        float* X = P1 + 4 * g4 * LD + col;
        float* Y = P2 + 4 * g4 * LD + col;
        auto put = [&](float* p, int i, const f32x4& x) {
#pragma unroll
            for (int r = 0; r < 4; ++r) p[(16 * i + r) * LD] = x[r];
        };
        auto get = [&](const float* p, int i) {
            const float* q = p + 16 * i * LD;
            return f32x4{q[0], q[LD], q[2 * LD], q[3 * LD]};
        };
        float et[4], ei[4];  // decay of each tile and its inverse (0 where it is steep)
        int steep = 0;
        f32x4 inc, exc, x, y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float t = scan16<true>(g[i], 0.f, L, inc, exc);
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = kk[i][r] * be[i][r] * fast_exp(exc[r]);
            put(X, i, x);  // W to its tile's end
            const bool st = __any(t < -GB_TILE);
            steep |= st ? 1 << i : 0;
            et[i] = fast_exp(t);
            ei[i] = st ? 0.f : fast_exp(-t);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f32x4 a = zero4(), b = zero4();
#pragma unroll
            for (int j = 0; j <= i; ++j) {
                const f32x4 u = j == i ? get(X, i) * ei[i] : get(X, j);
                a = mma(row_frag(sA + tl(i, j) * TSZ, TSR, L), u, j && j < i ? a * et[j] : a);
                b = mma(row_frag(sL + tl(i, j) * TSZ, TSR, L), u, j && j < i ? b * et[j] : b);
            }
            scan16<false>(g[i], 0.f, L, inc, exc);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                aq[i][r] = fmaf(a[r], fast_exp(inc[r]), aq[i][r]);
                ab[i][r] = fmaf(b[r], fast_exp(exc[r]), ab[i][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            scan16<false>(g[i], 0.f, L, inc, exc);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[r] = q[i][r] * fast_exp(inc[r]);
                y[r] = kk[i][r] * fast_exp(exc[r]);
            }
            put(X, i, x);
            put(Y, i, y);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 a = zero4();
#pragma unroll
            for (int i = 3; i > j; --i) {
                a = mma(col_frag(sA + tl(i, j) * TSZ, TSR, L), get(X, i), i < 3 ? a * et[i] : a);
                a = mma(col_frag(sL + tl(i, j) * TSZ, TSR, L), get(Y, i), a);
            }
            // the later tiles' sums decay from this tile's end, its own from its start
            f32x4 b = mma(col_frag(sA + tl(j, j) * TSZ, TSR, L), get(X, j), zero4());
            b = mma(col_frag(sL + tl(j, j) * TSZ, TSR, L), get(Y, j), b);
            scan16<true>(g[j], 0.f, L, inc, exc);
#pragma unroll
            for (int r = 0; r < 4; ++r) aw[j][r] = fmaf(fmaf(b[r], ei[j], a[r]), fast_exp(exc[r]), aw[j][r]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (steep) {
            float* be_w = red + w * GC;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 16 * i + 4 * g4 + r;
                    P1[t * LD + col] = q[i][r];
                    P2[t * LD + col] = fast_exp(g[i][r]);
                    sO[t * LO + col] = (T)kk[i][r];
                    if (r16 == 0) be_w[t] = be[i][r];
                }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            // the chunk's M, S and D have been read: their places take the sums
            float* o0 = p.ws_m + k.id * (D * D) + col;
            float* o1 = p.ws_s + k.id * (D * D) + col;
            float* o2 = p.ws_d + k.id * (D * D) + col;
            steep_pairs<T, D>(P1 + col, P2 + col, sO + col, be_w, sA, sL, steep, L, o0, o1, o2);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (steep >> i & 1)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int o = (16 * i + 4 * g4 + r) * D;
                        aq[i][r] += o0[o];
                        ab[i][r] += o1[o];
                        aw[i][r] += o2[o];
                    }
        }
    }
    // dg_t takes what crosses t's decay: S to D, S to the tokens from t on (q dq and k dkB), the tokens
    // before t to D (w dw), and in the pair sums x = q dq - w dw and k dkB over the tokens from t on, where
    // the pairs on one side of t cancel.  A token's pair with itself (dA) is on one side of every t, and
    // joins dq and dw afterwards.  In a steep chunk most of dg is far smaller than what cancels, so there
    // a token's pair with the one before it (dL, no decay between them) joins afterwards too, and w dw
    // through D is summed up to t instead of over all tokens less those from t on.
    f32x4 y[4], inc[4], exc[4], pre[4];
    if constexpr (!WIDE) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4 d = *reinterpret_cast<const f32x4*>(sD + 16 * i + 4 * g4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float wt = kk[i][r] * be[i][r], qt = q[i][r];
                q[i][r] = qt * aq[i][r] - wt * aw[i][r];
                y[i][r] = q[i][r] + kk[i][r] * ab[i][r];
                aq[i][r] = fmaf(d[r], wt, aq[i][r]);
                aw[i][r] = fmaf(d[r], qt, aw[i][r]);
                ab[i][r] = fmaf(be[i][r], aw[i][r], ab[i][r]);
                aw[i][r] *= kk[i][r];
            }
            pre[i] = zero4();
        }
    } else {
        float wv[4], kn[4];  // w of the token before the lane's four, k of the one behind them
        float w3 = 0.f, k0 = 0.f;  // w of the last token of the tile before, k of the first one behind
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const RowPair a = swap16(kk[i][3] * be[i][3]), b = swap32(a.hi);
            wv[i] = g4 == 2 ? b.lo : (g4 ? a.lo : w3);
            w3 = b.hi;
        }
#pragma unroll
        for (int i = 3; i >= 0; --i) {
            const RowPair a = swap16(kk[i][0]), b = swap32(a.lo);
            kn[i] = g4 == 1 ? b.hi : (g4 < 3 ? a.hi : k0);
            k0 = b.lo;
        }
        f32x4 c[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = 16 * i + 4 * g4;
            const f32x4 d = *reinterpret_cast<const f32x4*>(sD + t), e = *reinterpret_cast<const f32x4*>(sE + t);
            const f32x4 en = {e[1], e[2], e[3], sE[t + 4]};
            const f32x4 k1 = {kk[i][1], kk[i][2], kk[i][3], kn[i]};
            float wp = wv[i];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float wt = kk[i][r] * be[i][r], qt = q[i][r];
                c[i][r] = wt * ad[i][r];
                q[i][r] = qt * aq[i][r] - wt * aw[i][r];
                y[i][r] = q[i][r] + kk[i][r] * ab[i][r];
                aq[i][r] = fmaf(d[r], wt, aq[i][r]);
                aw[i][r] = fmaf(d[r], qt, fmaf(en[r], k1[r], aw[i][r])) + ad[i][r];
                ab[i][r] = fmaf(be[i][r], aw[i][r], fmaf(e[r], wp, ab[i][r]));
                aw[i][r] *= kk[i][r];
                wp = wt;
            }
        }
        token_scan<false>(c, L, inc, pre);
    }
    store_rows<T>(out_rows<T, D>(p, p.dq, k, col, L), aq);
    store_rows<T>(out_rows<T, D>(p, p.dk, k, col, L), ab);
    token_scan<true>(y, L, inc, exc);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) exc[i][r] = (pass >> (4 * i + r) & 1) ? exc[i][r] + q[i][r] + (pre[i][r] + es) : 0.f;
    if (!p.g_head) store_rows<T>(out_rows<T, D>(p, p.dg, k, col, L), exc);
    const bool dbeta = p.f.beta_kind == BETA_HEAD;
    if (!p.g_head && !dbeta) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float a = dpp_sum16(exc[i][r]), b = dpp_sum16(aw[i][r]);
            const int t = 16 * i + 4 * g4 + r;
            if (r16 == 0) {
                red[w * GC + t] = a;
                red[(NW + w) * GC + t] = b;
            }
        }
    __syncthreads();
    if (threadIdx.x < 2 * GC) {
        const int t = threadIdx.x & (GC - 1), which = threadIdx.x >> 6;
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < NW; ++u) s += red[(which * NW + u) * GC + t];
        void* o = which ? (dbeta ? p.dbeta : nullptr) : (p.g_head ? p.dg : nullptr);
        const int64_t at = (k.b * p.f.T + k.c * GC + t) * p.f.H + k.h;
        if (o && t < k.nv) reinterpret_cast<T*>(o)[at] = (T)s;
    }
}

// MFMA-bound: 680 products of 32 cycles per wave and chunk at D = 64 (2 workgroups per CU).
template <typename T, int D>
__global__ __launch_bounds__(4 * D, 2) void gdn_bwd_grad_kernel(GdnChunkBwdParams p) {
    __shared__ __attribute__((aligned(16))) char smem[GradLay<D>::BYTES];
    const Lane L;
    const int col = 16 * L.w + L.r16;
    const Chunk k = chunk_of(p);
    f32x4 q[4], kk[4], g[4], be[4], G[4], Gp[4];
    load_gate<T, D>(p, k, col, L, g);
    load_in<T, D>(p.f.q, p.f.q_sb, p.f.q_st, p.f.q_sh, k, col, L, q);
    load_in<T, D>(p.f.k, p.f.k_sb, p.f.k_st, p.f.k_sh, k, col, L, kk);
    load_beta<T>(p, k, L, be);
    uint32_t pass = 0;  // tokens whose gate takes a gradient: not clamped, and not reset to 0
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (!(g[i][r] > 0.f) && g[i][r] > GB_GMIN) pass |= 1u << (4 * i + r);
            g[i][r] = gate_val(g[i][r]);
        }
    asm volatile("" : "+v"(pass));  // the bits, not the sixteen gates, stay in registers
    const float gc = token_scan<false>(g, L, G, Gp);
    const bool wide = __syncthreads_or(gc < -GB_SPAN / GC * k.nv);
    if (wide) grad_chunk<T, D, true>(p, k, L, smem, q, kk, g, be, G, Gp, gc, pass);
    else grad_chunk<T, D, false>(p, k, L, smem, q, kk, g, be, G, Gp, gc, pass);
}

template <typename T, int D>
hipError_t launch_t(const GdnChunkBwdParams& p, hipStream_t stream) {
    const unsigned chunks = (unsigned)(p.f.B * p.f.H * p.nc);
    hipError_t e;
    hipLaunchKernelGGL((gdn_bwd_map_kernel<T, D>), dim3(chunks), dim3(4 * D), 0, stream, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const unsigned pairs8 = (unsigned)((p.f.B * p.f.H + 7) / 8 * 8);
    hipLaunchKernelGGL((gdn_bwd_scan_kernel<D>), dim3(pairs8 * 2 * (D / 16)), dim3(4 * D), 0, stream, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL((gdn_bwd_grad_kernel<T, D>), dim3(chunks), dim3(4 * D), 0, stream, p);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gdn_bwd_chunk(const GdnChunkBwdParams& p, int D, hipStream_t stream) {
    if (p.f.io_dt == DT_BF16) {
        if (D == 64) return launch_t<__bf16, 64>(p, stream);
        if (D == 128) return launch_t<__bf16, 128>(p, stream);
    } else if (p.f.io_dt == DT_F16) {
        if (D == 64) return launch_t<_Float16, 64>(p, stream);
        if (D == 128) return launch_t<_Float16, 128>(p, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace triune
