// gdn_bwd_chunk.hip -- gradients of the Gated DeltaNet reference variant in chunk (WY/UT) form on the
// matrix cores.
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
// Products run on v_mfma_f32_16x16x32_bf16 with both operands split into two bf16 parts (three MFMAs
// per product, bf16 rows of dO as they are), as in the forward kernels: every gradient is rounded to
// 16 bits, 2^-9 or 2^-12, far above the split's 2^-17.  A tile held in accumulator layout (lane 16 g4
// + r16: rows 4 g4 + r of column r16) is half of a B operand, and half of the A operand of its
// transpose, without moving lanes.  The solves with I + L are block substitutions with the inverses
// of the four diagonal blocks.
//
// Measured, forward and backward together (bf16): B=4, H=6, T=8192, D=64, gate and beta per head
// 3054 -> 494 us; B=4, H=12, T=2048, D=128, gate per key dim 5923 -> 737 us, against the token-serial
// kernels.  Of that, when the split products came in, the map kernel 118 / 156 us, the scan 89 / 158,
// the gradients 176 / 216; on the fp32 MFMA (a quarter of the K per pass, no splitting) they took
// 156 / 220, 106 / 211, 253 / 319.
// What bounds them now is the traffic of M, N, K, S and D: 16 D^2 bytes per chunk written and read
// by the scan, 300 / 600 MB of it at 3.4-3.8 TB/s.
//
// A chunk in which some key dim decays by more than GB_SPAN nats forms its pair sums from running
// products of the decays instead (L and A in the map kernel, [.] in the gradient kernel); the
// products with S and D use factors of at most 1 everywhere.
#include "chunk_common.h"

namespace triune {

namespace {

constexpr int GC = 64;            // tokens per chunk
constexpr float GB_SPAN = 128.f;  // factors within e^(+-64)
constexpr float GB_GMIN = -104.f; // e^-104 is 0 in fp32: gates below it (-inf resets) act alike
constexpr int TSR = 20;           // row stride of a 16 x 16 tile in LDS (elements)
constexpr int TSZ = 16 * TSR;     // a tile's fp32 elements, or its two bf16 parts' TSZ each
constexpr int TLB = TSZ * 4;      // bytes of a tile, either way
constexpr int NTL = 10;           // lower-triangular 16 x 16 tiles of a 64 x 64 matrix

__host__ __device__ constexpr int tl(int i, int j) { return i * (i + 1) / 2 + j; }

struct Lane {
    int w, g4, r16;
    __device__ __forceinline__ Lane() {
        const int l = threadIdx.x & 63;
        w = threadIdx.x >> 6;
        g4 = l >> 4;
        r16 = l & 15;
    }
};

// N, K, S and D in memory: 16 x 16 tiles, row tile major, each in accumulator order (lane's four
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

// M and M^T in memory as the scan's A operands: operand f = row tile * NKS + K step, its two bf16
// parts of 64 lanes x 8 slots each.  The four values x of a tile go to slots 4 half .. 4 half + 3.
__device__ __forceinline__ void mem_put_half(float* m, int f, int half, const f32x4& x) {
    float r[4] = {x[0], x[1], x[2], x[3]};
    uint32_t w[2][2];
    split_pairs<2, 2>(r, w);
    uint2* p = reinterpret_cast<uint2*>(m) + (uint32_t)(f * 256 + (threadIdx.x & 63) * 2 + half);
    p[0] = uint2{w[0][0], w[0][1]};
    p[128] = uint2{w[1][0], w[1][1]};
}
__device__ __forceinline__ Split8<2> mem_operand(const float* m, int f) {
    const uint4* p = reinterpret_cast<const uint4*>(m) + (uint32_t)(f * 128 + (threadIdx.x & 63));
    Split8<2> a;
    a.p[0] = __builtin_bit_cast(bf16x8, p[0]);
    a.p[1] = __builtin_bit_cast(bf16x8, p[64]);
    return a;
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
__device__ __forceinline__ float from16(uint16_t u) {
    if constexpr (std::is_same<T, __bf16>::value) return __uint_as_float((uint32_t)u << 16);
    else return (float)__builtin_bit_cast(_Float16, u);
}
// x[i][r] = row 16 i + 4 g4 + r of the lane's column.
template <typename T>
__device__ __forceinline__ void load_rows(const Rows& a, f32x4 (&x)[4]) {
    uint16_t u[16];
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

// ---- operands in bf16 parts ---------------------------------------------------------------
// A K = 32 operand covers two 16-wide blocks: K slots 0..3 of a lane are rows 4 g4 + r of the first
// block, 4..7 those of the second (as lds_frag and lds_frag_tr of chunk_common.h read them).
__device__ __forceinline__ Split8<2> split_pair(const f32x4& lo, const f32x4& hi) {
    const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return split8<2>(x);
}
// Three products of two split operands (two where a is bf16 as it stands).
template <int NA>
__device__ __forceinline__ f32x4 mms(const Split8<NA>& a, const Split8<2>& b, const f32x4& c) {
    return mfma_split<NA, 2, 2>(a, b, c);
}

// Column block x (accumulator layout) of rows row0 + [0, 16) and column col into NP planes.
template <int NP, int D>
__device__ __forceinline__ void put_col(char* base, int row0, int col, const Lane& L, const f32x4& x) {
    using PL = Plane<D>;
    float r[4] = {x[0], x[1], x[2], x[3]};
    uint32_t w[NP][2];
    split_pairs<NP, 2>(r, w);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = 4 * L.g4 + e;
        uint16_t* p = reinterpret_cast<uint16_t*>(base) + (row0 + row) * PL::RS + PL::unit(col & ~3, PL::swz(row)) + (col & 3);
#pragma unroll
        for (int pl = 0; pl < NP; ++pl) p[pl * (PL::BYTES / 2)] = (uint16_t)(w[pl][e >> 1] >> (16 * (e & 1)));
    }
}

// Lower-triangular tiles in two bf16 parts: part n of tile t at t * TLB + n * TLB / 2, rows TSR apart.
__device__ __forceinline__ void put_ltile(char* tiles, int t, const Lane& L, const f32x4& x) {
    float r[4] = {x[0], x[1], x[2], x[3]};
    uint32_t w[2][2];
    split_pairs<2, 2>(r, w);
    uint16_t* p = reinterpret_cast<uint16_t*>(tiles + t * TLB) + 4 * L.g4 * TSR + L.r16;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int pl = 0; pl < 2; ++pl) p[pl * TSZ + e * TSR] = (uint16_t)(w[pl][e >> 1] >> (16 * (e & 1)));
}
__device__ __forceinline__ bf16x4 tile_row(const char* tiles, int t, int part, const Lane& L) {
    return *reinterpret_cast<const bf16x4*>(reinterpret_cast<const __bf16*>(tiles + t * TLB + part * (TLB / 2)) +
                                            L.r16 * TSR + 4 * L.g4);
}
__device__ __forceinline__ bf16x4 tile_col(const char* tiles, int t, int part, const Lane& L) {
    return lds_read_tr(reinterpret_cast<const __bf16*>(tiles + t * TLB + part * (TLB / 2)) +
                       (4 * L.g4 + (L.r16 >> 2)) * TSR + 4 * (L.r16 & 3));
}
// Operand over tiles t0 (K slots 0..3) and t1 (4..7); a negative index stands for a zero tile.
// TR: the tiles' transposes.
template <bool TR>
__device__ __forceinline__ Split8<2> tile_frag(const char* tiles, int t0, int t1, const Lane& L) {
    Split8<2> f;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        bf16x4 a = {}, b = {};
        if (t0 >= 0) a = TR ? tile_col(tiles, t0, n, L) : tile_row(tiles, t0, n, L);
        if (t1 >= 0) b = TR ? tile_col(tiles, t1, n, L) : tile_row(tiles, t1, n, L);
        f.p[n] = bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    }
    return f;
}
// Element (row, col) of the lower-triangular matrix.
__device__ __forceinline__ float tile_at(const char* tiles, int row, int col) {
    const __bf16* p = reinterpret_cast<const __bf16*>(tiles + tl(row >> 4, col >> 4) * TLB) + (row & 15) * TSR + (col & 15);
    return (float)p[0] + (float)p[TSZ];
}
__device__ __forceinline__ int lower_index(int i, int j) { return i >= j ? tl(i, j) : -1; }

// X <- Lt X (or Lt^T X) for a lower-triangular Lt in tiles and a 64-row column block X given as the
// two K = 32 operands b: acc[i] += ...
template <bool TR>
__device__ __forceinline__ void mul_lower(const char* tiles, const Split8<2> (&b)[2], const Lane& L, f32x4 (&acc)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            if (TR ? ks < i / 2 : ks > i / 2) continue;
            const int t0 = TR ? lower_index(2 * ks, i) : lower_index(i, 2 * ks);
            const int t1 = TR ? lower_index(2 * ks + 1, i) : lower_index(i, 2 * ks + 1);
            acc[i] = mms(tile_frag<TR>(tiles, t0, t1, L), b[ks], acc[i]);
        }
}
// The same for rows of 16-bit elements known to fit NX bf16 parts.
template <int NX>
__device__ __forceinline__ void mul_lower_x(const char* tiles, const Split8<NX> (&b)[2], const Lane& L, f32x4 (&acc)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int ks = i / 2; ks < 2; ++ks)
            acc[i] = mfma_split<2, NX, 2>(
                tile_frag<true>(tiles, lower_index(2 * ks, i), lower_index(2 * ks + 1, i), L), b[ks], acc[i]);
}
template <int NX>
__device__ __forceinline__ Split8<NX> split_pair_x(const f32x4& lo, const f32x4& hi) {
    const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return split8<NX>(x);
}

// Sum over the four row groups, in every lane.
__device__ __forceinline__ float g4_sum(float x) { return xor_sum<32>(xor_sum<16>(x)); }

// Sums over the chunk's tokens of the lane's column in accumulator layout: inc[i][r] over tokens up
// to and with 16 i + 4 g4 + r, exc[i][r] without it; the total is returned.  REV: from the end.
template <bool REV>
__device__ __forceinline__ float token_scan(const f32x4 (&x)[4], const Lane& L, f32x4 (&inc)[4], f32x4 (&exc)[4]) {
    float run = 0.f;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
        const int i = REV ? 3 - ii : ii;
        float s = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) s += x[i][r];
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
            exc[i][r] = e;
            e += x[i][r];
            inc[i][r] = e;
        }
        run += b.lo + b.hi;
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

// X_i = T_ii (R_i - sum_{j<i} L_ij X_j), in place (TR: with the transpose, X_i = T_ii^T (R_i -
// sum_{j>i} L_ji^T X_j)).  tiles: T_ii on the diagonal, -L_ij below it.
template <bool TR>
__device__ __forceinline__ void solve(const char* tiles, const Lane& L, f32x4 (&x)[4]) {
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
        const int i = TR ? 3 - ii : ii;
        f32x4 a = x[i];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            // blocks 2 ks and 2 ks + 1 that are already solved
            const bool u0 = TR ? 2 * ks > i : 2 * ks < i, u1 = TR ? 2 * ks + 1 > i : 2 * ks + 1 < i;
            if (!u0 && !u1) continue;
            const int t0 = u0 ? (TR ? tl(2 * ks, i) : tl(i, 2 * ks)) : -1;
            const int t1 = u1 ? (TR ? tl(2 * ks + 1, i) : tl(i, 2 * ks + 1)) : -1;
            a = mms(tile_frag<TR>(tiles, t0, t1, L),
                    split_pair(u0 ? x[2 * ks] : zero4(), u1 ? x[2 * ks + 1] : zero4()), a);
        }
        x[i] = mms(tile_frag<TR>(tiles, tl(i, i), -1, L), split_pair(a, zero4()), zero4());
    }
}

__device__ __forceinline__ void tile_ij(int n, int& i, int& j) {
    i = n >= 6 ? 3 : (n >= 3 ? 2 : (n >= 1 ? 1 : 0));
    j = n - tl(i, 0);
}

// x where the tile entry lies below (or, with diag, on) the diagonal of tile (i, j), else 0.
__device__ __forceinline__ f32x4 lower(const f32x4& x, bool on_diag, bool with_diag, const Lane& L) {
    if (!on_diag) return x;
    f32x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int t = 4 * L.g4 + r;
        y[r] = (t > L.r16 || (with_diag && t == L.r16)) ? x[r] : 0.f;
    }
    return y;
}

// The 2 NTL split tiles between LDS (padded rows) and memory (1 KB each).  NT: threads.
template <bool OUT, int NT>
__device__ __forceinline__ void copy_tiles(char* tiles, float* mem) {
    for (int n = threadIdx.x; n < 2 * NTL * 64; n += NT) {
        uint2* l = reinterpret_cast<uint2*>(tiles + (n >> 6) * TLB + ((n >> 5) & 1) * (TLB / 2) +
                                            ((n >> 1) & 15) * (TSR * 2) + (n & 1) * 16);
        uint4* m = reinterpret_cast<uint4*>(mem) + n;
        if constexpr (OUT) {
            *m = uint4{l[0].x, l[0].y, l[1].x, l[1].y};
        } else {
            const uint4 u = *m;
            l[0] = uint2{u.x, u.y};
            l[1] = uint2{u.z, u.w};
        }
    }
}

// ---------------------------------------------------------------------------------------
// Chunk maps
// ---------------------------------------------------------------------------------------
template <int D>
struct MapLay {
    static constexpr int NW = D / 16;
    static constexpr int ROWP = Plane<D>::BYTES;
    static constexpr int BYTES = 3 * 2 * ROWP + 2 * NTL * TLB + GC * 4;
};

// Element (t, s) of a lower-triangular matrix into the split tiles (wide chunks).
__device__ __forceinline__ void put_at(char* tiles, int t, int s, float x) {
    __bf16* p = reinterpret_cast<__bf16*>(tiles + tl(t >> 4, s >> 4) * TLB) + (t & 15) * TSR + (s & 15);
    p[0] = (__bf16)x;
    p[TSZ] = (__bf16)(x - (float)p[0]);
}

template <typename T, int D>
__global__ __launch_bounds__(4 * D, 2) void gdn_bwd_map_kernel(GdnChunkBwdParams p) {
    using Y = MapLay<D>;
    using PL = Plane<D>;
    constexpr int NW = Y::NW, NKS = D / 32, NX = Prec<T>::NX;
    __shared__ __attribute__((aligned(16))) char smem[Y::BYTES];
    char* P0 = smem;                   // Qt rows, then Q0
    char* P1 = P0 + 2 * Y::ROWP;       // Bt rows, then B0
    char* P2 = P1 + 2 * Y::ROWP;       // Wt rows, then Wc
    char* sL = P2 + 2 * Y::ROWP;       // T_ii and -L_ij (L_ii in fp32 until it is inverted)
    char* sA = sL + NTL * TLB;         // A
    float* sB = reinterpret_cast<float*>(sA + NTL * TLB);  // beta (wide chunks)
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
    const bool wide = __syncthreads_or(gc < -GB_SPAN);
    const float ec = fast_exp(gc);
    // V and dO fly until the products with them
    f32x4 v[4], dO[4];
    load_in<T, D>(p.f.v, p.f.v_sb, p.f.v_st, p.f.v_sh, k, col, L, v);
    load_dout<T, D>(p, k, col, L, dO);

    if (!wide) {
        const float m = 0.5f * gc, em = fast_exp(m);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                q[i][r] *= fast_exp(G[i][r] - m);
                g[i][r] = kk[i][r] * be[i][r] * fast_exp(m - G[i][r]);  // g holds the W rows from here on
                kk[i][r] *= fast_exp(Gp[i][r] - m);
            }
            put_col<2, D>(P0, 16 * i, col, L, q[i]);
            put_col<2, D>(P1, 16 * i, col, L, kk[i]);
            put_col<2, D>(P2, 16 * i, col, L, g[i]);
        }
        lds_sync();
        for (int n = w; n < NTL; n += NW) {
            int i, j;
            tile_ij(n, i, j);
            f32x4 a = zero4();
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
                a = mms(PL::template frag<2>(P1, 16 * i, r16, ks, g4),
                        PL::template frag<2>(P2, 16 * j, r16, ks, g4), a);
            if (i == j) {
                a = lower(a, true, false, L);
                float* t = reinterpret_cast<float*>(sL + n * TLB) + 4 * g4 * TSR + r16;
#pragma unroll
                for (int r = 0; r < 4; ++r) t[r * TSR] = a[r];
            } else {
                put_ltile(sL, n, L, -a);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            q[i] *= em;
            kk[i] *= em;
            g[i] *= em;
        }
    } else {
        // rows of q, k and the decays in fp32; L and A from running products of the decays, a lane
        // (pair of lanes' elements at D = 128) per key dim
        constexpr int LD = D;
        float* F0 = reinterpret_cast<float*>(P0);
        float* F1 = reinterpret_cast<float*>(P1);
        float* F2 = reinterpret_cast<float*>(P2);
        for (int n = threadIdx.x; n < 2 * NTL * TSZ; n += 4 * D) reinterpret_cast<uint32_t*>(sL)[n] = 0u;
        f32x4 S[4], Se[4];
        token_scan<true>(g, L, S, Se);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = 16 * i + 4 * g4 + r;
                F0[t * LD + col] = q[i][r];
                F1[t * LD + col] = kk[i][r];
                F2[t * LD + col] = fast_exp(g[i][r]);
                if (w == 0 && r16 == 0) sB[t] = be[i][r];
                q[i][r] *= fast_exp(G[i][r]);
                g[i][r] = kk[i][r] * be[i][r] * fast_exp(Se[i][r]);
                kk[i][r] *= fast_exp(Gp[i][r]);
            }
        __syncthreads();
        const int lane = threadIdx.x & 63;
        for (int s = w; s < GC; s += NW) {
            float run[D / 64], dot = 0.f;
#pragma unroll
            for (int e = 0; e < D / 64; ++e) {
                run[e] = sB[s] * F1[s * LD + lane + 64 * e];
                dot += F0[s * LD + lane + 64 * e] * run[e];
            }
            dot = g4_sum(dpp_sum16(dot));
            if (lane == 0) put_at(sA, s, s, dot);
            for (int t = s + 1; t < GC; ++t) {
                float l = 0.f, a = 0.f;
#pragma unroll
                for (int e = 0; e < D / 64; ++e) {
                    const int o = t * LD + lane + 64 * e;
                    l += F1[o] * run[e];
                    run[e] *= F2[o];
                    a += F0[o] * run[e];
                }
                l = g4_sum(dpp_sum16(l));
                a = g4_sum(dpp_sum16(a));
                if (lane == 0) {
                    put_at(sA, t, s, a);
                    if ((t >> 4) == (s >> 4))
                        reinterpret_cast<float*>(sL + tl(t >> 4, s >> 4) * TLB)[(t & 15) * TSR + (s & 15)] = l;
                    else
                        put_at(sL, t, s, -l);
                }
            }
        }
    }
    lds_sync();
    if (w == 0) {
        // T = (I + L_ii)^-1 of the four diagonal blocks, one column per lane: T[i] = 1[i = c] - sum L[i][k] T[k]
        char* tile = sL + (g4 * (g4 + 3) / 2) * TLB;
        const float* t = reinterpret_cast<const float*>(tile);
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
        asm volatile("" ::: "memory");  // the parts take the place of the fp32 tile just read
        __bf16* o = reinterpret_cast<__bf16*>(tile) + r16;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const __bf16 h = (__bf16)x[i];
            o[i * TSR] = h;
            o[TSZ + i * TSR] = (__bf16)(x[i] - (float)h);
        }
    } else if (!wide) {
        for (int n = w - 1; n < NTL; n += NW - 1) {
            int i, j;
            tile_ij(n, i, j);
            f32x4 a = zero4();
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
                a = mms(PL::template frag<2>(P0, 16 * i, r16, ks, g4),
                        PL::template frag<2>(P2, 16 * j, r16, ks, g4), a);
            put_ltile(sA, n, L, lower(a, i == j, true, L));
        }
    }
    lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        put_col<2, D>(P0, 16 * i, col, L, q[i]);
        put_col<2, D>(P1, 16 * i, col, L, kk[i]);
        put_col<2, D>(P2, 16 * i, col, L, g[i]);
    }
    copy_tiles<true, 4 * D>(sL, p.ws_t + k.id * (2 * NTL * 256));
    lds_sync();

    float* wm = p.ws_m + k.id * (2 * D * D);  // M, then M^T
    float* wn = p.ws_s + k.id * (D * D);
    float* wk = p.ws_d + k.id * (D * D);
    solve<false>(sL, L, kk);
    solve<false>(sL, L, v);
    const Split8<NX> ds[2] = {split_pair_x<NX>(dO[0], dO[1]), split_pair_x<NX>(dO[2], dO[3])};
    f32x4 z[4] = {zero4(), zero4(), zero4(), zero4()};  // -dR from A^T dO alone
    mul_lower_x<NX>(sA, ds, L, z);
    solve<true>(sL, L, z);
    const Split8<2> xs[2] = {split_pair(kk[0], kk[1]), split_pair(kk[2], kk[3])};
    const Split8<2> vs[2] = {split_pair(v[0], v[1]), split_pair(v[2], v[3])};
    const Split8<2> zs[2] = {split_pair(-z[0], -z[1]), split_pair(-z[2], -z[3])};
#pragma unroll 1
    for (int rt = 0; rt < NW; ++rt) {
        f32x4 am = zero4(), at = zero4(), an = zero4(), ak = zero4();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const Split8<2> a = PL::template frag_tr<2>(P2, 32 * ks, rt, g4, r16);
            am = mms(a, xs[ks], am);
            at = mms(xs[ks], a, at);  // the same tile transposed
            an = mms(a, vs[ks], an);
            ak = mfma_split<2, NX, 2>(PL::template frag_tr<2>(P0, 32 * ks, rt, g4, r16), ds[ks], ak);
            ak = mms(PL::template frag_tr<2>(P1, 32 * ks, rt, g4, r16), zs[ks], ak);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float e = (rt == w && r16 == 4 * g4 + r) ? ec : 0.f;
            am[r] = e - am[r];
            at[r] = e - at[r];
        }
        mem_put_half(wm, rt * NKS + w / 2, w & 1, at);
        mem_put_half(wm + D * D, w * NKS + rt / 2, rt & 1, am);
        mem_put(wn, rt * NW + w, L, an);
        mem_put(wk, rt * NW + w, L, ak);
    }
}

// ---------------------------------------------------------------------------------------
// Scan over the chunks: S_next = M S + N forwards, D_prev = M^T D + K backwards
// ---------------------------------------------------------------------------------------
// One workgroup per (b, h, direction, strip of CT * 16 columns), one wave per 16-row tile.  A step is
// one chain: the strip's state, split into bf16 parts, crosses the waves through LDS (one barrier),
// then 3 D / 32 MFMAs.  The operands of the next PF chunks are in flight.  The strips of a (b, h)
// read the same maps, so its workgroups share an XCD (workgroup x runs on XCD x mod 8); at D = 128
// two column tiles per wave halve what they read from its L2.
template <int D, int CT, int PF, bool REV>
__device__ __forceinline__ void scan_walk(const GdnChunkBwdParams& p, char* sX, int64_t bh, int strip) {
    constexpr int NW = D / 16, NKS = D / 32, XB = NKS * 2048;  // bytes of a column tile's operands
    const Lane L;
    const int w = L.w, lane = threadIdx.x & 63;
    const int64_t DD = (int64_t)D * D, base = bh * p.nc;
    float* io = REV ? p.ws_d : p.ws_s;
    const int own = w * NW + strip * CT;  // this wave's first tile of the state
    const float* x0 = REV ? p.dsf : p.f.s0;
    const int64_t flat = bh * DD + (16 * w + 4 * L.g4) * D + 16 * strip * CT + L.r16;
    f32x4 x[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        x[c] = zero4();
        if (x0)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[c][r] = x0[flat + r * D + 16 * c];
    }
    Split8<2> mf[PF][NKS];
    f32x4 yf[PF][CT];
    auto slot = [&](int64_t n) { return base + (REV ? p.nc - 1 - n : n); };
    auto fetch = [&](int64_t n, Split8<2>(&m)[NKS], f32x4(&y)[CT]) {
        const int64_t c = slot(n);
        const float* M = p.ws_m + c * 2 * DD + (REV ? DD : 0);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) m[ks] = mem_operand(M, w * NKS + ks);
#pragma unroll
        for (int t = 0; t < CT; ++t) y[t] = mem_col(io + c * DD, own + t, L);
    };
    auto step = [&](int64_t n, const Split8<2>(&m)[NKS], const f32x4(&y)[CT]) {
        char* X = sX + (n & 1) * CT * XB;
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            mem_put(io + slot(n) * DD, own + t, L, x[t]);
            float r[4] = {x[t][0], x[t][1], x[t][2], x[t][3]};
            uint32_t u[2][2];
            split_pairs<2, 2>(r, u);
#pragma unroll
            for (int pl = 0; pl < 2; ++pl)
                *reinterpret_cast<uint2*>(X + t * XB + ((w >> 1) * 2 + pl) * 1024 + lane * 16 + (w & 1) * 8) =
                    uint2{u[pl][0], u[pl][1]};
        }
        lds_sync();  // LDS only: the maps in flight need not land
        f32x4 a[CT][NKS];
        Split8<2> b[CT][NKS];
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                a[t][ks] = ks ? zero4() : y[t];
#pragma unroll
                for (int pl = 0; pl < 2; ++pl)
                    b[t][ks].p[pl] = *reinterpret_cast<const bf16x8*>(X + t * XB + (ks * 2 + pl) * 1024 + lane * 16);
            }
        // CT * NKS independent chains of three
#pragma unroll
        for (int e = 0; e < 3; ++e)
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks)
                    a[t][ks] = mfma(m[ks].p[e == 2], b[t][ks].p[e == 1], a[t][ks]);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            x[t] = a[t][0] + a[t][1];
            if constexpr (NKS == 4) x[t] += a[t][2] + a[t][3];
        }
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
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) p.ds0[flat + r * D + 16 * c] = x[c][r];
}

template <int D>
struct ScanPlan {
    static constexpr int CT = D == 128 ? 2 : 1, PF = D == 128 ? 2 : 4, NS = D / 16 / CT;  // NS: strips
};
template <int D>
__global__ __launch_bounds__(4 * D, 2) void gdn_bwd_scan_kernel(GdnChunkBwdParams p) {
    using P = ScanPlan<D>;
    __shared__ __attribute__((aligned(16))) char sX[2 * P::CT * (D / 32) * 2048];
    const int64_t BH = p.f.B * p.f.H;
    const int64_t slot = blockIdx.x / 8;
    const int64_t bh = slot / (2 * P::NS) * 8 + blockIdx.x % 8;
    if (bh >= BH) return;
    const int s = (int)(slot % (2 * P::NS));
    if (s < P::NS) scan_walk<D, P::CT, P::PF, false>(p, sX, bh, s);
    else scan_walk<D, P::CT, P::PF, true>(p, sX, bh, s - P::NS);
}

// ---------------------------------------------------------------------------------------
// Gradients
// ---------------------------------------------------------------------------------------
template <int D, int NX>
struct GradLay {
    static constexpr int NW = D / 16;
    static constexpr int ROWP = Plane<D>::BYTES;
    static constexpr int BYTES = (2 * 2 + NX) * ROWP + 2 * NTL * TLB + 2 * NW * GC * 4;
};

// The pair sums of a wide chunk for the lane's key dim and its 16 tokens: running products of the
// decays from each token outwards, with the other tokens' rows read again from memory.  pq and pb
// go to rows of two LDS planes, pw to rows of D floats in memory (the lane's own elements).
template <typename T, int D, int LD>
__device__ __forceinline__ void wide_pairs(const GdnChunkBwdParams& p, const Chunk& k, int col, const char* sdA,
                                        const char* sdL, float* pq, float* pb, float* pw) {
    const Lane L;
    auto row0 = [&](const void* x, int64_t sb, int64_t st, int64_t sh, int c) {
        return reinterpret_cast<const T*>(x) + k.b * sb + k.c * GC * st + k.h * sh + c;
    };
    const T* q = row0(p.f.q, p.f.q_sb, p.f.q_st, p.f.q_sh, col);
    const T* kr = row0(p.f.k, p.f.k_sb, p.f.k_st, p.f.k_sh, col);
    const T* gr = row0(p.f.g, p.f.g_sb, p.f.g_st, p.f.g_sh, p.g_head ? 0 : col);
    const T* br = row0(p.f.beta, p.f.b_sb, p.f.b_st, p.f.b_sh, 0);
    auto decay = [&](int t) { return fast_exp(gate_val((float)gr[t * p.f.g_st])); };
    auto wrow = [&](int t) {
        const float b = p.f.beta_kind == BETA_HEAD ? (float)br[t * p.f.b_st] : 1.f;
        return b * (float)kr[t * p.f.k_st];
    };
#pragma unroll 1
    for (int e = 0; e < 16; ++e) {
        const int t = 16 * (e >> 2) + 4 * L.g4 + (e & 3);
        float aq = 0.f, ab = 0.f, aw = 0.f;
        if (t < k.nv) {
            float rq = 1.f, rb = 1.f;  // products of the decays over (s, t] and (s, t - 1]
#pragma unroll 1
            for (int s = t; s >= 0; --s) {
                const float ws = wrow(s), a = decay(s);
                aq += tile_at(sdA, t, s) * ws * rq;
                if (s < t) {
                    ab += tile_at(sdL, t, s) * ws * rb;
                    rb *= a;
                }
                rq *= a;
            }
            float rw = 1.f;
            aw = tile_at(sdA, t, t) * (float)q[t * p.f.q_st];
#pragma unroll 1
            for (int s = t + 1; s < k.nv; ++s) {
                aw += tile_at(sdL, s, t) * (float)kr[s * p.f.k_st] * rw;
                rw *= decay(s);
                aw += tile_at(sdA, s, t) * (float)q[s * p.f.q_st] * rw;
            }
        }
        pq[t * LD + col] = aq;
        pb[t * LD + col] = ab;
        pw[t * D + col] = aw;
    }
}

template <typename T, int D>
__global__ __launch_bounds__(4 * D, 2) void gdn_bwd_grad_kernel(GdnChunkBwdParams p) {
    constexpr int NX = Prec<T>::NX;
    using Y = GradLay<D, NX>;
    using PL = Plane<D>;
    constexpr int NW = Y::NW, NKS = D / 32;
    __shared__ __attribute__((aligned(16))) char smem[Y::BYTES];
    char* P1 = smem;                  // B0 rows, then U
    char* P2 = P1 + 2 * Y::ROWP;      // Wc rows, then dR
    char* sO = P2 + 2 * Y::ROWP;      // dO rows
    char* sL = sO + NX * Y::ROWP;     // T_ii and -L_ij, then dL
    char* sA = sL + NTL * TLB;        // A, then dA
    float* red = reinterpret_cast<float*>(sA + NTL * TLB);  // [2][NW][64] sums over each wave's key dims
    const Lane L;
    const int w = L.w, g4 = L.g4, r16 = L.r16, col = 16 * w + r16;
    const Chunk k = chunk_of(p);

    f32x4 q[4], kk[4], g[4], be[4], G[4], Gp[4];
    load_gate<T, D>(p, k, col, L, g);
    load_in<T, D>(p.f.q, p.f.q_sb, p.f.q_st, p.f.q_sh, k, col, L, q);
    load_in<T, D>(p.f.k, p.f.k_sb, p.f.k_st, p.f.k_sh, k, col, L, kk);
    load_beta<T>(p, k, L, be);
    f32x4 v[4], dO[4];
    load_in<T, D>(p.f.v, p.f.v_sb, p.f.v_st, p.f.v_sh, k, col, L, v);
    load_dout<T, D>(p, k, col, L, dO);
    uint32_t pass = 0;  // tokens whose gate takes a gradient: not clamped, and not reset to 0
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (!(g[i][r] > 0.f) && g[i][r] > GB_GMIN) pass |= 1u << (4 * i + r);
            g[i][r] = gate_val(g[i][r]);
        }
    const float gc = token_scan<false>(g, L, G, Gp);
    const bool wide = __syncthreads_or(gc < -GB_SPAN);
    const float m = wide ? 0.f : 0.5f * gc;
    f32x4 ew[4];  // e^(G_C - G)
    if (wide) {
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
    for (int i = 0; i < 4; ++i) {
        f32x4 b0, wc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            b0[r] = kk[i][r] * fast_exp(Gp[i][r]);
            wc[r] = kk[i][r] * be[i][r] * ew[i][r];
        }
        put_col<2, D>(P1, 16 * i, col, L, b0);
        put_col<2, D>(P2, 16 * i, col, L, wc);
        put_col<NX, D>(sO, 16 * i, col, L, dO[i]);
    }
    copy_tiles<false, 4 * D>(sL, p.ws_t + k.id * (2 * NTL * 256));
    lds_sync();

    const float* S = p.ws_s + k.id * (D * D);
    const float* Dn = p.ws_d + k.id * (D * D);
    // value columns [16 w, 16 w + 16): U in v, dR in z
    f32x4 z[4] = {zero4(), zero4(), zero4(), zero4()};
    {
        const Split8<NX> ds[2] = {split_pair_x<NX>(dO[0], dO[1]), split_pair_x<NX>(dO[2], dO[3])};
        mul_lower_x<NX>(sA, ds, L, z);
    }
#pragma unroll 1
    for (int ks = 0; ks < NKS; ++ks) {
        const int o = 2 * ks * NW + w;
        const Split8<2> s = split_pair(-mem_col(S, o, L), -mem_col(S, o + NW, L));
        const Split8<2> d = split_pair(mem_col(Dn, o, L), mem_col(Dn, o + NW, L));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = mms(PL::template frag<2>(P1, 16 * i, r16, ks, g4), s, v[i]);
            z[i] = mms(PL::template frag<2>(P2, 16 * i, r16, ks, g4), d, z[i]);
        }
    }
    solve<false>(sL, L, v);
    solve<true>(sL, L, z);
    store_rows<T>(out_rows<T, D>(p, p.dv, k, col, L), z);
    lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        put_col<2, D>(P1, 16 * i, col, L, v[i]);
        put_col<2, D>(P2, 16 * i, col, L, z[i]);
    }
    lds_sync();
    for (int n = w; n < 2 * NTL; n += NW) {
        const bool isA = n < NTL;
        int i, j;
        tile_ij(isA ? n : n - NTL, i, j);
        f32x4 a = zero4();
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const Split8<2> u = PL::template frag<2>(P1, 16 * j, r16, ks, g4);
            if (isA) a = mms(PL::template frag<NX>(sO, 16 * i, r16, ks, g4), u, a);
            else a = mms(PL::template frag<2>(P2, 16 * i, r16, ks, g4), u, a);
        }
        if (isA) put_ltile(sA, n, L, lower(a, i == j, true, L));
        else put_ltile(sL, n - NTL, L, -lower(a, i == j, false, L));
    }
    lds_sync();

    // key dims [16 w, 16 w + 16): products with the states first
    f32x4 aq[4], ab[4], aw[4];
    float es = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) aq[i] = ab[i] = aw[i] = zero4();
#pragma unroll 1
    for (int ks = 0; ks < NKS; ++ks) {
        const int o = w * NW + 2 * ks;
        const f32x4 s0 = mem_row(S, o, L), s1 = mem_row(S, o + 1, L);
        const f32x4 d0 = mem_row(Dn, o, L), d1 = mem_row(Dn, o + 1, L);
#pragma unroll
        for (int r = 0; r < 4; ++r) es = fmaf(s0[r], d0[r], fmaf(s1[r], d1[r], es));
        const Split8<2> s = split_pair(s0, s1), d = split_pair(d0, d1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            aq[i] = mms(PL::template frag<NX>(sO, 16 * i, r16, ks, g4), s, aq[i]);
            ab[i] = mms(PL::template frag<2>(P2, 16 * i, r16, ks, g4), s, ab[i]);
            aw[i] = mms(PL::template frag<2>(P1, 16 * i, r16, ks, g4), d, aw[i]);
        }
    }
    es = g4_sum(es) * fast_exp(gc);
    float ew_sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            aq[i][r] *= fast_exp(G[i][r]);
            ab[i][r] *= -fast_exp(Gp[i][r]);
            aw[i][r] *= ew[i][r];
            ew_sum = fmaf(kk[i][r] * be[i][r], aw[i][r], ew_sum);
        }
    es += g4_sum(ew_sum);  // sum over the value columns of D * S_next

    if (!wide) {
        f32x4 x[4], y[4], a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) x[i][r] = kk[i][r] * be[i][r] * fast_exp(m - G[i][r]);
            a[i] = b[i] = zero4();
        }
        {
            const Split8<2> xs[2] = {split_pair(x[0], x[1]), split_pair(x[2], x[3])};
            mul_lower<false>(sA, xs, L, a);
            mul_lower<false>(sL, xs, L, b);
        }
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
        {
            const Split8<2> xs[2] = {split_pair(x[0], x[1]), split_pair(x[2], x[3])};
            const Split8<2> ys[2] = {split_pair(y[0], y[1]), split_pair(y[2], y[3])};
            mul_lower<true>(sA, xs, L, a);
            mul_lower<true>(sL, ys, L, a);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) aw[j][r] = fmaf(a[j][r], fast_exp(m - G[j][r]), aw[j][r]);
    } else {
        // once every wave is past its reads of U, dR and D, their places take the three sums
        __syncthreads();
        constexpr int LD = D;  // an fp32 row takes the place of the two parts' rows
        float* F1 = reinterpret_cast<float*>(P1);
        float* F2 = reinterpret_cast<float*>(P2);
        float* F3 = p.ws_d + k.id * (D * D);
        wide_pairs<T, D, LD>(p, k, col, sA, sL, F1, F2, F3);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int a = (16 * i + 4 * g4 + r) * LD + col;
                aq[i][r] += F1[a];
                ab[i][r] += F2[a];
                aw[i][r] += F3[(16 * i + 4 * g4 + r) * D + col];
            }
    }
    store_rows<T>(out_rows<T, D>(p, p.dq, k, col, L), aq);
    // q dq - w dw (x) and k dkB (y): dg_t = D * S_next + sum_{r >= t} x_r + sum_{r > t} y_r
    f32x4 y[4], inc[4], exc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float wdw = kk[i][r] * be[i][r] * aw[i][r];
            q[i][r] = q[i][r] * aq[i][r] - wdw;
            y[i][r] = q[i][r] + kk[i][r] * ab[i][r];
            ab[i][r] = fmaf(be[i][r], aw[i][r], ab[i][r]);
            aw[i][r] *= kk[i][r];
        }
    store_rows<T>(out_rows<T, D>(p, p.dk, k, col, L), ab);
    token_scan<true>(y, L, inc, exc);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) exc[i][r] = (pass >> (4 * i + r) & 1) ? exc[i][r] + q[i][r] + es : 0.f;
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

template <typename T, int D>
hipError_t launch_t(const GdnChunkBwdParams& p, hipStream_t stream) {
    const unsigned chunks = (unsigned)(p.f.B * p.f.H * p.nc);
    hipError_t e;
    hipLaunchKernelGGL((gdn_bwd_map_kernel<T, D>), dim3(chunks), dim3(4 * D), 0, stream, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const unsigned pairs8 = (unsigned)((p.f.B * p.f.H + 7) / 8 * 8);
    hipLaunchKernelGGL((gdn_bwd_scan_kernel<D>), dim3(pairs8 * 2 * ScanPlan<D>::NS), dim3(4 * D), 0, stream, p);
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
