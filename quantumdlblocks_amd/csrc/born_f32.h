// fp32 flash-Born and purified-Born attention for head dims up to 128 (but for
// the launches of f32_staged): forward, dQ and dK/dV on v_mfma_f32_32x32x2_f32 (the reference runs its
// fp32 dots with allow_tf32=False, flash_born.py:160, 298).
//
// What bounds it: the fp32 matrix pipe (64 cycles per 32x32x2 MFMA, 153
// TFLOP/s over the card), and at the sizes fp32 is used for, the longest
// serial chain of tiles: 128-row blocks of four waves left half of the SIMDs
// without a wave at B2 H8 T1000, each running up to 32 tiles one after the
// other (D = 64: 83 us forward, 119 us dQ, 158 us dK/dV).
//
// So a workgroup owns 32 stationary rows (queries in the forward and dQ, keys
// in dK/dV) and its four waves take every fourth tile of the streamed operand
// (the weights of a row have no running maximum, so the partial sums only
// add); the waves' partial accumulators and row sums meet in LDS once, at the
// end.  That gives four times the workgroups, a quarter of the chain, and no
// barrier in the tile loop: each wave keeps its own tile of each streamed
// operand in LDS, filled by LDS-DMA loads and read in both operand layouts.
// One buffer per operand is enough, because every contraction reads only one
// of them: an operand's next tile is issued as soon as its last contraction is
// done, and lands under the next contraction of the other one.  (Operands
// straight from L2 into registers need no LDS either, but a row-layout load
// touches 64 separate 16-byte pieces: 37 + 85 + 104 us.)
//
// B2 H8 T1000 D64 causal: forward 84 -> 30 us, dQ 120 -> 44, dK/dV 159 -> 53
// (7.2 GFLOP in 127 us, 57 TFLOP/s of the 153 the matrix pipe reaches; a
// block's start, its short last round of tiles and the reduction take the
// rest); B8 H8 T1024: 115 -> 101, 168 -> 150, 222 -> 182 us.
//
// Operand layouts (the contraction index and the output columns may be
// permuted freely, see born_common.h):
//   rows:    lane (c, g) holds row c, columns 8u + 4g .. + 3 of chunk u: the
//            A operand of the overlaps (contraction over the head dim);
//   columns: lane (c, g) holds row acc_row(r, g), columns DB c .. DB c + DB-1
//            (DB = DP / 32): the A operand of the products whose contraction
//            runs over the tile's rows.  Accumulator db, register r of lane
//            (c, g) is then output row c, column DB acc_row(r, g) + db.
// Rows past T and columns past D (a multiple of 8) read as zeros through the
// buffer descriptor's range check.
#pragma once

#include <type_traits>

#include "born_common.h"
#include "born_fwd_fast.h"
#include "f32_rule.h"
#include "purified_args.h"
#include "split16_rule.h"

namespace qdl {

// A descriptor over the 32 rows from r0 (uniform) of a slice of `width` floats
// per row; loads past row T return zeros.
__device__ __forceinline__ i32x4 f32_rows_rsrc(const float* slice, int r0, int T, int width) {
    i32x4 rs = buffer_rsrc(slice + (size_t)r0 * width, (uint32_t)(max(0, min(kF32Rows, T - r0)) * width * 4));
#pragma unroll
    for (int i = 0; i < 4; ++i) rs[i] = __builtin_amdgcn_readfirstlane(rs[i]);  // the DMA takes it in SGPRs
    return rs;
}

// Stationary rows, straight into registers (row layout).
template <int KQ>
__device__ __forceinline__ void f32_load_rows(f32x4 (&x)[KQ], const float* slice, int row, int T, int D, int g) {
#pragma unroll
    for (int u = 0; u < KQ; ++u) {
        const int d = 8 * u + 4 * g;
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
        if (row < T && d < D) y = *reinterpret_cast<const f32x4*>(slice + (size_t)row * D + d);
        x[u] = y;
    }
}

// A wave's 32-row tile of one streamed operand in LDS: rows of 4 DP bytes,
// 16-byte chunks XOR-swizzled per row so that 16 lanes reading one chunk of 16
// rows (a ds_read_b128 quarter) spread over the banks: rows that start on one
// bank (256- and 512-byte rows) by row & 15, rows of alternating halves (128
// and 384 bytes) by lds_swz within each 8 chunks.
template <int DP>
struct F32Tile {
    static constexpr int RB = 4 * DP, CPR = RB / 16, BYTES = kF32Rows * RB, LOADS = BYTES / 1024, DB = DP / 32;
    uint8_t* lds;
    __device__ __forceinline__ static int swz(int row) { return DP % 64 == 0 ? row & 15 : lds_swz(row); }
    __device__ __forceinline__ void issue(const float* slice, int r0, int T, int D, int lane) const {
        const i32x4 rs = f32_rows_rsrc(slice, r0, T, D);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int slot = 64 * i + lane, row = slot / CPR, chunk = (slot % CPR) ^ swz(row);
            dma_load16(rs, lds_addr(lds + 1024 * i), 4 * chunk < D ? row * D * 4 + 16 * chunk : kBufOOB);
        }
    }
    __device__ __forceinline__ f32x4 rows(int u, int c, int g) const {
        return *reinterpret_cast<const f32x4*>(lds + c * RB + (((2 * u + g) ^ swz(c)) << 4));
    }
    __device__ __forceinline__ void columns(float (&x)[DB], int r, int c, int g) const {
        const int row = acc_row(r, g);
        const uint8_t* b = lds + row * RB;
        if constexpr (DB == 2) {
            const f32x2 y = *reinterpret_cast<const f32x2*>(b + (((c >> 1) ^ swz(row)) << 4) + 8 * (c & 1));
            x[0] = y[0];
            x[1] = y[1];
        } else if constexpr (DB == 4) {
            const f32x4 y = *reinterpret_cast<const f32x4*>(b + ((c ^ swz(row)) << 4));
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = y[i];
        } else {
#pragma unroll
            for (int i = 0; i < DB; ++i) {
                const int d = DB * c + i;
                x[i] = *reinterpret_cast<const float*>(b + (((d >> 2) ^ swz(row)) << 4) + 4 * (d & 3));
            }
        }
    }
};

// At most N of this wave's vector-memory operations outstanding: without a
// barrier behind it, the wait itself has to keep LDS reads below it.
template <int N>
__device__ __forceinline__ void f32_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// 32 values (row sums, ids) of a (T) vector from r0 -> 128 bytes of LDS.
__device__ __forceinline__ void f32_issue_values(const void* v, int r0, int T, void* lds, int lane) {
    const i32x4 rs = f32_rows_rsrc(reinterpret_cast<const float*>(v), r0, T, 1);
    if (lane < 8) dma_load16(rs, lds_addr(lds), 16 * lane);
}

// Block of a workgroup: the longest tile ranges first (split_rank).
struct SplitBlock {
    int bh, mb;
    __device__ __forceinline__ SplitBlock(int bid, int grid, int BH, int nmb, bool longest_last, bool two_per_cu) {
        const int rank = split_rank(bid, grid, two_per_cu);
        bh = rank % BH;
        mb = longest_last ? nmb - 1 - rank / BH : rank / BH;
    }
};

// Document of a block's own row; past T the last row's.  Those rows are not
// stored and add nothing, but an id of their own would send every tile of the
// last block through the masked body (Born bf16 B1 H4 T1300 D128 dense, one document:
// forward 46.2 -> 29.4 us, backward 94 -> 68).
__device__ __forceinline__ int split_row_doc(const int32_t* docb, int row, int T) { return docb[min(row, T - 1)]; }

// Which (query, key) pairs a block's rows see.
struct SplitMask {
    bool causal, has_doc;
    int window;
    __device__ __forceinline__ bool visible(int i, int j, int di, int dj) const {
        return !(causal && j > i) && !(window > 0 && i - j >= window) && !(has_doc && di != dj);
    }
    // Whether the 32 queries from i0 and 32 keys from j0 may hold masked pairs.
    __device__ __forceinline__ bool cuts(int i0, int j0) const {
        return (causal && j0 + 31 > i0) || (window > 0 && i0 + 31 - j0 >= window);
    }
};

// A wave's accumulators -> its [32][DP + 4] share of the reduction buffer.
template <int DB>
__device__ __forceinline__ void f32_put(float* red, const f32x16 (&acc)[DB], int c, int g) {
    constexpr int RS = 32 * DB + 4;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int db = 0; db < DB; ++db) red[c * RS + DB * (8 * j + 4 * g + e) + db] = acc[db][4 * j + e];
}

// The waves' shares summed in wave order and finished by the row's finish(row,
// sum), to rows r0 .. of a (T, D) slice.
template <int DB, int NW, class F>
__device__ __forceinline__ void f32_reduce_store(const float* red, float* out, int r0, int T, int D, F&& finish) {
    constexpr int DP = 32 * DB, RS = DP + 4, CH = DP / 4;
    for (int idx = threadIdx.x; idx < kF32Rows * CH; idx += 64 * NW) {
        const int row = idx / CH, col = 4 * (idx % CH);
        if (r0 + row >= T || col >= D) continue;
        f32x4 x = *reinterpret_cast<const f32x4*>(red + row * RS + col);
#pragma unroll
        for (int w = 1; w < NW; ++w) x += *reinterpret_cast<const f32x4*>(red + (w * kF32Rows + row) * RS + col);
        *reinterpret_cast<f32x4*>(out + (size_t)(r0 + row) * D + col) = finish(row, x);
    }
}

template <bool PUR, class Args>
struct F32Weights {
    float gam = 0.f, tau = 0.f, eb = 0.f;
    __device__ __forceinline__ F32Weights(const Args& p, int h) {
        if constexpr (PUR) {
            gam = arg_scale(p, h);
            tau = arg_tau(p, h);
            eb = p.eps_base;
        }
    }
};

// ---------------------------------------------------------------------------
// Forward: S^T = K Q^T per tile, the weights in place, O^T += V^T P^T.
// ---------------------------------------------------------------------------
template <int DP, bool PUR, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DP <= 64 ? 2 : 1)))
void born_f32_fwd_kernel(typename std::conditional<PUR, PurArgs, FwdArgs>::type p) {
    using Args = decltype(p);
    constexpr int KQ = DP / 8, DB = DP / 32;
    // Each wave's K and V tile; the reduction buffer once they are done with.
    __shared__ __attribute__((aligned(1024))) uint8_t tiles[NW * 2 * F32Tile<DP>::BYTES];
    __shared__ __attribute__((aligned(16))) int32_t kd_lds[NW][kF32Rows];
    __shared__ float zred[NW][kF32Rows];
    __shared__ int32_t span_red[4];
    float* const red = reinterpret_cast<float*>(tiles);
    static_assert(sizeof(tiles) >= NW * kF32Rows * (DP + 4) * 4, "reduction buffer");

    const int T = p.T, D = p.D, BH = p.B * p.H;
    const int nmb = (T + kF32Rows - 1) / kF32Rows;
    const SplitMask m = {p.is_causal != 0, p.doc != nullptr, p.window};
    const SplitBlock blk((int)blockIdx.x, (int)gridDim.x, BH, nmb, m.causal, split_two_per_cu(sizeof(tiles)));
    const int b = blk.bh / p.H, h = blk.bh % p.H, m0 = blk.mb * kF32Rows;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;
    const int qi = m0 + c;

    const size_t base = (size_t)blk.bh * T * D;
    const float* __restrict__ Q = reinterpret_cast<const float*>(p.q) + base;
    const float* __restrict__ K = reinterpret_cast<const float*>(p.k) + base;
    const float* __restrict__ V = reinterpret_cast<const float*>(p.v) + base;
    const int32_t* __restrict__ docb = m.has_doc ? p.doc + (size_t)b * T : nullptr;
    const float sc = arg_scale(p, h);
    const F32Weights<PUR, Args> pw(p, h);

    int t_lo = 0, t_hi = ((m.causal ? min(T, m0 + kF32Rows) : T) + 31) / 32 - 1;  // first and last key tile
    if (m.window > 0) t_lo = max(0, m0 - m.window + 1) / 32;
    if (m.has_doc) {
        const int2 sp = doc_tile_span<32>(docb, T, m0, min(T, m0 + kF32Rows), t_lo, t_hi, span_red);
        t_lo = __builtin_amdgcn_readfirstlane(sp.x);
        t_hi = __builtin_amdgcn_readfirstlane(sp.y);
    }
    const int qdoc = m.has_doc ? split_row_doc(docb, qi, T) : -1;

    f32x4 qr[KQ];
    f32_load_rows(qr, Q, qi, T, D, g);
    if constexpr (!PUR) {
        const float sgn = sc < 0.f ? -1.f : 1.f;
#pragma unroll
        for (int u = 0; u < KQ; ++u) qr[u] *= sgn;
    }
    f32x16 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = zero16();
    float zacc = 0.f;

    const F32Tile<DP> kt = {tiles + (2 * wave) * F32Tile<DP>::BYTES}, vt = {tiles + (2 * wave + 1) * F32Tile<DP>::BYTES};
    constexpr int LOADS = F32Tile<DP>::LOADS;
    // A tile's key ids travel with its K rows.
    auto issue_k = [&](int t) __attribute__((always_inline)) {
        if (m.has_doc) f32_issue_values(docb, 32 * t, T, kd_lds[wave], lane);
        kt.issue(K, 32 * t, T, D, lane);
    };
    int t = t_lo <= t_hi ? t_lo + wave : 1 << 30;
    if (t <= t_hi) {
        issue_k(t);
        vt.issue(V, 32 * t, T, D, lane);
    }
    for (; t <= t_hi; t += NW) {
        const int key0 = 32 * t;
        const bool more = t + NW <= t_hi;
        f32_wait<LOADS>();  // K; V's loads were issued after it
        f32x16 s = zero16();
#pragma unroll
        for (int u = 0; u < KQ; ++u) {
            const f32x4 a = kt.rows(u, c, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) s = mfma_f32(a[e], qr[u][e], s);
        }
        int kdoc = m.has_doc && key0 + c < T ? kd_lds[wave][c] : -2;
        asm volatile("" : "+v"(kdoc));  // read for good before the next ids are sent into its place
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_k(t + NW);
        bool cut = m.cuts(m0, key0) || (PUR && key0 + 32 > T);
        if (m.has_doc) {
            const int d0 = __builtin_amdgcn_readfirstlane(kdoc);
            cut = cut || __ballot(kdoc != d0 || qdoc != d0) != 0;
        }
        if constexpr (PUR) {
            uint32_t keep = 0xffffu;
            if (cut) {
                keep = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kk = key0 + acc_row(r, g);
                    const int kd = m.has_doc ? __shfl(kdoc, acc_row(r, g)) : 0;
                    if (kk < T && m.visible(qi, kk, qdoc, kd)) keep |= 1u << r;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const bool vis = (keep >> r) & 1u;
                const float x = s[r];
                const float uu = vis ? fmaxf(pw.gam * (x - pw.tau), 0.f) : 0.f;
                const float bb = vis ? fmaxf(x, 0.f) : 0.f;
                const float u2 = uu * uu;
                const float pr = u2 * u2 + pw.eb * (bb * bb);
                zacc += pr;
                s[r] = pr;
            }
        } else {
            if (cut) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kd = m.has_doc ? __shfl(kdoc, acc_row(r, g)) : 0;
                    if (!m.visible(qi, key0 + acc_row(r, g), qdoc, kd)) s[r] = 0.f;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float x = fmaxf(s[r], 0.f);
                const float pr = x * x;
                zacc += pr;
                s[r] = pr;
            }
        }
        if (more) f32_wait<LOADS>();  // V; the next K's loads were issued after it
        else f32_wait<0>();
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float a[DB];
            vt.columns(a, r, c, g);
#pragma unroll
            for (int db = 0; db < DB; ++db) oacc[db] = mfma_f32(a[db], s[r], oacc[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) vt.issue(V, key0 + 32 * NW, T, D, lane);
    }

    __syncthreads();
    f32_put<DB>(red + wave * kF32Rows * (DP + 4), oacc, c, g);
    const float zw = zacc + __shfl_xor(zacc, 32);
    if (g == 0) zred[wave][c] = zw;
    __syncthreads();
    const float s2 = sc * sc;
    const float eps_s = (PUR || p.eps == 0.f) ? p.eps : p.eps / s2;
    auto zsum = [&](int row) {
        float z = zred[0][row];
#pragma unroll
        for (int w = 1; w < NW; ++w) z += zred[w][row];
        return z;
    };
    f32_reduce_store<DB, NW>(red, reinterpret_cast<float*>(p.o) + base, m0, T, D,
                         [&](int row, f32x4 x) -> f32x4 {
                             const float zd = zsum(row) + eps_s;
                             return PUR ? x / zd : x * (1.0f / zd);
                         });
    if (tid < kF32Rows && m0 + tid < T)
        p.z[(size_t)blk.bh * T + m0 + tid] = PUR ? zsum(tid) + p.eps : s2 * zsum(tid) + p.eps;
}

// ---------------------------------------------------------------------------
// dQ: S^T = K Q^T, dP^T = V dO^T per tile, dQ^T += K^T dS^T.  Also forms
// -delta = -(dO . O) and 1 / Z per row for the dK/dV kernel (and delta / Z for
// dscale), so no pre-pass reads dO and O again.
// ---------------------------------------------------------------------------
template <int DP, bool PUR, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DP <= 64 ? 2 : 1)))
void born_f32_dq_kernel(typename std::conditional<PUR, PurArgs, BwdArgs>::type p) {
    using Args = decltype(p);
    constexpr int KQ = DP / 8, DB = DP / 32;
    __shared__ __attribute__((aligned(1024))) uint8_t tiles[NW * 2 * F32Tile<DP>::BYTES];
    __shared__ __attribute__((aligned(16))) int32_t kd_lds[NW][kF32Rows];
    __shared__ int32_t span_red[4];
    float* const red = reinterpret_cast<float*>(tiles);

    const int T = p.T, D = p.D, BH = p.B * p.H;
    const int nmb = (T + kF32Rows - 1) / kF32Rows;
    const SplitMask m = {p.is_causal != 0, p.doc != nullptr, p.window};
    const SplitBlock blk((int)blockIdx.x, (int)gridDim.x, BH, nmb, m.causal, split_two_per_cu(sizeof(tiles)));
    const int b = blk.bh / p.H, h = blk.bh % p.H, m0 = blk.mb * kF32Rows;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;
    const int qi = m0 + c;

    const size_t base = (size_t)blk.bh * T * D;
    const float* __restrict__ Q = reinterpret_cast<const float*>(p.q) + base;
    const float* __restrict__ K = reinterpret_cast<const float*>(p.k) + base;
    const float* __restrict__ V = reinterpret_cast<const float*>(p.v) + base;
    const float* __restrict__ dO = reinterpret_cast<const float*>(p.dout) + base;
    const float* __restrict__ O;
    const float* __restrict__ Zr;
    if constexpr (PUR) {
        O = p.o_in + base;
        Zr = p.z_in + (size_t)blk.bh * T;
    } else {
        O = reinterpret_cast<const float*>(p.o) + base;
        Zr = p.z + (size_t)blk.bh * T;
    }
    const int32_t* __restrict__ docb = m.has_doc ? p.doc + (size_t)b * T : nullptr;
    const float sc = arg_scale(p, h);
    const F32Weights<PUR, Args> pw(p, h);

    int t_lo = 0, t_hi = ((m.causal ? min(T, m0 + kF32Rows) : T) + 31) / 32 - 1;
    if (m.window > 0) t_lo = max(0, m0 - m.window + 1) / 32;
    if (m.has_doc) {
        const int2 sp = doc_tile_span<32>(docb, T, m0, min(T, m0 + kF32Rows), t_lo, t_hi, span_red);
        t_lo = __builtin_amdgcn_readfirstlane(sp.x);
        t_hi = __builtin_amdgcn_readfirstlane(sp.y);
    }
    const int qdoc = m.has_doc ? split_row_doc(docb, qi, T) : -1;

    f32x4 qr[KQ], dr[KQ];
    f32_load_rows(qr, Q, qi, T, D, g);
    f32_load_rows(dr, dO, qi, T, D, g);
    float delta = 0.f;
    {
        f32x4 orow[KQ];
        f32_load_rows(orow, O, qi, T, D, g);
#pragma unroll
        for (int u = 0; u < KQ; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) delta = fmaf(orow[u][e], dr[u][e], delta);
        delta += __shfl_xor(delta, 32);
    }
    const bool qok = qi < T;
    const float z = qok ? Zr[qi] : 1.f;
    const float zinv = qok ? 1.0f / z : 0.f;
    // Born: dP / Z = dP^T . 1/Z - delta / Z; purified: (dP^T - delta) . 1/Z.
    const float dz = qok ? delta / z : 0.f;
    if (wave == 0 && g == 0 && qok) {
        const size_t i = (size_t)blk.bh * T + qi;
        p.ndelta[i] = -delta;
        p.zinv[i] = zinv;
        if constexpr (!PUR) p.delta_z[i] = dz;
    }
    if constexpr (!PUR) {
        const float sgn = sc < 0.f ? -1.f : 1.f;
#pragma unroll
        for (int u = 0; u < KQ; ++u) qr[u] *= sgn;
    }
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = zero16();

    const F32Tile<DP> kt = {tiles + (2 * wave) * F32Tile<DP>::BYTES}, vt = {tiles + (2 * wave + 1) * F32Tile<DP>::BYTES};
    constexpr int LOADS = F32Tile<DP>::LOADS;
    // A tile's key ids travel with its V rows.
    auto issue_v = [&](int t) __attribute__((always_inline)) {
        if (m.has_doc) f32_issue_values(docb, 32 * t, T, kd_lds[wave], lane);
        vt.issue(V, 32 * t, T, D, lane);
    };
    int t = t_lo <= t_hi ? t_lo + wave : 1 << 30;
    if (t <= t_hi) {
        issue_v(t);
        kt.issue(K, 32 * t, T, D, lane);
    }
    for (; t <= t_hi; t += NW) {
        const int key0 = 32 * t;
        const bool more = t + NW <= t_hi;
        f32_wait<LOADS>();  // V; K's loads were issued after it
        f32x16 s = zero16(), tt = zero16();
#pragma unroll
        for (int u = 0; u < KQ; ++u) {
            const f32x4 a = vt.rows(u, c, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) tt = mfma_f32(a[e], dr[u][e], tt);
        }
        int kdoc = m.has_doc && key0 + c < T ? kd_lds[wave][c] : -2;
        asm volatile("" : "+v"(kdoc));  // read for good before the next ids are sent into its place
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
            issue_v(t + NW);
            f32_wait<LOADS>();  // K; the next V's loads were issued after it
        } else {
            f32_wait<0>();
        }
#pragma unroll
        for (int u = 0; u < KQ; ++u) {
            const f32x4 a = kt.rows(u, c, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) s = mfma_f32(a[e], qr[u][e], s);
        }
        bool cut = m.cuts(m0, key0) || (PUR && key0 + 32 > T);
        if (m.has_doc) {
            const int d0 = __builtin_amdgcn_readfirstlane(kdoc);
            cut = cut || __ballot(kdoc != d0 || qdoc != d0) != 0;
        }
        uint32_t keep = 0xffffu;
        if (cut) {
            keep = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int kk = key0 + acc_row(r, g);
                const int kd = m.has_doc ? __shfl(kdoc, acc_row(r, g)) : 0;
                if (kk < T && m.visible(qi, kk, qdoc, kd)) keep |= 1u << r;
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const bool vis = (keep >> r) & 1u;
            if constexpr (PUR) {
                const float x = s[r], dpz = (tt[r] - delta) * zinv;
                const float uu = vis ? fmaxf(pw.gam * (x - pw.tau), 0.f) : 0.f;
                const float bb = vis ? fmaxf(x, 0.f) : 0.f;
                const float du = 4.0f * (uu * uu * uu) * dpz;
                s[r] = du * pw.gam + 2.0f * pw.eb * bb * dpz;
            } else {
                const float x = vis ? fmaxf(s[r], 0.f) : 0.f;
                s[r] = x * fmaf(tt[r], zinv, -dz);
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float a[DB];
            kt.columns(a, r, c, g);
#pragma unroll
            for (int db = 0; db < DB; ++db) acc[db] = mfma_f32(a[db], s[r], acc[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) kt.issue(K, key0 + 32 * NW, T, D, lane);
    }
    __syncthreads();
    f32_put<DB>(red + wave * kF32Rows * (DP + 4), acc, c, g);
    __syncthreads();
    const float f = PUR ? 1.f : 2.f * sc * fabsf(sc);
    f32_reduce_store<DB, NW>(red, reinterpret_cast<float*>(p.dq) + base, m0, T, D, [&](int, f32x4 x) -> f32x4 { return x * f; });
}

// ---------------------------------------------------------------------------
// dK / dV (purified: with a fixed scale and tau, whose gradients these kernels
// do not form; see purified_split_ok).  Keys stationary; per query tile S = Q K^T, dP = dO V^T - delta, dV^T += dO^T W, dK^T += Q^T dS.
// ---------------------------------------------------------------------------
template <int DP, bool PUR, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DP <= 64 ? 2 : 1)))
void born_f32_dkdv_kernel(typename std::conditional<PUR, PurArgs, BwdArgs>::type p) {
    using Args = decltype(p);
    constexpr int KQ = DP / 8, DB = DP / 32;
    __shared__ __attribute__((aligned(1024))) uint8_t tiles[NW * 2 * F32Tile<DP>::BYTES];
    // Per wave: the tile's -delta, 1 / Z and query ids.
    __shared__ __attribute__((aligned(16))) float rv_lds[NW][3][kF32Rows];
    __shared__ int32_t span_red[4];
    float* const red = reinterpret_cast<float*>(tiles);

    const int T = p.T, D = p.D, BH = p.B * p.H;
    const int nkb = (T + kF32Rows - 1) / kF32Rows;
    const SplitMask m = {p.is_causal != 0, p.doc != nullptr, p.window};
    const SplitBlock blk((int)blockIdx.x, (int)gridDim.x, BH, nkb, false, split_two_per_cu(sizeof(tiles)));
    const int b = blk.bh / p.H, h = blk.bh % p.H, k0 = blk.mb * kF32Rows;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;
    const int key = k0 + c;

    const size_t base = (size_t)blk.bh * T * D;
    const float* __restrict__ Q = reinterpret_cast<const float*>(p.q) + base;
    const float* __restrict__ K = reinterpret_cast<const float*>(p.k) + base;
    const float* __restrict__ V = reinterpret_cast<const float*>(p.v) + base;
    const float* __restrict__ dO = reinterpret_cast<const float*>(p.dout) + base;
    const float* __restrict__ NDl = p.ndelta + (size_t)blk.bh * T;
    const float* __restrict__ ZIl = p.zinv + (size_t)blk.bh * T;
    const int32_t* __restrict__ docb = m.has_doc ? p.doc + (size_t)b * T : nullptr;
    const float sc = arg_scale(p, h);
    const F32Weights<PUR, Args> pw(p, h);

    int t_lo = m.causal ? blk.mb : 0, t_hi = (T + 31) / 32 - 1;  // first and last query tile
    if (m.window > 0) t_hi = min(t_hi, (k0 + 31 + m.window - 1) / 32);
    if (m.has_doc) {
        const int2 sp = doc_tile_span<32>(docb, T, k0, min(T, k0 + kF32Rows), t_lo, t_hi, span_red);
        t_lo = __builtin_amdgcn_readfirstlane(sp.x);
        t_hi = __builtin_amdgcn_readfirstlane(sp.y);
    }
    const int kdoc = m.has_doc ? split_row_doc(docb, key, T) : -2;

    f32x4 kr[KQ], vr[KQ];
    f32_load_rows(kr, K, key, T, D, g);
    f32_load_rows(vr, V, key, T, D, g);
    if constexpr (!PUR) {
        const float sgn = sc < 0.f ? -1.f : 1.f;
#pragma unroll
        for (int u = 0; u < KQ; ++u) kr[u] *= sgn;
    }
    f32x16 dv[DB], dk[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) dv[db] = zero16(), dk[db] = zero16();

    const F32Tile<DP> qt = {tiles + (2 * wave) * F32Tile<DP>::BYTES}, dt = {tiles + (2 * wave + 1) * F32Tile<DP>::BYTES};
    constexpr int LOADS = F32Tile<DP>::LOADS;
    // A tile's row values travel with its dO rows, its ids with its Q rows.
    auto issue_d = [&](int t) __attribute__((always_inline)) {
        f32_issue_values(NDl, 32 * t, T, rv_lds[wave][0], lane);
        f32_issue_values(ZIl, 32 * t, T, rv_lds[wave][1], lane);
        dt.issue(dO, 32 * t, T, D, lane);
    };
    auto issue_q = [&](int t) __attribute__((always_inline)) {
        if (m.has_doc) f32_issue_values(docb, 32 * t, T, rv_lds[wave][2], lane);
        qt.issue(Q, 32 * t, T, D, lane);
    };
    auto row_values = [&](int which, f32x16& x) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 y = *reinterpret_cast<const f32x4*>(&rv_lds[wave][which][8 * j + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * j + e] = y[e];
        }
    };
    int t = t_lo <= t_hi ? t_lo + wave : 1 << 30;
    if (t <= t_hi) {
        issue_d(t);
        issue_q(t);
    }
    for (; t <= t_hi; t += NW) {
        const int i0 = 32 * t;
        const bool more = t + NW <= t_hi;
        f32_wait<LOADS>();  // dO and the row values; Q's loads were issued after them
        f32x16 s = zero16(), dp, zi;
        row_values(0, dp);
        row_values(1, zi);
#pragma unroll
        for (int u = 0; u < KQ; ++u) {
            const f32x4 a = dt.rows(u, c, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) dp = mfma_f32(a[e], vr[u][e], dp);
        }
        f32_wait<0>();  // Q
#pragma unroll
        for (int u = 0; u < KQ; ++u) {
            const f32x4 a = qt.rows(u, c, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) s = mfma_f32(a[e], kr[u][e], s);
        }
        const int qdoc = m.has_doc && i0 + c < T ? __float_as_int(rv_lds[wave][2][c]) : -1;
        bool cut = m.cuts(i0, k0) || (PUR && (k0 + 32 > T || i0 + 32 > T));
        if (m.has_doc) {
            const int d0 = __builtin_amdgcn_readfirstlane(qdoc);
            cut = cut || __ballot(qdoc != d0 || kdoc != d0) != 0;
        }
        uint32_t keep = 0xffffu;
        if (cut) {
            keep = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int qq = i0 + acc_row(r, g);
                const int qd = m.has_doc ? __shfl(qdoc, acc_row(r, g)) : 0;
                if (qq < T && key < T && m.visible(qq, key, qd, kdoc)) keep |= 1u << r;
            }
        }
        f32x16 w;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const bool vis = (keep >> r) & 1u;
            if constexpr (PUR) {
                const float x = s[r];
                const float uu = vis ? fmaxf(pw.gam * (x - pw.tau), 0.f) : 0.f;
                const float bb = vis ? fmaxf(x, 0.f) : 0.f;
                const float u2 = uu * uu;
                const float pr = u2 * u2 + pw.eb * (bb * bb);
                w[r] = pr * zi[r];
                const float dpz = dp[r] * zi[r];
                const float du = 4.0f * (u2 * uu) * dpz;
                s[r] = du * pw.gam + 2.0f * pw.eb * bb * dpz;
            } else {
                const float a = vis ? fmaxf(s[r], 0.f) : 0.f;
                const float tz = a * zi[r];
                w[r] = tz * a;
                s[r] = tz * dp[r];
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float a[DB];
            dt.columns(a, r, c, g);
#pragma unroll
            for (int db = 0; db < DB; ++db) dv[db] = mfma_f32(a[db], w[r], dv[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_d(t + NW);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float a[DB];
            qt.columns(a, r, c, g);
#pragma unroll
            for (int db = 0; db < DB; ++db) dk[db] = mfma_f32(a[db], s[r], dk[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_q(t + NW);
    }
    __syncthreads();

    const float fk = PUR ? 1.f : 2.f * sc * fabsf(sc), fv = PUR ? 1.f : sc * sc;
    float* const mine = red + wave * kF32Rows * (DP + 4);
    f32_put<DB>(mine, dv, c, g);
    __syncthreads();
    f32_reduce_store<DB, NW>(red, reinterpret_cast<float*>(p.dv) + base, k0, T, D, [&](int, f32x4 x) -> f32x4 { return x * fv; });
    __syncthreads();
    f32_put<DB>(mine, dk, c, g);
    __syncthreads();
    f32_reduce_store<DB, NW>(red, reinterpret_cast<float*>(p.dk) + base, k0, T, D, [&](int, f32x4 x) -> f32x4 { return x * fk; });
}

inline int f32_groups(int B, int H, int T) { return (int)f32_blocks((int64_t)B * H, T); }

#define QDL_F32_DP(D, BODY)                          \
    switch (((D) + 31) / 32) {                       \
        case 1: { constexpr int DPV = 32; BODY } break;  \
        case 2: { constexpr int DPV = 64; BODY } break;  \
        case 3: { constexpr int DPV = 96; BODY } break;  \
        case 4: { constexpr int DPV = 128; BODY } break; \
        default: return hipErrorInvalidValue;        \
    }
#define QDL_F32_NW(NWRT, BODY)                       \
    switch (NWRT) {                                  \
        case 1: { constexpr int NWV = 1; BODY } break;   \
        default: { constexpr int NWV = 4; BODY } break;  \
    }

template <bool PUR, class Args>
hipError_t launch_f32_fwd(const Args& a, hipStream_t st) {
    const dim3 grid((unsigned)f32_groups(a.B, a.H, a.T));
    const int nw = f32_waves((int64_t)a.B * a.H, a.T, a.D, a.is_causal != 0, a.window, a.doc != nullptr);
    QDL_F32_DP(a.D, {
        QDL_F32_NW(nw, {
            hipLaunchKernelGGL((born_f32_fwd_kernel<DPV, PUR, NWV>), grid, dim3(64 * NWV), 0, st, a);
        })
    })
    return hipGetLastError();
}

// dQ first (it forms the rows' -delta and 1 / Z), then dK/dV.
template <bool PUR, class Args>
hipError_t launch_f32_bwd(const Args& a, hipStream_t st) {
    const dim3 grid((unsigned)f32_groups(a.B, a.H, a.T));
    const int nw = f32_waves((int64_t)a.B * a.H, a.T, a.D, a.is_causal != 0, a.window, a.doc != nullptr);
    QDL_F32_DP(a.D, {
        QDL_F32_NW(nw, {
            hipLaunchKernelGGL((born_f32_dq_kernel<DPV, PUR, NWV>), grid, dim3(64 * NWV), 0, st, a);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            hipLaunchKernelGGL((born_f32_dkdv_kernel<DPV, PUR, NWV>), grid, dim3(64 * NWV), 0, st, a);
        })
    })
    return hipGetLastError();
}

}  // namespace qdl
