// 16-bit flash-Born and purified-Born attention of few blocks: forward, dQ and
// dK/dV for launches that would leave the tuned kernels' CUs idle.
//
// What bounds such a launch is its longest block, not the matrix pipe: the
// tuned kernels (born_fwd_fast.h and its kin) give a workgroup 128 to 256 rows
// and walk all of a block's tiles in one chain.  Here, as in the fp32 kernels
// (born_f32.h), a workgroup owns 32 or 64 stationary rows and its four waves
// take every fourth 32-row tile of the streamed operands; the waves' partial
// accumulators and row sums meet in LDS once, at the end.  Each wave keeps its
// own ring of tiles in LDS, filled by LDS-DMA loads, so there is no barrier in
// the tile loop.  The price is that every wave reads its tiles alone: 64 rows
// (two MFMA column blocks) share a tile where the registers allow it, which
// holds the L2 reads to 16 KiB per ~1400 cycles and SIMD at D = 128; the
// launches take these kernels only where they have CUs to spare
// (split16_pays).
//
// Arithmetic, masks and results are the tuned kernels': Born weights with the
// scale folded out for bf16 (born_weight_pair), purified weights split into
// bf16 hi + lo terms for P.V, fp32 sums throughout.
#pragma once

#include <type_traits>

#include "born_common.h"
#include "born_f32.h"
#include "born_fwd_fast.h"
#include "purified_args.h"
#include "split16_rule.h"

namespace qdl {

constexpr int kSplitNW = 4;

// A wave's 32-row tile of one streamed 16-bit operand in LDS: rows of 2 DP
// bytes, 16-byte chunks XOR-swizzled per row so that neither a row read (16
// rows, one chunk) nor a transposed read (4 consecutive rows, 64 bytes each)
// meets a bank twice: rows that all start on bank 0 (256 and 512 bytes) by
// all four bits of the row, rows of alternating halves (128) by lds_swz, rows
// on four starts (64 and 192) by the row's upper bits.
template <int DP>
struct Tile16 {
    static constexpr int RB = 2 * DP, CPR = RB / 16, BYTES = 32 * RB, LOADS = BYTES / 1024;
    static_assert(BYTES % 1024 == 0, "whole loads");
    uint8_t* lds;
    __device__ __forceinline__ static int swz(int row) {
        if constexpr (RB % 256 == 0) return ((row & 3) << 2) | ((row >> 2) & 3);
        else if constexpr (RB % 256 == 128) return lds_swz(row);
        else return (row >> 2) & 3;
    }
    // Lane's byte offsets of a tile's loads within a (T, D) slice; chunks past
    // D read out of range (zeros).
    __device__ __forceinline__ static void offsets(uint32_t (&off)[LOADS], int D, int lane) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int slot = 64 * i + lane, row = slot / CPR, chunk = (slot % CPR) ^ swz(row);
            off[i] = 8 * chunk < D ? (uint32_t)(row * D * 2 + 16 * chunk) : kSplitPastD;
        }
    }
    // The rows from byte `at` of the slice (rows past T: out of range).
    __device__ __forceinline__ void issue(i32x4 slice, const uint32_t (&off)[LOADS], int at) const {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            dma_load16(slice, lds_addr(lds + 1024 * i), (int)split16_load_at(off[i], (uint32_t)at));
    }
    // A operand of a contraction over the head dim: row c, columns 16 ks + 8 g .. + 7.
    __device__ __forceinline__ u32x4 row(int ks, int c, int g) const {
        return *reinterpret_cast<const u32x4*>(lds + c * RB + (((2 * ks + g) ^ swz(c)) << 4));
    }
    // A operand of a contraction over the tile's rows 16 hh .. + 15 (in the
    // accumulator's row order): columns 32 db .. + 31 across the lanes.
    __device__ __forceinline__ u32x4 transposed(int hh, int db, int lane) const {
        const int g = lane >> 5, r = 16 * hh + 4 * g + ((lane & 15) >> 2);
        const int col = 32 * db + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        auto at = [&](int row) {
            return reinterpret_cast<const uint16_t*>(lds + row * RB + (((col >> 3) ^ swz(row)) << 4) + (col & 7) * 2);
        };
        const u32x2 x = lds_read_tr16(at(r)), y = lds_read_tr16(at(r + 8));
        const u32x4 a = {x[0], x[1], y[0], y[1]};
        return a;
    }
};

template <int DP>
struct Split16Cfg {
    static constexpr int KS = DP / 16, DB = DP / 32;
    // Column blocks of 32 stationary queries (forward, dQ).
    static constexpr int NQB = DP <= 128 ? 2 : 1;
    // Ring stages: 64 KiB of tiles (two workgroups per CU) at DP = 64, 96 and
    // 128 KiB at DP = 96 and 128, and one stage (128 KiB) above.
    static constexpr int NST = DP <= 128 ? 2 : 1;
    static constexpr int WPE = DP <= 64 ? 2 : 1;
    // One tile body per stage (stage offsets as immediates) where two bodies
    // keep the accumulators in place; above, they are moved between the two
    // register files on every tile.
    static constexpr bool UNROLL = DP <= 64 && NST == 2;
    static constexpr int RING = NST * 2 * Tile16<DP>::BYTES;  // per wave
    static constexpr int REDUCE = 32 * (DP + 4) * 4;          // per wave
    static constexpr int SMEM = kSplitNW * (RING > REDUCE ? RING : REDUCE);
    // Operand A's tile t + NST is issued after its last use of tile t, then
    // B's likewise, so at each first use of a tile this many loads are younger
    // (more where ids travel along: a stricter wait).
    static constexpr int YOUNGER = Tile16<DP>::LOADS * (2 * NST - 1);
    static_assert(YOUNGER < 64, "vmcnt range");
};

// tile(i, stage) for a wave's n tiles.
template <bool UNROLL, int NST, class F>
__device__ __forceinline__ void split_tiles(int n, F&& tile) {
    if constexpr (UNROLL) {
        for (int i = 0; i < n; i += 2) {
            tile(i, std::integral_constant<int, 0>{});
            if (i + 1 < n) tile(i + 1, std::integral_constant<int, 1>{});
        }
    } else {
        for (int i = 0; i < n; ++i) tile(i, i % NST);
    }
}

// f(true) for a tile that may hold masked pairs, f(false) for the others
// (uniform): the plain body carries no mask code.
template <class F>
__device__ __forceinline__ void split_if_cut(bool cut, F&& f) {
    if (cut) f(std::true_type{});
    else f(std::false_type{});
}

// 32 rows of a wave's accumulators -> its [32][DP + 4] share.
template <int DB>
__device__ __forceinline__ void split_put(float* red, const f32x16 (&acc)[DB], int c, int g) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 w = {acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]};
            *reinterpret_cast<f32x4*>(red + c * (32 * DB + 4) + 32 * db + 8 * j + 4 * g) = w;
        }
}

// The waves' shares summed in wave order and finished by finish(row, sum), to
// rows r0 .. of a (T, D) slice: 16-bit (out) and fp32 (out32), or one of them.
template <class E, int DB, class F>
__device__ __forceinline__ void split_store(const float* red, uint16_t* out, float* out32, int r0, int T, int D,
                                            F&& finish) {
    constexpr int DP = 32 * DB, RS = DP + 4, CH = DP / 8;
    for (int idx = threadIdx.x; idx < 32 * CH; idx += 64 * kSplitNW) {
        const int row = idx / CH, col = 8 * (idx % CH);
        if (r0 + row >= T || col >= D) continue;
        f32x4 x = *reinterpret_cast<const f32x4*>(red + row * RS + col);
        f32x4 y = *reinterpret_cast<const f32x4*>(red + row * RS + col + 4);
#pragma unroll
        for (int w = 1; w < kSplitNW; ++w) {
            x += *reinterpret_cast<const f32x4*>(red + (32 * w + row) * RS + col);
            y += *reinterpret_cast<const f32x4*>(red + (32 * w + row) * RS + col + 4);
        }
        x = finish(row, x);
        y = finish(row, y);
        const size_t at = (size_t)(r0 + row) * D + col;
        if (out32 != nullptr) {
            *reinterpret_cast<f32x4*>(out32 + at) = x;
            *reinterpret_cast<f32x4*>(out32 + at + 4) = y;
        }
        if (out != nullptr) {
            const u32x4 w = {E::pack(x[0], x[1]), E::pack(x[2], x[3]), E::pack(y[0], y[1]), E::pack(y[2], y[3])};
            *reinterpret_cast<u32x4*>(out + at) = w;
        }
    }
}

// Descriptors of a (T, D) slice and of a (T) vector, in SGPRs.
__device__ __forceinline__ i32x4 split_slice(const uint16_t* slice, int T, int D) {
    return buffer_rsrc(slice, (uint32_t)T * (uint32_t)D * 2u);
}
__device__ __forceinline__ i32x4 split_slice32(const void* v, int T) { return buffer_rsrc(v, (uint32_t)T * 4u); }

// 32 values from row r0 -> 128 bytes of LDS.
__device__ __forceinline__ void split_issue_values(i32x4 rs, int r0, void* lds, int lane) {
    if (lane < 8) dma_load16(rs, lds_addr(lds), 4 * r0 + 16 * lane);
}

// Stationary 16-bit rows as B operands: lane (c, g) holds its row's columns 16
// ks + 8 g .. + 7, zeros past T and D.
template <int KS>
__device__ __forceinline__ void split_load_rows(u32x4 (&x)[KS], const uint16_t* slice, int row, int T, int D, int g) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int d = 16 * ks + 8 * g;
        u32x4 y = {0u, 0u, 0u, 0u};
        if (row < T && d < D) y = ldg16(slice + (size_t)row * D + d);
        x[ks] = y;
    }
}

// Bit r: whether the pair of stationary row `mine` and streamed row r0 +
// acc_row(r, g) is visible and inside T; sdoc: streamed row r0 + c's id.
template <bool QUERY_STATIONARY>
__device__ __forceinline__ uint32_t split_visible(const SplitMask& m, int mine, int mdoc, int r0, int sdoc, int T, int g) {
    uint32_t keep = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int other = r0 + acc_row(r, g);
        const int od = m.has_doc ? __shfl(sdoc, acc_row(r, g)) : 0;
        const bool v = QUERY_STATIONARY ? m.visible(mine, other, mdoc, od) : m.visible(other, mine, od, mdoc);
        if (other < T && v) keep |= 1u << r;
    }
    return keep;
}

// ---------------------------------------------------------------------------
// Forward.
// ---------------------------------------------------------------------------
template <class E, int DP, bool PUR>
__global__ __launch_bounds__(64 * kSplitNW) __attribute__((amdgpu_waves_per_eu(Split16Cfg<DP>::WPE)))
void born_split16_fwd_kernel(typename std::conditional<PUR, PurArgs, FwdArgs>::type p) {
    using C = Split16Cfg<DP>;
    using Tile = Tile16<DP>;
    constexpr int KS = C::KS, DB = C::DB, NQB = C::NQB, NST = C::NST, NW = kSplitNW, BM = 32 * NQB;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::SMEM];
    __shared__ __attribute__((aligned(16))) int32_t kd_lds[NW][NST][32];
    __shared__ float zred[NQB][NW][32];
    __shared__ int32_t span_red[4];
    float* const red = reinterpret_cast<float*>(smem);

    const int T = p.T, D = p.D, BH = p.B * p.H;
    const int nmb = (T + BM - 1) / BM;
    const SplitMask m = {p.is_causal != 0, p.doc != nullptr, p.window};
    const SplitBlock blk((int)blockIdx.x, (int)gridDim.x, BH, nmb, m.causal, split_two_per_cu(C::SMEM));
    const int b = blk.bh / p.H, h = blk.bh % p.H, m0 = blk.mb * BM;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;

    const size_t base = (size_t)blk.bh * T * D;
    const uint16_t* __restrict__ Q = reinterpret_cast<const uint16_t*>(p.q) + base;
    const uint16_t* __restrict__ K = reinterpret_cast<const uint16_t*>(p.k) + base;
    const uint16_t* __restrict__ V = reinterpret_cast<const uint16_t*>(p.v) + base;
    const int32_t* __restrict__ docb = m.has_doc ? p.doc + (size_t)b * T : nullptr;
    const float sc = arg_scale(p, h);
    const uint32_t flip = (!PUR && sc < 0.f) ? 0x80008000u : 0u;
    const float sq_pre = E::kScaleInSquare ? fabsf(sc) : 1.f;
    float pg = 0.f, pgt = 0.f, pse = 0.f;
    if constexpr (PUR) {
        pg = sc;
        pgt = -sc * arg_tau(p, h);
        pse = sqrtf(p.eps_base);
    }

    int t_lo = 0, t_hi = ((m.causal ? min(T, m0 + BM) : T) + 31) / 32 - 1;
    if (m.window > 0) t_lo = max(0, m0 - m.window + 1) / 32;
    if (m.has_doc) {
        const int2 sp = doc_tile_span<32>(docb, T, m0, min(T, m0 + BM), t_lo, t_hi, span_red);
        t_lo = __builtin_amdgcn_readfirstlane(sp.x);
        t_hi = __builtin_amdgcn_readfirstlane(sp.y);
    }
    const int n = t_lo <= t_hi ? (t_hi - t_lo - wave + NW) / NW : 0;  // this wave's tiles

    uint8_t* const ring = smem + wave * C::RING;
    auto kt = [&](int st) { return Tile{ring + st * 2 * Tile::BYTES}; };
    auto vt = [&](int st) { return Tile{ring + st * 2 * Tile::BYTES + Tile::BYTES}; };
    uint32_t off[Tile::LOADS];
    Tile::offsets(off, D, lane);
    const i32x4 rk = split_slice(K, T, D), rv = split_slice(V, T, D);
    // This wave's tile i; past the last one its loads are out of range and land
    // as zeros in a stage nobody reads, so the waits stay constant.
    auto row0 = [&](int i) { return i < n ? 32 * (t_lo + wave + NW * i) : T; };
    const i32x4 rdoc = split_slice32(docb, m.has_doc ? T : 0);
    auto issue_k = [&](int i, int st) __attribute__((always_inline)) {
        if (m.has_doc) split_issue_values(rdoc, row0(i), kd_lds[wave][st], lane);
        kt(st).issue(rk, off, row0(i) * D * 2);
    };
    auto issue_v = [&](int i, int st) __attribute__((always_inline)) { vt(st).issue(rv, off, row0(i) * D * 2); };

    u32x4 qr[NQB][KS];
    int qdoc[NQB];
    f32x16 oacc[NQB][DB];
    float zacc[NQB][2];
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        const int qi = m0 + 32 * qb + c;
        split_load_rows(qr[qb], Q, qi, T, D, g);
        qdoc[qb] = m.has_doc ? split_row_doc(docb, qi, T) : -1;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qr[qb][ks] ^= flip;
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[qb][db] = zero16();
        zacc[qb][0] = zacc[qb][1] = 0.f;
    }
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {  // landed before the ring's loads are counted
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qr[qb][ks]));
        asm volatile("" : "+v"(qdoc[qb]));
    }
#pragma unroll
    for (int i = 0; i < NST; ++i) {
        issue_k(i, i);
        issue_v(i, i);
    }

    auto tile = [&](int i, auto stage) __attribute__((always_inline)) {
        const int st = stage;
        const int key0 = row0(i);
        f32_wait<C::YOUNGER>();
        f32x16 s[NQB];
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) s[qb] = zero16();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const u32x4 a = kt(st).row(ks, c, g);
#pragma unroll
            for (int qb = 0; qb < NQB; ++qb) s[qb] = E::mfma(a, qr[qb][ks], s[qb]);
        }
        int kdoc = m.has_doc && key0 + c < T ? kd_lds[wave][st][c] : -2;
        asm volatile("" : "+v"(kdoc));  // read for good before the next ids are sent into its place
        __builtin_amdgcn_sched_barrier(0);
        issue_k(i + NST, st);
        uint32_t pk[NQB][8], pl[NQB][PUR ? 8 : 1];
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) {
            bool cut = m.cuts(m0 + 32 * qb, key0) || (PUR && key0 + 32 > T);
            if (m.has_doc) {
                const int d0 = __builtin_amdgcn_readfirstlane(kdoc);
                cut = cut || __ballot(kdoc != d0 || qdoc[qb] != d0) != 0;
            }
            split_if_cut(cut, [&](auto masked) __attribute__((always_inline)) {
                uint32_t keep = 0xffffu;
                if constexpr (masked.value) keep = split_visible<true>(m, m0 + 32 * qb + c, qdoc[qb], key0, kdoc, T, g);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float w[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float x = s[qb][2 * j + e];
                        if constexpr (PUR) {
                            const float u = relu_f32(fmaf(x, pg, pgt)), bq = relu_f32(x * pse), u2 = u * u;
                            w[e] = fmaf(u2, u2, bq * bq);
                        } else {
                            w[e] = x;
                        }
                        if (masked.value && !((keep >> (2 * j + e)) & 1u)) w[e] = 0.f;
                    }
                    if constexpr (PUR) {
                        zacc[qb][0] += w[0] + w[1];
                        const uint32_t hi = BF16::pack(w[0], w[1]);
                        pk[qb][j] = hi;
                        pl[qb][j] = BF16::pack(w[0] - BF16::lo(hi), w[1] - BF16::hi(hi));
                    } else {
                        pk[qb][j] = born_weight_pair<E>(w[0], w[1], sq_pre, zacc[qb][j & 1]);
                    }
                }
            });
        }
        f32_wait<C::YOUNGER>();
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const u32x4 a = vt(st).transposed(hh, db, lane);
#pragma unroll
                for (int qb = 0; qb < NQB; ++qb) {
                    const u32x4 bh = {pk[qb][4 * hh], pk[qb][4 * hh + 1], pk[qb][4 * hh + 2], pk[qb][4 * hh + 3]};
                    if constexpr (PUR) {
                        const u32x4 bl = {pl[qb][4 * hh], pl[qb][4 * hh + 1], pl[qb][4 * hh + 2], pl[qb][4 * hh + 3]};
                        oacc[qb][db] = pur_pv<E>(a, bh, bl, oacc[qb][db]);
                    } else {
                        oacc[qb][db] = E::mfma(a, bh, oacc[qb][db]);
                    }
                }
            }
        __builtin_amdgcn_sched_barrier(0);
        issue_v(i + NST, st);
    };
    split_tiles<C::UNROLL, NST>(n, tile);

    const float s2 = (sq_pre > 0.f) ? (sc / sq_pre) * (sc / sq_pre) : 0.f;
    const float eps_s = (PUR || p.eps == 0.f) ? p.eps : p.eps / s2;
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        const float zl = zacc[qb][0] + zacc[qb][1];
        const float zw = zl + __shfl_xor(zl, 32);
        if (g == 0) zred[qb][wave][c] = zw;
    }
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        f32_wait<0>();  // the ring's last (empty) loads
        __syncthreads();
        split_put<DB>(red + wave * 32 * (DP + 4), oacc[qb], c, g);
        __syncthreads();
        auto zsum = [&](int row) {
            float z = zred[qb][0][row];
#pragma unroll
            for (int w = 1; w < NW; ++w) z += zred[qb][w][row];
            return z;
        };
        const int r0 = m0 + 32 * qb;
        uint16_t* out;
        float* out32 = nullptr;
        if constexpr (PUR) {
            out = p.o16 != nullptr ? reinterpret_cast<uint16_t*>(p.o16) + base : nullptr;
            out32 = p.o != nullptr ? p.o + base : nullptr;
        } else {
            out = reinterpret_cast<uint16_t*>(p.o) + base;
        }
        split_store<E, DB>(red, out, out32, r0, T, D, [&](int row, f32x4 x) -> f32x4 {
            const float zd = zsum(row) + eps_s;
            return PUR ? x / zd : x * (1.0f / zd);
        });
        if (tid < 32 && r0 + tid < T)
            p.z[(size_t)blk.bh * T + r0 + tid] = PUR ? zsum(tid) + p.eps : s2 * zsum(tid) + p.eps;
    }
}

// ---------------------------------------------------------------------------
// dQ; also -delta and 1 / Z per row for the dK/dV kernel (and delta / Z).
// ---------------------------------------------------------------------------
template <class E, int DP, bool PUR>
__global__ __launch_bounds__(64 * kSplitNW) __attribute__((amdgpu_waves_per_eu(Split16Cfg<DP>::WPE)))
void born_split16_dq_kernel(typename std::conditional<PUR, PurArgs, BwdArgs>::type p) {
    using C = Split16Cfg<DP>;
    using Tile = Tile16<DP>;
    constexpr int KS = C::KS, DB = C::DB, NQB = C::NQB, NST = C::NST, NW = kSplitNW, BM = 32 * NQB;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::SMEM];
    __shared__ __attribute__((aligned(16))) int32_t kd_lds[NW][NST][32];
    __shared__ int32_t span_red[4];
    float* const red = reinterpret_cast<float*>(smem);

    const int T = p.T, D = p.D, BH = p.B * p.H;
    const int nmb = (T + BM - 1) / BM;
    const SplitMask m = {p.is_causal != 0, p.doc != nullptr, p.window};
    const SplitBlock blk((int)blockIdx.x, (int)gridDim.x, BH, nmb, m.causal, split_two_per_cu(C::SMEM));
    const int b = blk.bh / p.H, h = blk.bh % p.H, m0 = blk.mb * BM;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;

    const size_t base = (size_t)blk.bh * T * D;
    const uint16_t* __restrict__ Q = reinterpret_cast<const uint16_t*>(p.q) + base;
    const uint16_t* __restrict__ K = reinterpret_cast<const uint16_t*>(p.k) + base;
    const uint16_t* __restrict__ V = reinterpret_cast<const uint16_t*>(p.v) + base;
    const uint16_t* __restrict__ dO = reinterpret_cast<const uint16_t*>(p.dout) + base;
    const int32_t* __restrict__ docb = m.has_doc ? p.doc + (size_t)b * T : nullptr;
    const float sc = arg_scale(p, h);
    const uint32_t flip = (!PUR && sc < 0.f) ? 0x80008000u : 0u;
    const float sq_pre = (E::kScaleInSquare && sc != 0.f) ? 2.f * fabsf(sc) : 1.f;
    float pg = 0.f, pgt = 0.f, p4g = 0.f, p2e = 0.f;
    if constexpr (PUR) {
        pg = sc;
        pgt = -sc * arg_tau(p, h);
        p4g = 4.f * sc;
        p2e = 2.f * p.eps_base;
    }

    int t_lo = 0, t_hi = ((m.causal ? min(T, m0 + BM) : T) + 31) / 32 - 1;
    if (m.window > 0) t_lo = max(0, m0 - m.window + 1) / 32;
    if (m.has_doc) {
        const int2 sp = doc_tile_span<32>(docb, T, m0, min(T, m0 + BM), t_lo, t_hi, span_red);
        t_lo = __builtin_amdgcn_readfirstlane(sp.x);
        t_hi = __builtin_amdgcn_readfirstlane(sp.y);
    }
    const int n = t_lo <= t_hi ? (t_hi - t_lo - wave + NW) / NW : 0;

    uint8_t* const ring = smem + wave * C::RING;
    auto kt = [&](int st) { return Tile{ring + st * 2 * Tile::BYTES}; };
    auto vt = [&](int st) { return Tile{ring + st * 2 * Tile::BYTES + Tile::BYTES}; };
    uint32_t off[Tile::LOADS];
    Tile::offsets(off, D, lane);
    const i32x4 rk = split_slice(K, T, D), rv = split_slice(V, T, D);
    auto row0 = [&](int i) { return i < n ? 32 * (t_lo + wave + NW * i) : T; };
    // V is used first (dP), K last (dQ): their order in the ring.
    const i32x4 rdoc = split_slice32(docb, m.has_doc ? T : 0);
    auto issue_v = [&](int i, int st) __attribute__((always_inline)) {
        if (m.has_doc) split_issue_values(rdoc, row0(i), kd_lds[wave][st], lane);
        vt(st).issue(rv, off, row0(i) * D * 2);
    };
    auto issue_k = [&](int i, int st) __attribute__((always_inline)) { kt(st).issue(rk, off, row0(i) * D * 2); };

    u32x4 qr[NQB][KS], dr[NQB][KS];
    int qdoc[NQB];
    float zinv[NQB], nd[NQB];
    f32x16 acc[NQB][DB];
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        const int qi = m0 + 32 * qb + c;
        const bool ok = qi < T;
        split_load_rows(qr[qb], Q, qi, T, D, g);
        split_load_rows(dr[qb], dO, qi, T, D, g);
        qdoc[qb] = m.has_doc ? split_row_doc(docb, qi, T) : -1;
        // delta = dO . O of the row (each half wave holds half of it).
        float dl = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int d = 16 * ks + 8 * g;
            if (!ok || d >= D) continue;
            if constexpr (PUR) {
                const float* o = p.o_in + base + (size_t)qi * D + d;
                const f32x4 oa = *reinterpret_cast<const f32x4*>(o), ob = *reinterpret_cast<const f32x4*>(o + 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float o0 = j < 2 ? oa[2 * j] : ob[2 * j - 4], o1 = j < 2 ? oa[2 * j + 1] : ob[2 * j - 3];
                    dl += o0 * E::lo(dr[qb][ks][j]) + o1 * E::hi(dr[qb][ks][j]);
                }
            } else {
                const u32x4 o = ldg16(reinterpret_cast<const uint16_t*>(p.o) + base + (size_t)qi * D + d);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    dl += E::lo(o[j]) * E::lo(dr[qb][ks][j]) + E::hi(o[j]) * E::hi(dr[qb][ks][j]);
            }
        }
        dl += __shfl_xor(dl, 32);
        const size_t row = (size_t)blk.bh * T + qi;
        float z = 1.f;
        if (ok) {
            if constexpr (PUR) z = p.z_in[row];
            else z = p.z[row];
        }
        zinv[qb] = ok ? 1.0f / z : 0.f;
        nd[qb] = ok ? -(dl / z) : 0.f;
        if (ok && g == 0 && wave == 0) {
            p.ndelta[row] = -dl;
            p.zinv[row] = zinv[qb];
            if constexpr (!PUR) p.delta_z[row] = dl / z;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qr[qb][ks] ^= flip;
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[qb][db] = zero16();
    }
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qr[qb][ks]), "+v"(dr[qb][ks]));
        asm volatile("" : "+v"(zinv[qb]), "+v"(nd[qb]), "+v"(qdoc[qb]));
    }
#pragma unroll
    for (int i = 0; i < NST; ++i) {
        issue_v(i, i);
        issue_k(i, i);
    }

    auto tile = [&](int i, auto stage) __attribute__((always_inline)) {
        const int st = stage;
        const int key0 = row0(i);
        f32_wait<C::YOUNGER>();
        f32x16 s[NQB], t[NQB];
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) s[qb] = zero16(), t[qb] = zero16();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const u32x4 a = vt(st).row(ks, c, g);
#pragma unroll
            for (int qb = 0; qb < NQB; ++qb) t[qb] = E::mfma(a, dr[qb][ks], t[qb]);
        }
        int kdoc = m.has_doc && key0 + c < T ? kd_lds[wave][st][c] : -2;
        asm volatile("" : "+v"(kdoc));  // read for good before the next ids are sent into its place
        __builtin_amdgcn_sched_barrier(0);
        issue_v(i + NST, st);
        f32_wait<C::YOUNGER>();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const u32x4 a = kt(st).row(ks, c, g);
#pragma unroll
            for (int qb = 0; qb < NQB; ++qb) s[qb] = E::mfma(a, qr[qb][ks], s[qb]);
        }
        uint32_t pk[NQB][8];
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) {
            bool cut = m.cuts(m0 + 32 * qb, key0) || (PUR && key0 + 32 > T);
            if (m.has_doc) {
                const int d0 = __builtin_amdgcn_readfirstlane(kdoc);
                cut = cut || __ballot(kdoc != d0 || qdoc[qb] != d0) != 0;
            }
            split_if_cut(cut, [&](auto masked) __attribute__((always_inline)) {
                uint32_t keep = 0xffffu;
                if constexpr (masked.value) keep = split_visible<true>(m, m0 + 32 * qb + c, qdoc[qb], key0, kdoc, T, g);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float w[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int r = 2 * j + e;
                        const float dp = fmaf(t[qb][r], zinv[qb], nd[qb]);
                        float f;
                        if constexpr (PUR) {
                            const float x = s[qb][r], u = relu_f32(fmaf(x, pg, pgt));
                            f = fmaf(p4g, u * u * u, p2e * relu_f32(x));
                        } else {
                            f = relu_f32(E::kScaleInSquare ? s[qb][r] * sq_pre : s[qb][r]);
                        }
                        w[e] = f * dp;
                        if (masked.value && !((keep >> r) & 1u)) w[e] = 0.f;
                    }
                    pk[qb][j] = E::pack(w[0], w[1]);
                }
            });
        }
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const u32x4 a = kt(st).transposed(hh, db, lane);
#pragma unroll
                for (int qb = 0; qb < NQB; ++qb) {
                    const u32x4 bq = {pk[qb][4 * hh], pk[qb][4 * hh + 1], pk[qb][4 * hh + 2], pk[qb][4 * hh + 3]};
                    acc[qb][db] = E::mfma(a, bq, acc[qb][db]);
                }
            }
        __builtin_amdgcn_sched_barrier(0);
        issue_k(i + NST, st);
    };
    split_tiles<C::UNROLL, NST>(n, tile);

    const float f = PUR ? 1.f : E::kScaleInSquare ? sc : 2.f * sc * fabsf(sc);
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        f32_wait<0>();
        __syncthreads();
        split_put<DB>(red + wave * 32 * (DP + 4), acc[qb], c, g);
        __syncthreads();
        split_store<E, DB>(red, reinterpret_cast<uint16_t*>(p.dq) + base, nullptr, m0 + 32 * qb, T, D,
                                  [&](int, f32x4 x) -> f32x4 { return x * f; });
    }
}

// ---------------------------------------------------------------------------
// dK / dV (purified: with the dgamma / dtau partials), 32 keys per workgroup.
// ---------------------------------------------------------------------------
template <class E, int DP, bool PUR>
__global__ __launch_bounds__(64 * kSplitNW) __attribute__((amdgpu_waves_per_eu(Split16Cfg<DP>::WPE)))
void born_split16_dkdv_kernel(typename std::conditional<PUR, PurArgs, BwdArgs>::type p) {
    using C = Split16Cfg<DP>;
    using Tile = Tile16<DP>;
    constexpr int KS = C::KS, DB = C::DB, NST = C::NST, NW = kSplitNW;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::SMEM];
    __shared__ __attribute__((aligned(16))) float rv_lds[NW][NST][3][32];  // -delta, 1 / Z, query ids
    __shared__ float pred[2][NW];
    __shared__ int32_t span_red[4];
    float* const red = reinterpret_cast<float*>(smem);

    const int T = p.T, D = p.D, BH = p.B * p.H;
    const int nkb = (T + 31) / 32;
    const SplitMask m = {p.is_causal != 0, p.doc != nullptr, p.window};
    const SplitBlock blk((int)blockIdx.x, (int)gridDim.x, BH, nkb, false, split_two_per_cu(C::SMEM));
    const int b = blk.bh / p.H, h = blk.bh % p.H, k0 = blk.mb * 32;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;
    const int key = k0 + c;

    const size_t base = (size_t)blk.bh * T * D;
    const uint16_t* __restrict__ Q = reinterpret_cast<const uint16_t*>(p.q) + base;
    const uint16_t* __restrict__ K = reinterpret_cast<const uint16_t*>(p.k) + base;
    const uint16_t* __restrict__ V = reinterpret_cast<const uint16_t*>(p.v) + base;
    const uint16_t* __restrict__ dO = reinterpret_cast<const uint16_t*>(p.dout) + base;
    const float* __restrict__ NDl = p.ndelta + (size_t)blk.bh * T;
    const float* __restrict__ ZIl = p.zinv + (size_t)blk.bh * T;
    const int32_t* __restrict__ docb = m.has_doc ? p.doc + (size_t)b * T : nullptr;
    const float sc = arg_scale(p, h);
    const uint32_t flip = (!PUR && sc < 0.f) ? 0x80008000u : 0u;
    const float sq_pre = (E::kScaleInSquare && sc != 0.f) ? 2.f * fabsf(sc) : 1.f;
    float pg = 0.f, pgt = 0.f, ptau = 0.f, p4g = 0.f, p2e = 0.f, pe = 0.f;
    if constexpr (PUR) {
        ptau = arg_tau(p, h);
        pg = sc;
        pgt = -sc * ptau;
        p4g = 4.f * sc;
        p2e = 2.f * p.eps_base;
        pe = p.eps_base;
    }
    float dg_acc = 0.f, dt_acc = 0.f;  // sum u^3 dP (r - tau), sum u^3 dP

    int t_lo = m.causal ? blk.mb : 0, t_hi = (T + 31) / 32 - 1;  // query tiles
    if (m.window > 0) t_hi = min(t_hi, (k0 + 31 + m.window - 1) / 32);
    if (m.has_doc) {
        const int2 sp = doc_tile_span<32>(docb, T, k0, min(T, k0 + 32), t_lo, t_hi, span_red);
        t_lo = __builtin_amdgcn_readfirstlane(sp.x);
        t_hi = __builtin_amdgcn_readfirstlane(sp.y);
    }
    const int n = t_lo <= t_hi ? (t_hi - t_lo - wave + NW) / NW : 0;

    uint8_t* const ring = smem + wave * C::RING;
    auto dt = [&](int st) { return Tile{ring + st * 2 * Tile::BYTES}; };
    auto qt = [&](int st) { return Tile{ring + st * 2 * Tile::BYTES + Tile::BYTES}; };
    uint32_t off[Tile::LOADS];
    Tile::offsets(off, D, lane);
    const i32x4 rq = split_slice(Q, T, D), rd = split_slice(dO, T, D);
    const i32x4 rnd = split_slice32(NDl, T), rzi = split_slice32(ZIl, T);
    auto row0 = [&](int i) { return i < n ? 32 * (t_lo + wave + NW * i) : T; };
    // The row values travel with dO; they are read at the tile's start.
    const i32x4 rdoc = split_slice32(docb, m.has_doc ? T : 0);
    auto issue_d = [&](int i, int st) __attribute__((always_inline)) {
        split_issue_values(rnd, row0(i), rv_lds[wave][st][0], lane);
        split_issue_values(rzi, row0(i), rv_lds[wave][st][1], lane);
        if (m.has_doc) split_issue_values(rdoc, row0(i), rv_lds[wave][st][2], lane);
        dt(st).issue(rd, off, row0(i) * D * 2);
    };
    auto issue_q = [&](int i, int st) __attribute__((always_inline)) { qt(st).issue(rq, off, row0(i) * D * 2); };

    u32x4 kr[KS], vr[KS];
    split_load_rows(kr, K, key, T, D, g);
    split_load_rows(vr, V, key, T, D, g);
    int kdoc = m.has_doc ? split_row_doc(docb, key, T) : -2;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        kr[ks] ^= flip;
        asm volatile("" : "+v"(kr[ks]), "+v"(vr[ks]));
    }
    asm volatile("" : "+v"(kdoc));
    f32x16 dv[DB], dk[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) dv[db] = zero16(), dk[db] = zero16();
#pragma unroll
    for (int i = 0; i < NST; ++i) {
        issue_d(i, i);
        issue_q(i, i);
    }

    auto tile = [&](int i, auto stage) __attribute__((always_inline)) {
        const int st = stage;
        const int i0 = row0(i);
        f32_wait<C::YOUNGER>();
        f32x16 s = zero16(), dp, zi;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 n4 = *reinterpret_cast<const f32x4*>(&rv_lds[wave][st][0][8 * j + 4 * g]);
            const f32x4 z4 = *reinterpret_cast<const f32x4*>(&rv_lds[wave][st][1][8 * j + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) dp[4 * j + e] = n4[e], zi[4 * j + e] = z4[e];
        }
        const int qdoc = m.has_doc && i0 + c < T ? __float_as_int(rv_lds[wave][st][2][c]) : -1;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) dp = E::mfma(dt(st).row(ks, c, g), vr[ks], dp);
        f32_wait<C::YOUNGER - Tile::LOADS>();  // Q: one operand's loads fewer are younger (dO's tile is still in use)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s = E::mfma(qt(st).row(ks, c, g), kr[ks], s);
        bool cut = m.cuts(i0, k0) || (PUR && (k0 + 32 > T || i0 + 32 > T));
        if (m.has_doc) {
            const int d0 = __builtin_amdgcn_readfirstlane(qdoc);
            cut = cut || __ballot(qdoc != d0 || kdoc != d0) != 0;
        }
        uint32_t w2[8], u2[8];
        split_if_cut(cut, [&](auto masked) __attribute__((always_inline)) {
            uint32_t keep = 0xffffu;
            if constexpr (masked.value) keep = split_visible<false>(m, key, kdoc, i0, qdoc, T, g);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                float ww[2], uu[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int r = 2 * j + e;
                    const bool out = masked.value && !((keep >> r) & 1u);
                    if constexpr (PUR) {
                        const float x = s[r];
                        float u = relu_f32(fmaf(x, pg, pgt)), bb = relu_f32(x);
                        if (out) u = bb = 0.f;
                        const float usq = u * u, dpz = dp[r] * zi[r], a = usq * u * dpz;
                        dg_acc = fmaf(a, x - ptau, dg_acc);
                        dt_acc += a;
                        ww[e] = fmaf(usq, usq, pe * bb * bb) * zi[r];
                        uu[e] = fmaf(p4g, usq * u, p2e * bb) * dpz;
                    } else {
                        float a = relu_f32(E::kScaleInSquare ? s[r] * sq_pre : s[r]);
                        if (out) a = 0.f;
                        const float tz = a * zi[r];
                        ww[e] = tz * a;
                        uu[e] = tz * dp[r];
                    }
                }
                w2[j] = E::pack(ww[0], ww[1]);
                u2[j] = E::pack(uu[0], uu[1]);
            }
        });
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const u32x4 bw = {w2[4 * hh], w2[4 * hh + 1], w2[4 * hh + 2], w2[4 * hh + 3]};
#pragma unroll
            for (int db = 0; db < DB; ++db) dv[db] = E::mfma(dt(st).transposed(hh, db, lane), bw, dv[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
        issue_d(i + NST, st);
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const u32x4 bu = {u2[4 * hh], u2[4 * hh + 1], u2[4 * hh + 2], u2[4 * hh + 3]};
#pragma unroll
            for (int db = 0; db < DB; ++db) dk[db] = E::mfma(qt(st).transposed(hh, db, lane), bu, dk[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
        issue_q(i + NST, st);
    };
    split_tiles<C::UNROLL, NST>(n, tile);

    const float fk = PUR ? 1.f : E::kScaleInSquare ? sc : 2.f * sc * fabsf(sc);
    const float fv = PUR ? 1.f : E::kScaleInSquare ? (sc != 0.f ? 0.25f : 0.f) : sc * sc;
    if constexpr (PUR) {
        float a = key < T ? 4.f * dg_acc : 0.f, t2 = key < T ? -4.f * sc * dt_acc : 0.f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            a += __shfl_xor(a, off);
            t2 += __shfl_xor(t2, off);
        }
        if (lane == 0) pred[0][wave] = a, pred[1][wave] = t2;
    }
    f32_wait<0>();
    __syncthreads();
    float* const mine = red + wave * 32 * (DP + 4);
    split_put<DB>(mine, dv, c, g);
    __syncthreads();
    split_store<E, DB>(red, reinterpret_cast<uint16_t*>(p.dv) + base, nullptr, k0, T, D,
                              [&](int, f32x4 x) -> f32x4 { return x * fv; });
    if constexpr (PUR) {
        if (tid == 0) {
            float a = 0.f, t2 = 0.f;
            for (int w = 0; w < NW; ++w) a += pred[0][w], t2 += pred[1][w];
            const int slot = blk.mb * BH + blk.bh;
            p.part[slot] = a;
            p.part[gridDim.x + slot] = t2;
        }
    }
    __syncthreads();
    split_put<DB>(mine, dk, c, g);
    __syncthreads();
    split_store<E, DB>(red, reinterpret_cast<uint16_t*>(p.dk) + base, nullptr, k0, T, D,
                              [&](int, f32x4 x) -> f32x4 { return x * fk; });
}

#define QDL_SPLIT16_DP(D, BODY)                      \
    switch (((D) + 31) / 32) {                       \
        case 1: { constexpr int DPV = 32; BODY } break;  \
        case 2: { constexpr int DPV = 64; BODY } break;  \
        case 3: { constexpr int DPV = 96; BODY } break;  \
        case 4: { constexpr int DPV = 128; BODY } break; \
        default: { constexpr int DPV = 256; BODY } break; \
    }

template <class E, bool PUR, class Args>
hipError_t launch_split16_fwd(const Args& a, hipStream_t st) {
    QDL_SPLIT16_DP(a.D, {
        constexpr int BM = 32 * Split16Cfg<DPV>::NQB;
        hipLaunchKernelGGL((born_split16_fwd_kernel<E, DPV, PUR>), dim3((unsigned)((a.T + BM - 1) / BM * a.B * a.H)),
                           dim3(64 * kSplitNW), 0, st, a);
    })
    return hipGetLastError();
}

// dQ first (it forms the rows' -delta and 1 / Z), then dK/dV.
template <class E, bool PUR, class Args>
hipError_t launch_split16_bwd(const Args& a, hipStream_t st) {
    QDL_SPLIT16_DP(a.D, {
        constexpr int BM = 32 * Split16Cfg<DPV>::NQB;
        hipLaunchKernelGGL((born_split16_dq_kernel<E, DPV, PUR>), dim3((unsigned)((a.T + BM - 1) / BM * a.B * a.H)),
                           dim3(64 * kSplitNW), 0, st, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((born_split16_dkdv_kernel<E, DPV, PUR>), dim3((unsigned)f32_groups(a.B, a.H, a.T)),
                           dim3(64 * kSplitNW), 0, st, a);
    })
    return hipGetLastError();
}

}  // namespace qdl
