// qr_chunk_f32.hip -- causal multi-query attention in fp32 arithmetic on fp32 MFMA tiles,
// gfx950: fp32 caches (head_dim 64, 96, 128, 256) and 16-bit caches whose pages are
// token-major (head_dim 96, 256), any whole group of up to 64 heads per kv head.
//
// Semantics as qr_chunk.hip: query i of the chunk sits at position pos0 + i and attends
// positions 0..pos0 + i (StreamingEngine.cs:831-836).  K, V, q and P all enter in fp32 and
// every product and sum is fp32, as in the decode kernels.
//
// Bound by the fp32 MFMA rate (v_mfma_f32_16x16x4_f32: 256 flop per clk and CU, 153 TFLOP/s in
// a large product).  As one decode entry per query, the path before, every query read its own
// K/V: 512 queries after 1536 positions (32 heads over 8 kv heads, head_dim 128, 15 GFLOP: 98 us
// at that rate) took 8 launches of 61 us, 506 us per call with the append; in two splits here 158
// (traced, which slows each: kernel 162, merge 7.5, append 6.6).  The matrix units are busy 77% of
// the cycles in which waves are resident (1.0 LDS conflict cycle per MFMA); the rest is the sums,
// the softmax and the tile barriers.
// Error against 64-bit results there: 2.9e-7 (decode entries 3.15e-7).
//
// A row is one (query, query head) pair.  Workgroup = 4 waves; the K/V tile of 32 positions is
// copied into LDS by buffer-load DMA (two stages) and serves 64 / PG rows:
//   PG = 1  each wave scores all 32 positions for its own 16 rows;
//   PG = 2  (few rows) two waves per 16 rows, one 16-position half of the tile each, merged
//           through LDS at the end.
// Layouts (checked on gfx950): A[m = lane%16][k = lane/16], B[k = lane/16][n = lane%16],
// D[m = 4(lane/16) + r][n = lane%16].
//   QK  S^T[pos][row]: lane (q4, l16) holds chunk 4j + q4 of K row l16 (A) and of q row l16 (B):
//       k-slot q4 of MFMA e is element e of that 16-byte chunk.  q stays in registers, scaled
//       by scale log2 e.
//   PV  O^T[dim][row]: lane quarter q4 holds the scores of positions 4q4 + r; step r takes
//       those four positions as its k-slots, so P enters from the lane's own registers.  A is
//       V row 4q4 + r, PE consecutive dims per lane: one LDS read feeds PE MFMAs.
// Sums are blocked, because an fp32 MFMA chain rounds at the size of its running sum (one chain
// over 512 positions: 9.5e-7 from 64-bit results where the decode entries have 3.1e-7).  A score is
// chains of two MFMAs (8 dims), added in pairs and then to the sum of the even or the odd steps;
// an output adds chains of two MFMAs (8 positions; four for 16-bit head_dim 256) in pairs before
// they go to the accumulator.  Distance from 64-bit results, decode entries and here: 3.15e-7 and
// 2.92e-7 at the shape above, 1.85e-7 and 1.84e-7 for 1000 queries from scratch (chains of four
// and eight MFMAs: 3.34e-7 and 2.25e-7; chains of one and two 2.90e-7 and 1.83e-7, 7% slower).
// 16-byte chunk c of an LDS row r sits at c ^ (r & SW): the 16 rows that a QK read takes lie a
// multiple of 128 bytes apart.
#include "qr_chunk.hpp"
#include "qr_mfma.hpp"

#include <algorithm>

namespace qr {
namespace {

constexpr int kTP = 32;               // positions per tile

struct ChunkF32K {
    const char* pool;
    const int* page_table;   // row of (sequence, layer)
    long long page_elems;
    long long plane_elems;
    int heads;
    int group;
    int pos0;
    int nq;
    int q_dtype;
    const void* q;           // [nq][heads][D]
    float* out;              // [nq][heads][D]
    float* part_acc;         // [nq*heads][splits][D]
    float2* part_ml;         // [nq*heads][splits]
    float qscale;            // scale * log2(e)
    int queries_per_block;
    int splits;
    int qblocks;
    int units;               // splits x qblocks x kv_heads
    int per_xcd;             // launch slots per XCD: ceil(units / 8)
};

template <typename ST, int D>
struct F32Geom {
    static constexpr int EPC = Chunk<ST>::kElems;        // cache elements per 16-byte chunk
    static constexpr int ESZ = 16 / EPC;
    static constexpr int RB = D * ESZ;                   // bytes of a row
    static constexpr int NCH = RB / 16;                  // chunks of a row
    static constexpr int SW = NCH % 8 == 0 ? 7 : 3;      // swizzle mask (a row is whole groups of SW + 1)
    static constexpr int NJ = NCH / 4;                   // QK steps (4 chunks)
    static constexpr int KB = kTP * RB;                  // bytes of a K (or V) tile
    static constexpr int NI = KB / 1024;                 // DMA loads of a K (or V) tile
    static constexpr int NIW = (NI + 3) / 4;             // of one wave
    static constexpr int PE = D % 64 == 0 ? 4 : 2;       // dims per lane and PV read
    static constexpr int NG = D / (16 * PE);             // PV reads of a row
    static_assert(NCH % 4 == 0 && KB % 1024 == 0 && D % (16 * PE) == 0, "whole steps");
    // resident workgroups per CU (one wave per SIMD each): the LDS of two stages of K and V, and
    // about 60 + D registers a lane
    // (head_dim 256: more than 256 with two M tiles, so 16-bit pages prefer position halves)
    static constexpr int kByLds = 160 * 1024 / (4 * KB);
    static constexpr int by_regs(int pg) { return D <= 64 ? 4 : D <= 128 ? 3 : pg; }
    static constexpr int wg_per_cu(int pg) { return kByLds < by_regs(pg) ? kByLds : by_regs(pg); }
};

// q elements 4 EPC j + EPC q4 + e of the row at `row`, scaled.  Element loads: the caller's q
// needs only element alignment; the dtype branch sits outside the loads.
template <int NJ, int EPC>
__device__ __forceinline__ void load_q(const void* q, int dtype, size_t row, int q4, float scale, float (&x)[NJ][EPC]) {
    if (dtype == QR_DTYPE_F32) {
        const float* f = static_cast<const float*>(q) + row;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < EPC; ++e) x[j][e] = f[4 * EPC * j + EPC * q4 + e];
    } else {
        const uint16_t* h = static_cast<const uint16_t*>(q) + row;
        const bool bf = dtype == QR_DTYPE_BF16;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < EPC; ++e) {
                const uint16_t u = h[4 * EPC * j + EPC * q4 + e];
                x[j][e] = bf ? bf16_bits_to_f32(u) : f16_bits_to_f32(u);
            }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < EPC; ++e) x[j][e] *= scale;
}

// N = 2 or 4 cache elements at p (LDS): the raw words, and widened to fp32
template <typename ST, int N> struct Elems {
    static constexpr int kWords = std::is_same<ST, float>::value ? N : N / 2;
    typedef uint32_t type __attribute__((ext_vector_type(kWords)));
    __device__ static __forceinline__ type read(const char* p) { return *reinterpret_cast<const type*>(p); }
    // a pair with the elements that are not kept cleared
    __device__ static __forceinline__ type keep(type w, bool k0, bool k1) {
        if constexpr (std::is_same<ST, float>::value) {
            if (!k0) w[0] = 0;
            if (!k1) w[1] = 0;
        } else {
            w[0] &= (k0 ? 0xFFFFu : 0u) | (k1 ? 0xFFFF0000u : 0u);
        }
        return w;
    }
    __device__ static __forceinline__ void widen(const type w, float (&o)[N]) {
        if constexpr (std::is_same<ST, float>::value) {
#pragma unroll
            for (int i = 0; i < N; ++i) o[i] = __uint_as_float(w[i]);
        } else {
#pragma unroll
            for (int i = 0; i < N / 2; ++i) {
                const uint32_t u = w[i];
                if constexpr (std::is_same<ST, BF16Tag>::value) {
                    o[2 * i] = __uint_as_float(u << 16);
                    o[2 * i + 1] = __uint_as_float(u & 0xFFFF0000u);
                } else {
                    o[2 * i] = f16_bits_to_f32(static_cast<uint16_t>(u & 0xFFFFu));
                    o[2 * i + 1] = f16_bits_to_f32(static_cast<uint16_t>(u >> 16));
                }
            }
        }
    }
};

// Sum of 1, 2 or 4 chains, pairwise.
template <int N> __device__ __forceinline__ f32x4_t chain_sum(const f32x4_t (&c)[N]) {
    if constexpr (N == 1) return c[0];
    else if constexpr (N == 2) return c[0] + c[1];
    else return (c[0] + c[1]) + (c[2] + c[3]);
}

template <typename ST, int D, int PG>
__global__ void __launch_bounds__(256, (F32Geom<ST, D>::wg_per_cu(PG))) chunk_f32_kernel(const ChunkF32K p) {
    using Gm = F32Geom<ST, D>;
    using El = Elems<ST, Gm::PE>;
    constexpr int EPC = Gm::EPC, RB = Gm::RB, NCH = Gm::NCH, SW = Gm::SW, NJ = Gm::NJ, KB = Gm::KB;
    constexpr int PE = Gm::PE, NG = Gm::NG;
    constexpr int NMT = kTP / 16 / PG;       // 16-position M tiles per wave and tile
    constexpr int RG = 4 / PG;               // row groups of 16 rows
    __shared__ __attribute__((aligned(1024))) char lds[2][2 * KB];

    // Launch slot b runs on XCD b % 8; XCD x takes contiguous units, splits fastest, then query
    // blocks, then kv heads, so the blocks of one kv head share an L2; the first half of a kv
    // head's blocks runs from the last (most keys) down, the second from the first up, so that
    // the two workgroups of a CU sum to about the same keys (as qr_chunk.hip, measured there).
    const int unit = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
    if (unit >= p.units) return;
    const int split = unit % p.splits;
    const int uq = (unit / p.splits) % p.qblocks;
    const int hq = (p.qblocks + 1) >> 1;
    const int qblk = uq < hq ? p.qblocks - 1 - uq : uq - hq;
    const int kvh = unit / (p.splits * p.qblocks);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int rw = wave % RG;
    const int ph = wave / RG;                // position half (PG = 2)
    const int q4 = lane >> 4;
    const int l16 = lane & 15;

    const int q_first = qblk * p.queries_per_block;
    const int q_last = min(p.nq, q_first + p.queries_per_block) - 1;
    const int rho = rw * 16 + l16;
    const int row_q = q_first + rho / p.group;
    const int row_h = kvh * p.group + rho % p.group;
    const bool row_on = row_q <= q_last;
    // the block's own keys spread evenly over the splits, in whole tiles
    const int keys = p.pos0 + q_last + 1;
    const int tiles = (keys + kTP - 1) / kTP;
    const int tile0 = static_cast<int>(static_cast<long long>(tiles) * split / p.splits);
    const int ntiles = static_cast<int>(static_cast<long long>(tiles) * (split + 1) / p.splits) - tile0;
    const int unmasked_end = p.pos0 + q_first + 1;  // positions below it are seen by every row

    // ---- DMA of a tile: rows past the last key lie outside the buffer range and read as zeros
    const long long kblk = static_cast<long long>(kvh) * kPageTokens * D;
    uint32_t voff[Gm::NIW];
#pragma unroll
    for (int i = 0; i < Gm::NIW; ++i) {
        const int n = 64 * (wave + 4 * i) + lane;  // LDS chunk of the tile
        const int r = n / NCH, c = n - r * NCH;
        voff[i] = static_cast<uint32_t>(r * RB + 16 * (c ^ (r & SW)));
    }
    auto page_entry = [&](int it) {  // a scalar load: no kernel writes the table while this one runs
        return reinterpret_cast<const __attribute__((address_space(4))) int*>(
            reinterpret_cast<uintptr_t>(p.page_table))[((tile0 + it) * kTP) >> kPageShift];
    };
    auto dma = [&](int it, int phys_entry) {
        const int t0 = (tile0 + it) * kTP;
        const long long phys = phys_entry;
        char* dst = lds[it & 1];
        const char* kbase =
            p.pool + (phys * p.page_elems + kblk + static_cast<long long>(t0 & (kPageTokens - 1)) * D) * Gm::ESZ;
        const int bytes = min(kTP, keys - t0) * RB;
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kbase), 0, bytes, kBufferFlags);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char*>(kbase + p.plane_elems * Gm::ESZ), 0, bytes, kBufferFlags);
#pragma unroll
        for (int i = 0; i < Gm::NIW; ++i)
            if (Gm::NI % 4 == 0 || wave + 4 * i < Gm::NI) {
                buffer_load_lds16(rk, dst + 1024 * (wave + 4 * i), voff[i], 0);
                buffer_load_lds16(rv, dst + KB + 1024 * (wave + 4 * i), voff[i], 0);
            }
    };
    if (ntiles > 0) dma(0, page_entry(0));
    int phys_pf = ntiles > 1 ? page_entry(1) : 0;

    float qv[NJ][EPC];
    load_q<NJ, EPC>(p.q, p.q_dtype, (static_cast<size_t>(row_on ? row_q : q_first) * p.heads + row_h) * D, q4, p.qscale, qv);

    f32x4_t acc[NG][PE];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int e = 0; e < PE; ++e) acc[g][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int row_lim = p.pos0 + min(row_q, q_last);  // last position the row sees
    // QK reads: chunk 4j + q4 of row l16 of an M tile at kx[j & 1] + 128 (j >> 1)
    const int half0 = ph * NMT * 16;  // first position of this wave in a tile
    int kx[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) kx[i] = (half0 + l16) * RB + 16 * ((4 * i + q4) ^ (l16 & SW));
    // PV reads: PE dims from 16 PE g + PE l16 of row 4q4 + r at vx[r] + 16 PE ESZ g
    int vx[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = half0 + 4 * q4 + r, b = l16 * PE * Gm::ESZ;
        vx[r] = KB + row * RB + 16 * ((b >> 4) ^ (row & SW)) + (b & 15);
    }

    for (int it = 0; it < ntiles; ++it) {
        const int t0 = (tile0 + it) * kTP;
        wait_dma();     // this wave's part of tile `it` has landed
        lds_barrier();  // everyone's has, and the stage refilled next was consumed
        if (it + 1 < ntiles) {
            dma(it + 1, phys_pf);
            if (it + 2 < ntiles) phys_pf = page_entry(it + 2);
        }
        const char* const base = lds[it & 1];

        // ---- scores: the K chunks of step jj + 1 are read before the MFMAs of step jj, whose
        // partial sums are added during step jj + 1
        f32x4_t sc[NMT];
        {
            constexpr int NC = EPC / 2;  // chains of two MFMAs
            U32x4 raw[2][NMT];
            f32x4_t part[2][NMT][NC], sum[2][NMT];
            auto add = [&](int jj) __attribute__((always_inline)) {  // step jj's chains to the sum of its parity
#pragma unroll
                for (int mt = 0; mt < NMT; ++mt) {
                    const f32x4_t s = chain_sum<NC>(part[jj & 1][mt]);
                    sum[jj & 1][mt] = jj < 2 ? s : sum[jj & 1][mt] + s;
                }
            };
            auto kread = [&](int jj) __attribute__((always_inline)) {
#pragma unroll
                for (int mt = 0; mt < NMT; ++mt) raw[jj & 1][mt] = load16(base + kx[jj & 1] + 128 * (jj >> 1) + 16 * mt * RB);
            };
            kread(0);
#pragma unroll
            for (int jj = 0; jj < NJ; ++jj) {
                if (jj + 1 < NJ) kread(jj + 1);
                __builtin_amdgcn_sched_barrier(0);
                float kv[NMT][EPC];
#pragma unroll
                for (int mt = 0; mt < NMT; ++mt) {
                    Chunk<ST>::widen(raw[jj & 1][mt], kv[mt]);
#pragma unroll
                    for (int c = 0; c < NC; ++c) part[jj & 1][mt][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int e = 0; e < EPC; ++e) {
                    if (jj > 0 && e == EPC / 2) {
                        __builtin_amdgcn_sched_barrier(0);
                        add(jj - 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int mt = 0; mt < NMT; ++mt)
                        part[jj & 1][mt][e % NC] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(kv[mt][e], qv[jj][e], part[jj & 1][mt][e % NC], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            add(NJ - 1);
#pragma unroll
            for (int mt = 0; mt < NMT; ++mt) sc[mt] = sum[0][mt] + sum[1][mt];
        }

        // ---- causal mask, only on tiles that reach past the block's first query (the keys'
        // end lies past every row's own limit)
        const bool edge = t0 + kTP > unmasked_end;
        bool bad = false;  // a V element of an edge tile is not finite
        if (edge) {
#pragma unroll
            for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    sc[mt][r] = t0 + half0 + 16 * mt + 4 * q4 + r <= row_lim ? sc[mt][r] : -INFINITY;
            // the whole tile, so that every wave finds the same; V times zero is zero or NaN
            float z = 0.f;
#pragma unroll 4
            for (int i = 0; i < kTP * NCH / 64; ++i) {
                float v[EPC];
                Chunk<ST>::widen(load16(base + KB + 16 * (lane + 64 * i)), v);
#pragma unroll
                for (int e = 0; e < EPC; ++e) z = fmaf(v[e], 0.f, z);
            }
            bad = __builtin_amdgcn_ballot_w64(!(z == 0.f)) != 0;
        }

        // ---- online softmax.  The maximum does not lag, so that P <= 1 as in the decode kernels: a V
        // of more than 2^120 would overflow under P <= 256.
        float tm = -INFINITY;
#pragma unroll
        for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) tm = fmaxf(tm, sc[mt][r]);
        tm = max_xor32(max_xor16(tm));
        const bool grow = tm > m;
        const bool rescale = grow && m != -INFINITY;
        if (__builtin_amdgcn_ballot_w64(rescale)) {
            const float corr = rescale ? fast_exp2(m - tm) : 1.f;
            l *= corr;
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int e = 0; e < PE; ++e) acc[g][e] *= corr;
        }
        if (grow) m = tm;
        const float mref = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[mt][r] = fast_exp2(sc[mt][r] - mref);
        f32x4_t ls = sc[0];
#pragma unroll
        for (int mt = 1; mt < NMT; ++mt) ls += sc[mt];
        l += (ls[0] + ls[1]) + (ls[2] + ls[3]);

        if (bad) {
            // A row must not meet the V of a position that it does not see: 0 x inf is NaN.  The
            // elements that are not finite are added here, only where the row sees their position
            // (rare), and cleared for the products below.
#pragma unroll 1
            for (int k = 0; k < NMT * 16; ++k) {  // position 16 (k / 16) + 4 ((k / 4) % 4) + k % 4
                const int pos = half0 + k;
                float own = 0.f;
#pragma unroll
                for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) own = (k >> 4) == mt && (k & 3) == r ? sc[mt][r] : own;
                const float w = __shfl(own, 16 * ((k >> 2) & 3) + l16, 64);
                const bool see = t0 + pos <= row_lim;
#pragma unroll
                for (int g = 0; g < NG; ++g) {
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const int b = (16 * g + 4 * q4 + rr) * PE * Gm::ESZ;
                        float v[PE];
                        El::widen(El::read(base + KB + pos * RB + 16 * ((b >> 4) ^ (pos & SW)) + (b & 15)), v);
#pragma unroll
                        for (int e = 0; e < PE; ++e)
                            if (see && !(fabsf(v[e]) < INFINITY)) acc[g][e][rr] = fmaf(w, v[e], acc[g][e][rr]);
                        asm volatile("" ::: "memory");  // no registers for all reads at once
                    }
                }
            }
            lds_barrier();  // every wave has read them
            for (int c = threadIdx.x; c < kTP * NCH; c += 256) {
                typedef typename Elems<ST, 2>::type Pair;
#pragma unroll
                for (int i = 0; i < EPC / 2; ++i) {
                    Pair* const w = reinterpret_cast<Pair*>(const_cast<char*>(base) + KB + 16 * c) + i;
                    float v[2];
                    Elems<ST, 2>::widen(*w, v);
                    const bool b0 = !(fabsf(v[0]) < INFINITY), b1 = !(fabsf(v[1]) < INFINITY);
                    if (b0 || b1) *w = Elems<ST, 2>::keep(*w, !b0, !b1);
                }
            }
            lds_barrier();
        }

        // ---- weighted sum of V (step st = 4 mt + r of dim group g; V read two steps ahead)
        constexpr int CL = D == 256 && EPC == 8 ? 4 : 2;  // steps of a chain
        constexpr int NS = 4 * NMT, NC = NS / CL, NO = NC + 1;
        typename El::type vb[3];
        auto vread = [&](int i) __attribute__((always_inline)) {
            const int g = i / NS, st = i % NS;
            vb[i % 3] = El::read(base + vx[st & 3] + 16 * (st >> 2) * RB + 16 * PE * Gm::ESZ * g);
        };
        vread(0);
        vread(1);
        f32x4_t o[NO][PE];  // chain c of group g in o[(NC g + c) % NO]: the next group's first chain leaves g's alone
        auto add = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < PE; ++e) {
                f32x4_t s[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) s[c] = o[(NC * g + c) % NO][e];
                acc[g][e] += chain_sum<NC>(s);
            }
        };
#pragma unroll
        for (int g = 0; g < NG; ++g) {
#pragma unroll
            for (int st = 0; st < NS; ++st) {
                const int i = NS * g + st, c = i / CL % NO;
                if (st % CL == 0) {
#pragma unroll
                    for (int e = 0; e < PE; ++e) o[c][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                }
                if (i + 2 < NS * NG) vread(i + 2);
                __builtin_amdgcn_sched_barrier(0);
                float v[PE];
                El::widen(vb[i % 3], v);
#pragma unroll
                for (int e = 0; e < PE; ++e)
                    o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], sc[st >> 2][st & 3], o[c][e], 0, 0, 0);
                if (g > 0 && st == 1) add(g - 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        add(NG - 1);
    }
    l = sum_xor32(sum_xor16(l));

    if constexpr (PG == 2) {
        // the upper halves hand (m, l, o) to the lower ones through LDS
        constexpr int NA = NG * PE;
        static_assert(RG * 64 * (NA * 16 + 8) <= 4 * KB, "the handed-over rows fit the tile buffers");
        f32x4_t* xo = reinterpret_cast<f32x4_t*>(lds[0]) + rw * NA * 64 + lane;
        float2* xm = reinterpret_cast<float2*>(lds[0] + RG * NA * 64 * 16) + rw * 64 + lane;
        __syncthreads();
        if (ph == 1) {
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int e = 0; e < PE; ++e) xo[(g * PE + e) * 64] = acc[g][e];
            *xm = make_float2(m, l);
        }
        __syncthreads();
        if (ph == 1) return;
        const float2 o = *xm;
        const float M = fmaxf(m, o.x);
        const float c0 = m == -INFINITY ? 0.f : fast_exp2(m - M);
        const float c1 = o.x == -INFINITY ? 0.f : fast_exp2(o.x - M);
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int e = 0; e < PE; ++e) acc[g][e] = acc[g][e] * c0 + xo[(g * PE + e) * 64] * c1;
        l = l * c0 + o.y * c1;
        m = M;
    }

    // lane (q4, l16) holds dims 16 PE g + PE (4q4 + r) + e of row l16 in acc[g][e][r]
    if (!row_on) return;
    const size_t r0 = static_cast<size_t>(row_q) * p.heads + row_h;
    const size_t slot = r0 * p.splits + split;
    const float by = p.splits == 1 ? 1.f / l : 1.f;
    float* o = (p.splits == 1 ? p.out + r0 * D : p.part_acc + slot * D) + 4 * PE * q4;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int e = 0; e < PE; ++e) {
                const float a = acc[g][e][r];
                float x = a * by;
                if (p.splits == 1 && fabsf(x) < INFINITY) x = fmaf(fmaf(-x, l, a), by, x);  // a / l to the last bit or so
                o[16 * PE * g + PE * r + e] = x;
            }
    if (p.splits > 1 && q4 == 0) p.part_ml[slot] = make_float2(m, l);
}

// Merge of the splits: D / 4 threads per (query, head) row, 4 dims each; the (max, sum) pairs
// of up to 8 splits and their partials are loaded at once.
template <int D>
__global__ void __launch_bounds__(256) chunk_f32_combine_kernel(const ChunkF32K p, long long rows) {
    constexpr int TPR = D / 4, RPB = 256 / TPR;
    const int rr = threadIdx.x / TPR;
    const long long r = static_cast<long long>(blockIdx.x) * RPB + rr;
    if (rr >= RPB || r >= rows) return;
    const int c = threadIdx.x - rr * TPR;
    const size_t base = static_cast<size_t>(r) * p.splits;
    const f32x4_t* part = reinterpret_cast<const f32x4_t*>(p.part_acc) + c;
    constexpr int kB = 8;
    float m = -INFINITY, l = 0.f;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < p.splits; s0 += kB) {
        f32x4_t a[kB];
        float2 ml[kB];
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            const int s = min(s0 + i, p.splits - 1);
            a[i] = part[(base + s) * TPR];
            ml[i] = p.part_ml[base + s];
        }
        float mb = m;
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            if (s0 + i >= p.splits) ml[i] = make_float2(-INFINITY, 0.f);  // a repeated split
            mb = fmaxf(mb, ml[i].x);
        }
        const float cm = m == -INFINITY ? 0.f : fast_exp2(m - mb);
        l *= cm;
        o *= cm;
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            const float w = ml[i].x == -INFINITY ? 0.f : fast_exp2(ml[i].x - mb);
            l = fmaf(ml[i].y, w, l);
            if (s0 + i < p.splits) o += a[i] * w;
        }
        m = mb;
    }
    float* out = p.out + static_cast<size_t>(r) * D + 4 * c;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = o[e] / l;
}

int cu_count() {
    static int n = 0;
    if (n == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
            n = prop.multiProcessorCount;
        if (n <= 0) n = 256;
    }
    return n;
}

int wgs_per_cu(int kv_dtype, int D, int pg) {
    if (kv_dtype != QR_DTYPE_F32) return D == 96 ? F32Geom<F16Tag, 96>::wg_per_cu(pg) : F32Geom<F16Tag, 256>::wg_per_cu(pg);
    switch (D) {
        case 64: return F32Geom<float, 64>::wg_per_cu(pg);
        case 96: return F32Geom<float, 96>::wg_per_cu(pg);
        case 128: return F32Geom<float, 128>::wg_per_cu(pg);
        default: return F32Geom<float, 256>::wg_per_cu(pg);
    }
}

template <typename ST, int D>
hipError_t launch_geom(const ChunkF32K& k, const ChunkPlan& pl, hipStream_t s, hipEvent_t after_split) {
    const dim3 grid(8 * k.per_xcd);
    if (pl.pg == 2) hipLaunchKernelGGL((chunk_f32_kernel<ST, D, 2>), grid, dim3(256), 0, s, k);
    else hipLaunchKernelGGL((chunk_f32_kernel<ST, D, 1>), grid, dim3(256), 0, s, k);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (after_split && (e = hipEventRecord(after_split, s)) != hipSuccess) return e;
    if (pl.splits == 1) return hipSuccess;
    const long long rows = static_cast<long long>(k.nq) * k.heads;
    constexpr int RPB = 256 / (D / 4);
    hipLaunchKernelGGL((chunk_f32_combine_kernel<D>), dim3(static_cast<unsigned>((rows + RPB - 1) / RPB)), dim3(256), 0, s,
                       k, rows);
    return hipGetLastError();
}

}  // namespace

bool chunk_f32_eligible(int kv_dtype, int head_dim, int heads, int kv_heads, int pos0, int nq) {
    if (heads % kv_heads || heads / kv_heads > 64) return false;
    if (nq < 2 || static_cast<long long>(nq) * (heads / kv_heads) < kChunkF32MinRows) return false;
    const bool f32 = kv_dtype == QR_DTYPE_F32;
    if (head_dim != 96 && head_dim != 256 && !(f32 && (head_dim == 64 || head_dim == 128))) return false;
    // More than 64 queries took several decode launches (128 from scratch, 32 heads over 8: 21.4 us
    // against 16.0 here).  Few queries over few keys: one launch of up to 64 entries, merged in the
    // kernel, costs less than this kernel and its merge.  The lines are by the K/V bytes that the
    // entries would read themselves (us as entries and here, the append included):
    //   32 to 64 queries, two heads per kv head: 200 MB 16.0 and 19.4 (64 after 349, head_dim 128), 300
    //   MB 18.2 and 19.5 or ahead; three: 200 MB 21.8 and 25.1; four and more: 100 MB 16.4 and 19.2, 140
    //   ahead; head_dim 256, two heads: 200 MB 23.5 and 35.0, 300 MB 28.7 and 31.7 in fp32, 140 MB 29.0
    //   and 30.5 in 16 bits;
    //   fewer: 66 MB 18.7 and 19.8 (4 after 2000), 197 MB 29.6 and 26.9; very few rows leave CUs idle
    //   here (4 queries of 8 heads over 1 after 48826: 34.0 and 36.6, head_dim 64);
    //   one head per kv head, where the entries do a third of the work per byte: 64 after 400 (226 MB)
    //   17.2 and 20.7 (head_dim 128), 32 after 1000 (266 MB) 17.8 and 19.8 (64), 16 after 2000 (263 MB)
    //   21.7 and 20.2; at head_dim 256, where two launches are still ahead, 64 after 300 (174 MB in 16
    //   bits, 8 heads) 23.8 and 27.7, 32 after 500 (271 MB, 16 heads) 30.3 and 30.8, 65 after 100 (141
    //   MB in fp32) 27.9 and 32.9, 64 after 400 (453 MB in fp32) 28.9 and 31.8.
    // The entries of head_dim 96 are slower (4 queries after 500, 32 heads over 8: 25.8 and 18.8); with
    // one head per kv head they are ahead over few keys (32 after 300 16.3 and 18.4, 8 after 500 16.9
    // and 18.9, 8 after 2000 26.9 and 18.7).
    const int g = heads / kv_heads;
    if (head_dim == 96) return nq > 64 || g > 1 || pos0 + nq > 540;
    if (nq > (g == 1 && head_dim == 256 ? 128 : 64)) return true;
    if (head_dim < 256 && nq * heads < 64) return false;
    const bool wide32 = head_dim == 256 && f32;
    double line = 96e6;
    if (g == 1) line = wide32 ? 500e6 : 280e6;
    else if (nq >= 32) line = g == 2 ? (wide32 ? 350e6 : head_dim == 256 ? 200e6 : 300e6) : g == 3 ? 210e6 : 140e6;
    const double bytes = 2.0 * nq * (pos0 + 0.5 * nq) * kv_heads * head_dim * (f32 ? 4 : 2);
    return bytes >= line;
}

ChunkPlan plan_chunk_f32(const ChunkArgs& a) {
    const int g = a.heads / a.geom.kv_heads, D = a.geom.head_dim;
    const long long rows = static_cast<long long>(a.nq) * a.heads;
    const int tiles = (a.pos0 + a.nq + kTP - 1) / kTP;
    ChunkPlan best{};
    double best_cost = 0;
    // Position halves and splits of the keys by the time of the matrix work plus the partials'
    // traffic (written and read once, about 4 TB/s) and the merge's launch.  A tile of 64 rows and
    // 32 positions is 32 D cycles of a CU's matrix units; with w workgroups resident a tile of each
    // takes 0.8 (w + 1) of that (a workgroup alone leaves the units idle in its softmax and
    // barriers, several overlap), position halves 0.65 of it instead of a half (a barrier per half
    // the work).  Query blocks of like lengths (many keys before them) run in whole rounds of the
    // longest; blocks from scratch mix, so they take the mean length.  Over 163 shapes the choice
    // took 2.6% more than the fastest of up to ten (by whole occupancy rounds alone 7.9%).  At the
    // shape above 64 rows in 1, 2, 3 and 4 splits 193, 158, 195 and 164 us with the append, halves in
    // 1 and 2 163 and 177; 1059 queries from scratch at head_dim 64: 64 rows 91, halves 68; 512 after
    // 1536 at head_dim 256 in 16 bits: 64 rows 468, halves 346.
    // Splits are for units that leave CUs idle: no more of them than fill the CUs four times over,
    // which bounds the partials too (4 x 768 workgroups x 64 rows of head_dim 96: 77 MB).
    const int cus = cu_count();
    const double like = static_cast<double>(a.pos0) / (a.pos0 + a.nq);  // 0 from scratch
    auto tile_cost = [](double w) { return 0.8 * (w + 1.0); };
    for (int pg = 1; pg <= 2; ++pg) {
        const int per_cu = wgs_per_cu(a.kv_dtype, D, pg), slots = cus * per_cu;
        const int wg_rows = 64 / pg;
        if (wg_rows < g) continue;
        const int qpb = wg_rows / g, qblocks = (a.nq + qpb - 1) / qpb;
        const long long units = static_cast<long long>(qblocks) * a.geom.kv_heads;
        const double tile_us = 32.0 * D / 2400 * (pg == 2 ? 0.65 : 1.0);
        const int smax = std::min(64, std::max(1, tiles / 4));
        auto bytes = [&](int s) { return static_cast<size_t>(rows) * s * (static_cast<size_t>(D) * 4 + 8); };
        for (int s = 1; s <= smax && (s == 1 || (units * s <= 4LL * slots && bytes(s) <= a.room)); ++s) {
            const long long full = units * s / slots, rest = units * s % slots;
            const double longest = (tiles + s - 1) / s + 1.0;
            const double mean = (a.pos0 + 0.5 * a.nq) / kTP / s + 1.0;
            const double per = static_cast<double>(units) * s / cus, w = std::min<double>(per_cu, std::max(1.0, per));
            const double rounds = (full * tile_cost(per_cu) + (rest ? tile_cost((rest + cus - 1) / cus) : 0.0)) * longest;
            const double mixed = std::max(longest * tile_cost(1), per * mean * tile_cost(w) / w);
            const double traffic = s > 1 ? 5.0 + static_cast<double>(rows) * s * D * 8 / 4e6 : 0.0;
            const double cost = (like * rounds + (1.0 - like) * mixed) * tile_us + traffic;
            if (best.splits == 0 || cost < best_cost) {
                best_cost = cost;
                best.nt = 1;
                best.pg = pg;
                best.queries_per_block = qpb;
                best.qblocks = qblocks;
                best.splits = s;
            }
        }
    }
    best.workspace_bytes = best.splits > 1 ? static_cast<size_t>(rows) * best.splits * (static_cast<size_t>(D) * 4 + 8) : 0;
    return best;
}

hipError_t launch_chunk_f32(const ChunkArgs& a, const ChunkPlan& pl, void* workspace, hipStream_t stream,
                            hipEvent_t after_split) {
    ChunkF32K k{};
    k.pool = static_cast<const char*>(a.pool);
    k.page_table = a.page_table;
    k.page_elems = a.geom.page_elems();
    k.plane_elems = a.geom.plane_elems();
    k.heads = a.heads;
    k.group = a.heads / a.geom.kv_heads;
    k.pos0 = a.pos0;
    k.nq = a.nq;
    k.q_dtype = a.q_dtype;
    k.q = a.q;
    k.out = a.out;
    k.part_acc = static_cast<float*>(workspace);
    k.part_ml = reinterpret_cast<float2*>(static_cast<char*>(workspace) +
                                          static_cast<size_t>(a.nq) * a.heads * pl.splits * a.geom.head_dim * 4);
    k.qscale = static_cast<float>(static_cast<double>(a.scale) * 1.4426950408889634);
    k.queries_per_block = pl.queries_per_block;
    k.splits = pl.splits;
    k.qblocks = pl.qblocks;
    k.units = pl.splits * pl.qblocks * a.geom.kv_heads;
    k.per_xcd = (k.units + 7) / 8;
    if (a.kv_dtype == QR_DTYPE_F32) {
        switch (a.geom.head_dim) {
            case 64: return launch_geom<float, 64>(k, pl, stream, after_split);
            case 96: return launch_geom<float, 96>(k, pl, stream, after_split);
            case 128: return launch_geom<float, 128>(k, pl, stream, after_split);
            default: return launch_geom<float, 256>(k, pl, stream, after_split);
        }
    }
    if (a.kv_dtype == QR_DTYPE_BF16)
        return a.geom.head_dim == 96 ? launch_geom<BF16Tag, 96>(k, pl, stream, after_split)
                                     : launch_geom<BF16Tag, 256>(k, pl, stream, after_split);
    return a.geom.head_dim == 96 ? launch_geom<F16Tag, 96>(k, pl, stream, after_split)
                                 : launch_geom<F16Tag, 256>(k, pl, stream, after_split);
}

}  // namespace qr
