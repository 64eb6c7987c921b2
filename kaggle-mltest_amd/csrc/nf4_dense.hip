// Plain 16-bit GEMM on gfx950 for the products whose token count pays for dequantizing the
// weight once into a workspace (the exact 16-bit weight the fused kernels multiply with), and
// the transposing dequantization that the input gradient's reduction over the weight's rows
// needs.  Both operands have the reduction contiguous: forward W [N, K] and X [M, K], input
// gradient W^T [K, N] and dY [M, N].

#include <cmath>

#include "nf4_dense.h"

namespace {

constexpr int HALF = 128 * 128;  // bytes of one staged half tile: 128 rows x 64 values
constexpr int kLds = 8 * HALF;   // 128 KB: two steps of a 256x256 tile, four of a 128x128 tile

template <int DT>
__device__ __forceinline__ float widen(uint32_t v) {
    if constexpr (DT == NF4_BF16) return __uint_as_float(v << 16);
    else return static_cast<float>(__builtin_bit_cast(half_t, static_cast<uint16_t>(v)));
}

// Values 0 .. 7 (zero from `lim` on) of a LoRA row, `step` elements apart.
__device__ __forceinline__ u32x4_t slab8(const uint16_t *row, int64_t step, int lim, int vec) {
    if (lim <= 0) return (u32x4_t){0u, 0u, 0u, 0u};
    if (vec && lim >= 8) return *reinterpret_cast<const u32x4_t *>(row);
    uint32_t e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = j < lim ? row[j * step] : 0;
    return (u32x4_t){e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
}

// A barrier that nothing is scheduled across (the LDS DMA is inline assembly, which the
// compiler's own waits do not cover).
__device__ __forceinline__ void segment_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// One tile of 128 HP rows p x 128 HM rows m, by 8 waves: wave (wp, wm) = (wave / 4, wave % 4)
// owns rows 64 wp .. + 63 of every p half and rows 32 wm .. + 31 of every m half.
//
// Bound: the matrix unit at the clock that the power cap leaves under random operands (a
// register-only MFMA loop reaches 1.68 PFLOP/s on this card, this kernel 1.24 (fp16) to 1.39
// (bf16) at M = N = K = 8192).  A SIMD's two waves (w, w + 4) alternate: while one wave's 16
// MFMAs of a segment run, the other reads its next fragments from LDS and issues its share of the next
// steps' DMA, then both cross a barrier and swap; waves 4-7 start one segment late.  One
// segment per m-half pair (HP segments per 64-deep step): four segments of 8 MFMAs, each with
// its own barriers, measured the same, one segment of 32 spills.  The operands arrive by
// 16-byte LDS DMA, up to two steps (256x256) or three (128x128) ahead, so that a step waits for nothing
// younger than one step.
//
// LDS half tile: 128 rows of 128 bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7): the 16
// rows of one fragment read pass hit distinct banks.
template <int DT, int HP, int HM>
__device__ __forceinline__ void dense_tile(const DenseArgs &a, uint8_t *lds, int64_t p0, int64_t m0,
                                           int u0, int u1, int split) {
    static_assert((HP == 2 && HM == 2) || (HP == 1 && HM == 1), "square tiles");
    constexpr int BUF = (HP + HM) * HALF;  // one step: p halves, then m halves
    constexpr int NB = kLds / BUF;
    const int lane = threadIdx.x & 63, r32 = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wp = wave >> 2, wm = wave & 3;

    // rows past an operand read as zero (buffer range check)
    auto window = [](const uint16_t *base, int64_t row, int64_t rows, int64_t ld, int64_t cols) {
        const int64_t n = rows - row < 128 ? rows - row : 128;
        return make_rsrc(base + (n > 0 ? row * ld : 0), n > 0 ? ((n - 1) * ld + cols) * 2 : 0);
    };
    const rsrc_t rx0 = window(a.act, m0, a.M, a.ld_act, a.R), rx1 = window(a.act, m0 + 128, a.M, a.ld_act, a.R);
    const int64_t strip = a.R * 256;  // bytes of 128 rows p
    const uint8_t *ws = reinterpret_cast<const uint8_t *>(a.w) + p0 / 128 * strip;
    const rsrc_t rw0 = make_rsrc(ws, strip), rw1 = make_rsrc(ws + strip, p0 + 128 < a.P ? strip : 0);
    int wo[2], xo[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // this wave's two blocks of 8 rows of a half
        const int row = (wave * 2 + j) * 8 + (lane >> 3);
        wo[j] = (wave * 2 + j) * 1024 + lane * 16;  // (the strips hold LDS images)
        xo[j] = row * static_cast<int>(a.ld_act) * 2 + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    }
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t *)lds)) +
        wave * 2048;
    auto send = [&](const rsrc_t &rs, const int (&o)[2], int half, int u) {
        const int kb = (u < u1 ? u : u1 - 1) * (half < HP ? HALF : 128);  // past the end: a reload nobody reads
        const uint32_t base = __builtin_amdgcn_readfirstlane(lds0 + ((u - u0) % NB) * BUF + half * HALF);
        lds_dma16(base, o[0], rs, kb);
        lds_dma16(base + 1024, o[1], rs, kb);
    };
    auto w0 = [&](int u) { send(rw0, wo, 0, u); };
    auto w1 = [&](int u) { send(rw1, wo, 1, u); };
    auto x0 = [&](int u) { send(rx0, xo, HP, u); };
    auto x1 = [&](int u) { send(rx1, xo, HP + 1, u); };

    float16_t acc[HP][HM][2];  // [p half][m half][32-row fragment of the wave's 64 rows]
#pragma unroll
    for (int h = 0; h < HP; ++h)
#pragma unroll
        for (int g = 0; g < HM; ++g) acc[h][g][0] = acc[h][g][1] = (float16_t){};

    int fo[4];  // fragment of k-substep ks inside a 32-row block
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) fo[ks] = r32 * 128 + (((ks * 2 + kh) ^ ((r32 >> 1) & 7)) << 4);
    const uint8_t *lw = lds + wp * 8192, *lx = lds + HP * HALF + wm * 4096;
    u32x4_t fw[2][4], fx[HM][4];
    auto read_w = [&](int b, int h) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fw[i][ks] = *reinterpret_cast<const u32x4_t *>(lw + b * BUF + h * HALF + i * 4096 + fo[ks]);
    };
    auto read_x = [&](int b) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int g = 0; g < HM; ++g)
                fx[g][ks] = *reinterpret_cast<const u32x4_t *>(lx + b * BUF + g * HALF + fo[ks]);
    };
    auto mma = [&](float16_t (&c)[HM][2]) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int g = 0; g < HM; ++g)
#pragma unroll
                for (int i = 0; i < 2; ++i) c[g][i] = mfma32<DT>(fw[i][ks], fx[g][ks], c[g][i]);
    };

    // A segment ends with this wave's fragment reads complete (so the next segment's DMA of
    // either wave group may overwrite what was read) and with its DMA of what the next segment
    // reads arrived; the barrier then makes that true of every wave.  Loads return in order:
    // vmcnt(N) leaves the N youngest in flight.
    if constexpr (HP == 2) {
        // in flight, oldest first: p half 0 and both m halves of step u, p half 1 of u, ...
        w0(u0), x0(u0), x1(u0), w1(u0), w0(u0 + 1), x0(u0 + 1);
        asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        segment_barrier();
        if (wp == 1) segment_barrier();  // waves 4-7 run one segment behind
        auto step = [&](int u, int b) {
            read_x(b), read_w(b, 0), x1(u + 1), w1(u + 1);
            asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");  // p half 1 of step u
            segment_barrier();
            mma(acc[0]);
            segment_barrier();
            read_w(b, 1), w0(u + 2), x0(u + 2);
            asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");  // the rest of step u + 1
            segment_barrier();
            mma(acc[HP - 1]);
            segment_barrier();
        };
        int u = u0;
        for (; u + 1 < u1; u += 2) step(u, 0), step(u + 1, 1);
        if (u < u1) step(u, 0);
    } else {
        w0(u0), x0(u0), w0(u0 + 1), x0(u0 + 1), w0(u0 + 2), x0(u0 + 2);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        segment_barrier();
        if (wp == 1) segment_barrier();
        auto step = [&](int u, int b) {
            read_x(b), read_w(b, 0), w0(u + 3), x0(u + 3);
            asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");  // step u + 1
            segment_barrier();
            mma(acc[0]);
            segment_barrier();
        };
        int u = u0;
        for (; u + 3 < u1; u += 4) step(u, 0), step(u + 1, 1), step(u + 2, 2), step(u + 3, 3);
        if (u < u1) step(u, 0);
        if (u + 1 < u1) step(u + 1, 1);
        if (u + 2 < u1) step(u + 2, 2);
    }
    if (wp == 0) segment_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    segment_barrier();  // no DMA in flight, no fragment read outstanding: the LDS is free

    // LoRA terms (of a split tile: split 0), 16 ranks at a time: the threads of waves 0-3 bring a
    // row p of the left operand each (dX: A's ranks are rows K apart, so the wave's loads of one
    // rank coalesce), those of waves 4-7 a row m of the right one, 32 bytes per LDS row.
    // Rows p outside the slab take nothing, not even 0 * t, which is NaN where a token's t is not
    // finite: a word per row masks the products (selects on the row index spill)
    for (int s = 0; s < (split > 0 ? 0 : a.nslab); ++s) {
        const DenseSlab &sl = a.slab[s];
        if (sl.p_hi <= p0 || sl.p_lo >= p0 + 128 * HP) continue;
        for (int k0 = 0; k0 < sl.rank; k0 += 16) {
            const int r = threadIdx.x & 255, lim = sl.rank - k0;
            if (r < 128 * HP) {
                const bool left = wave < 4;
                const int64_t row = (left ? p0 : m0) + r;
                const bool in = left ? row >= sl.p_lo && row < sl.p_hi : row < a.M;
                const uint16_t *src = left ? sl.l + (in ? row - sl.p_lo : 0) * sl.lp + k0 * sl.lr
                                           : sl.t + (in ? row : 0) * sl.rank + k0;
                const int64_t step = left ? sl.lr : 1;
                const int vec = left ? sl.vec_l : sl.vec_t;
                u32x4_t *dst = reinterpret_cast<u32x4_t *>(lds + (left ? 0 : 256 * 32) + r * 32);
                dst[0] = slab8(src, step, in ? lim : 0, vec);
                dst[1] = slab8(src + 8 * step, step, in ? lim - 8 : 0, vec);
                if (left) *reinterpret_cast<uint32_t *>(lds + 512 * 32 + r * 4) = in ? ~0u : 0u;
            }
            __syncthreads();
#pragma unroll
            for (int h = 0; h < HP; ++h)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const u32x4_t fl = *reinterpret_cast<const u32x4_t *>(
                        lds + (h * 128 + wp * 64 + i * 32 + r32) * 32 + kh * 16);
                    u32x4_t mask[4];
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4)
                        mask[r4] = *reinterpret_cast<const u32x4_t *>(
                            lds + 512 * 32 + (h * 128 + wp * 64 + i * 32 + r4 * 8 + kh * 4) * 4);
#pragma unroll
                    for (int g = 0; g < HM; ++g) {
                        const u32x4_t ft = *reinterpret_cast<const u32x4_t *>(
                            lds + 256 * 32 + (g * 128 + wm * 32 + r32) * 32 + kh * 16);
                        const float16_t v = sl.scale * mfma32<DT>(fl, ft, (float16_t){});
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            acc[h][g][i][e] += __uint_as_float(__float_as_uint(v[e]) & mask[e / 4][e % 4]);
                    }
                }
            __syncthreads();
        }
    }

    if (split >= 0) {
        // fp32 partials of one m half at a time: row m of 256 floats, 4-float chunk c at c ^ (m % 32)
        if constexpr (HP == 2) {
            const int c = threadIdx.x & 63;
            const int64_t p = p0 + 4 * c;
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int ml = wm * 32 + r32;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int r4 = 0; r4 < 4; ++r4) {
                            const int q = (h * 128 + wp * 64 + i * 32 + r4 * 8 + kh * 4) >> 2;
                            const float16_t &v = acc[h][g][i];
                            *reinterpret_cast<float4_t *>(lds + ml * 1024 + ((q ^ (ml & 31)) << 4)) =
                                (float4_t){v[r4 * 4], v[r4 * 4 + 1], v[r4 * 4 + 2], v[r4 * 4 + 3]};
                        }
                __syncthreads();
#pragma unroll 4
                for (int m = threadIdx.x >> 6; m < 128; m += 8) {
                    const int64_t gm = m0 + g * 128 + m;
                    if (gm >= a.M || p >= a.P) continue;
                    *reinterpret_cast<float4_t *>(a.partial + (split * a.M + gm) * a.P + p) =
                        *reinterpret_cast<const float4_t *>(lds + m * 1024 + ((c ^ (m & 31)) << 4));
                }
                __syncthreads();
            }
        }
        return;
    }

    // 16-bit output through LDS: row m of 128 HP values, 8-value chunk c at c ^ (m % (16 HP)),
    // then whole 16-byte stores
    constexpr int CPR = 16 * HP, RB = 256 * HP;
#pragma unroll
    for (int h = 0; h < HP; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const int p = h * 128 + wp * 64 + i * 32 + r4 * 8 + kh * 4;
                float bv[4] = {0.f, 0.f, 0.f, 0.f};
                if (a.bias) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (p0 + p + q < a.P) bv[q] = widen<DT>(a.bias[p0 + p + q]);
                }
#pragma unroll
                for (int g = 0; g < HM; ++g) {
                    const int m = g * 128 + wm * 32 + r32;
                    const float16_t &v = acc[h][g][i];
                    u32x2_t o;
                    o.x = pack2<DT>(v[r4 * 4] + bv[0], v[r4 * 4 + 1] + bv[1]);
                    o.y = pack2<DT>(v[r4 * 4 + 2] + bv[2], v[r4 * 4 + 3] + bv[3]);
                    *reinterpret_cast<u32x2_t *>(lds + m * RB + (((p >> 3) ^ (m & (CPR - 1))) << 4) + (p & 7) * 2) = o;
                }
            }
    __syncthreads();
    const int c = threadIdx.x & (CPR - 1);
    const int64_t p = p0 + 8 * c;
#pragma unroll 4
    for (int it = 0; it < 128 * HM * CPR / 512; ++it) {
        const int m = threadIdx.x / CPR + it * (512 / CPR);
        if (m0 + m >= a.M || p >= a.P) continue;
        const u32x4_t v = *reinterpret_cast<const u32x4_t *>(lds + m * RB + ((c ^ (m & (CPR - 1))) << 4));
        uint16_t *dst = a.out + (m0 + m) * a.ld_out + p;
        if (p + 8 <= a.P) {
            *reinterpret_cast<u32x4_t *>(dst) = v;
        } else {
            const uint32_t wv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (p + e < a.P) dst[e] = static_cast<uint16_t>(wv[e >> 1] >> ((e & 1) * 16));
        }
    }
}

// Work item of workgroup b of n, of an order in which neighbours share operand rows: workgroups
// are dealt to the 8 XCDs in turn, each with its own L2, so the workgroups of one XCD (b mod 8)
// take one contiguous run of the order.
__device__ __forceinline__ uint32_t xcd_run(uint32_t b, uint32_t n) {
    const uint32_t x = b & 7, q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// Tile t of pt x mt tiles, in bands of about five m tiles, p by p inside a band: 32 consecutive
// tiles, what an XCD runs at a time, read about 6 + 5 operand tiles.  With the tiles dealt m
// fastest to all XCDs, every XCD read all of W (M = 2048: 33 operand tiles per 32).
__device__ __forceinline__ void band_tile(uint32_t t, uint32_t pt, uint32_t mt, int64_t &p, int64_t &m) {
    const uint32_t bands = mt < 8 ? 1 : (mt + 2) / 5;
    const uint32_t band = ((t / pt + 1) * bands - 1) / mt;
    const uint32_t lo = band * mt / bands, hi = (band + 1) * mt / bands, r = t - lo * pt;
    p = uniform64(r / (hi - lo));
    m = uniform64(lo + r % (hi - lo));
}

// Workgroups [0, blocks0) run 256x256 tiles (of a split plan each over its share of the
// reduction, a share's tiles together), the rest 128x128 tiles of the rows from p_tail on.
template <int DT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void dense_kernel(const DenseArgs a) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];
    const uint32_t b = blockIdx.x, b0 = static_cast<uint32_t>(a.blocks0);
    const int steps = static_cast<int>(a.R / 64);
    int64_t p, m;
    if (b < b0) {
        const uint32_t mt = static_cast<uint32_t>((a.M + 255) / 256), tiles = b0 / static_cast<uint32_t>(a.splits);
        const uint32_t item = xcd_run(b, b0);
        const int split = __builtin_amdgcn_readfirstlane(static_cast<int>(item / tiles));
        band_tile(item % tiles, tiles / mt, mt, p, m);
        const int per = static_cast<int>(a.per_split), u0 = split * per;
        dense_tile<DT, 2, 2>(a, lds, p * 256, m * 256, u0, u0 + per < steps ? u0 + per : steps,
                             a.splits > 1 ? split : -1);
    } else {
        const uint32_t mt = static_cast<uint32_t>((a.M + 127) / 128), n = gridDim.x - b0;
        band_tile(xcd_run(b - b0, n), n / mt, mt, p, m);
        dense_tile<DT, 1, 1>(a, lds, a.p_tail + p * 128, m * 128, 0, steps, -1);
    }
}

// ------------------------------------------------------------ operand strips

struct StripArgs {
    DevWeight w[NF4_MAX_SEGMENTS];
    int64_t tile0[NF4_MAX_SEGMENTS + 1];  // cumulative 128-row tiles
    int64_t row0[NF4_MAX_SEGMENTS];       // first stacked row of the segment
    int nseg;
    uint8_t *out;
    int64_t strip;                        // bytes of a strip: 256 x the reduction length
};

// ds_read_b64_tr_b16: in each 16-lane group lane q points at 4 consecutive 16-bit columns of
// row r0 + q / 4 of a row-major LDS tile and receives column q of rows r0 .. r0 + 3.
typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16_t lds_v4i16_t;

__device__ __forceinline__ uint2 tr_read(const uint8_t *s, int off) {
    const v4i16_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_v4i16_t *)((__attribute__((address_space(3))) uint8_t *)s + off));
    return __builtin_bit_cast(uint2, v);
}

// Chunk c (8 columns k) of row n in the 128 x 128 tile: the four threads of four rows that
// store together, and the 4 rows that a transposed read takes, hit distinct banks.
__device__ __forceinline__ int chunk_t(int n, int c) {
    return n * 256 + ((c ^ ((n & 3) << 2) ^ (n & 3)) << 4);
}

// Chunk c (8 of 128 reduction values) of strip row r: two blocks of 64 values, LDS images of
// the GEMM's half tiles.
__device__ __forceinline__ int chunk_s(int r, int c) {
    return (c >> 3) * HALF + r * 128 + (((c & 7) ^ ((r >> 1) & 7)) << 4);
}

// The stacked weight as the GEMM's operand strips: 128 rows p by 64 reduction values at a time, each
// block the 16 KB image of an LDS half tile, so that a step's DMA reads 16 KB in a row.  (Kept
// row-major, a step read 128 bytes of each of 128 rows: from cold memory the down forward at
// M = 2048 took 92 us instead of 80.)  T false: p = n, reduction k; T true: p = k, reduction n.
//
// A workgroup takes 128 rows n x 128 columns k: thread t dequantizes 32 columns of rows t / 4 and
// t / 4 + 64 (half tables shared with thread t ^ 1: one absmax block per 64 columns) into LDS,
// and the two blocks leave as whole 4 KB per store of the workgroup.  T goes through LDS twice: the tile in its natural
// order, read back transposed, 8 rows n of one column per lane.  Bound: the 2-byte writes.
// Plain stores, unlike the standalone dequantization's: the GEMM reads the strips back at once
// (gate|up forward at M = 2048 127 -> 118 us).
template <int DT, bool T>
__global__ __launch_bounds__(256) void dequant_strips_kernel(const StripArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[128 * 256];
    __shared__ float s_code2[256];
    const uint32_t nt = static_cast<uint32_t>(a.tile0[a.nseg]);
    const int64_t ti = uniform64(blockIdx.x % nt), k0 = uniform64(int64_t(blockIdx.x / nt) * 128);
    int seg = 0;
#pragma unroll
    for (int i = 1; i < NF4_MAX_SEGMENTS; ++i)
        if (i < a.nseg && ti >= a.tile0[i]) seg = i;
    const DevWeight w = a.w[seg];
    const int64_t n0 = (ti - a.tile0[seg]) * 128;
    const int t = threadIdx.x;
    u32x4_t raw[2];
    int64_t blk[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        int64_t n = n0 + (t >> 2) + 64 * i;
        if (n >= w.rows) n = w.rows - 1;  // (not stored, or past the strip's last row)
        const int64_t e = n * w.cols + k0 + (t & 3) * 32;
        raw[i] = *reinterpret_cast<const u32x4_t *>(w.packed + (e >> 1));
        blk[i] = e >> w.bs_shift;
    }
    if (w.nested) s_code2[t] = w.code2[t];
    float code[16];
    load_code_sgpr(w.code, code);
    const Nf4HalfCodes hc = half_codes(code);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const Nf4Table tb = make_table_half<DT>(hc, absmax_of(w, s_code2, blk[i]));
        const int n = (t >> 2) + 64 * i;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t d = q == 0 ? raw[i].x : q == 1 ? raw[i].y : q == 2 ? raw[i].z : raw[i].w;
            const int c = (t & 3) * 4 + q;
            *reinterpret_cast<u32x4_t *>(tile + (T ? chunk_t(n, c) : chunk_s(n, c))) = lookup8s(tb, d, hc.selbase);
        }
    }
    __syncthreads();
    if constexpr (T) {
        const int lane = t & 63, wave = t >> 6, q = lane & 15, g = lane >> 4;
        u32x4_t v[8];
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int kl = (wave * 2 + (it >> 2)) * 16;  // 16 columns
            const int nl = (it & 3) * 32 + g * 8;        // 8 rows
            const int kq = kl + (q & 3) * 4, nr = nl + (q >> 2);
            const uint2 lo = tr_read(tile, chunk_t(nr, kq >> 3) + (kq & 7) * 2);
            const uint2 hi = tr_read(tile, chunk_t(nr + 4, kq >> 3) + (kq & 7) * 2);
            v[it] = (u32x4_t){lo.x, lo.y, hi.x, hi.y};
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < 8; ++it)
            *reinterpret_cast<u32x4_t *>(tile + chunk_s((wave * 2 + (it >> 2)) * 16 + q, (it & 3) * 4 + g)) = v[it];
        __syncthreads();
    }
    // natural: strip (row0 + n0) / 128 (segments may start inside one), blocks k0 / 64 and + 1;
    // transposed: strip k0 / 128, blocks (row0 + n0) / 64 and + 1 (the second past a segment's end is
    // another workgroup's)
    const int64_t r0 = a.row0[seg] + n0;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        const int o = it * 4096 + t * 16;  // 16 bytes of the tile's two blocks
        const u32x4_t v = *reinterpret_cast<const u32x4_t *>(tile + o);
        if constexpr (T) {
            if (n0 + (o >> 14) * 64 < w.rows)
                *reinterpret_cast<u32x4_t *>(a.out + k0 / 128 * a.strip + r0 / 64 * HALF + o) = v;
        } else {
            const int row = (o & (HALF - 1)) >> 7;
            if (n0 + row < w.rows) {
                // a segment's first row need not start a strip: the row's place, and its swizzle there
                const int64_t sr = r0 + row;
                const int lr = static_cast<int>(sr & 127);
                const int c = ((o >> 4) & 7) ^ ((row >> 1) & 7) ^ ((lr >> 1) & 7);
                *reinterpret_cast<u32x4_t *>(a.out + (sr >> 7) * a.strip + (k0 / 64 + (o >> 14)) * HALF +
                                             lr * 128 + (c << 4)) = v;
            }
        }
    }
}

}  // namespace

int dequant_strips(const nf4_weight *ws, int nw, bool transposed, void *out, int dtype, hipStream_t st) {
    StripArgs a = {};
    a.nseg = nw;
    a.out = static_cast<uint8_t *>(out);
    int64_t rows = 0;
    for (int i = 0; i < nw; ++i) {
        a.w[i] = to_dev(ws[i]);
        a.tile0[i + 1] = a.tile0[i] + (ws[i].rows + 127) / 128;
        a.row0[i] = rows;
        rows += ws[i].rows;
    }
    a.strip = (transposed ? rows : ws[0].cols) * 256;
    const dim3 grid(static_cast<unsigned>(a.tile0[nw] * (ws[0].cols / 128)));
    if (dtype == NF4_BF16) {
        if (transposed) hipLaunchKernelGGL((dequant_strips_kernel<NF4_BF16, true>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((dequant_strips_kernel<NF4_BF16, false>), grid, dim3(256), 0, st, a);
    } else {
        if (transposed) hipLaunchKernelGGL((dequant_strips_kernel<NF4_F16, true>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((dequant_strips_kernel<NF4_F16, false>), grid, dim3(256), 0, st, a);
    }
    return status_of(hipGetLastError());
}

// Time in us of `n` workgroups, one per CU, over `steps` 64-deep steps: whole rounds of 256, then
// the rest, whose step slows down with the share u of the CUs in use (power, L2 misses).
// Fitted to the seven Qwen2.5 projections of both models inside a layer's sequence of products
// (cold weights), both directions and dtypes, M = 384 .. 8192, every plan timed (5.9 % rms).
struct RoundTimes {
    double first, step, busy, power, next, full_step;
};
static constexpr RoundTimes kTimes256{6.2, 0.982, 0.46, 1.56, 5.4, 1.476};
static constexpr RoundTimes kTimes128{2.1, 0.0, 0.567, 0.105, 1.1, 0.547};

static double rounds_time(const RoundTimes &k, int64_t n, int64_t steps) {
    const double st = double(steps), u = double(n % 256) / 256.0;
    if (n == 256) return k.first + st * (k.step + k.busy);
    double t = double(n / 256) * (k.next + st * k.full_step);
    if (u > 0) t += (n < 256 ? k.first : k.next) + st * (k.step + k.busy * std::pow(u, k.power));
    return t;
}

// The cheapest of: 256x256 tiles; 128x128 tiles (a quarter of the work per workgroup at 1.5
// times the cost per product: LDS reads bound it); whole rounds of 256x256 tiles with the rows
// left in 128x128 tiles; 256x256 tiles with the reduction split (fp32 partials written, then
// added by a launch of their own; it has to be 2 us better, for the workspace).
DensePlan dense_plan(int64_t P, int64_t M, int64_t R) {
    const int64_t steps = R / 64, mt = (M + 255) / 256, mt1 = (M + 127) / 128, pt = (P + 255) / 256;
    DensePlan best{};
    best.cost = 1e30;
    auto offer = [&](double cost, int64_t hp, int splits) {
        if (cost >= best.cost) return;
        const int64_t p_tail = hp * 256 < P ? hp * 256 : P;
        best = DensePlan{cost, hp * mt * splits, (P - p_tail + 127) / 128 * mt1,
                         (steps + splits - 1) / splits, p_tail, splits};
    };
    offer(rounds_time(kTimes256, pt * mt, steps), pt, 1);
    offer(rounds_time(kTimes128, (P + 127) / 128 * mt1, steps), 0, 1);
    const int64_t hp = pt * mt / 256 * 256 / mt;
    if (hp > 0 && hp < pt)
        offer(rounds_time(kTimes256, hp * mt, steps) +
                  rounds_time(kTimes128, (P - hp * 256 + 127) / 128 * mt1, steps), hp, 1);
    if (P % 4 == 0) {  // (16-byte partial stores)
        for (int s = 2; s <= 8 && s * pt * mt <= 520; ++s) {
            const int64_t per = (steps + s - 1) / s;
            if (per < 4 || (s - 1) * per >= steps) continue;  // no empty split
            offer(rounds_time(kTimes256, pt * mt * s, per) + 4.2 + double(s) * double(M) * double(P) * 4.0 / 3.65e6 + 2.0,
                  pt, s);
        }
    }
    return best;
}

int dense_gemm(DenseArgs &a, const DensePlan &p, int dtype, hipStream_t st) {
    a.blocks0 = p.blocks0;
    a.per_split = p.per_split;
    a.splits = p.splits;
    a.p_tail = p.p_tail;
    const dim3 grid(static_cast<unsigned>(p.blocks0 + p.blocks1));
    if (dtype == NF4_BF16) hipLaunchKernelGGL(dense_kernel<NF4_BF16>, grid, dim3(512), 0, st, a);
    else hipLaunchKernelGGL(dense_kernel<NF4_F16>, grid, dim3(512), 0, st, a);
    return status_of(hipGetLastError());
}
