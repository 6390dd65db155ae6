// Channel-sum kernel of the TDD path on bit planes.
//
// A time tile of a workgroup is TILE = 32 * T output samples (T = 128), split
// into 32 runs of T consecutive samples; one 32-bit word holds, for one bit
// plane of the samples and one position p, that bit of the sample p of each
// run (bit r = run r). The rows are stored that way (dd_tdd_transpose_planes):
// word (q*T + p)*NB + b of a channel is plane b of samples q*TILE + r*T + p,
// r = 0..31. A window that starts at delay a reads position s = a + p as runs
// r + s/T at position s % T: one funnel shift of two words TILE samples apart,
// made once while the window is staged in LDS. A DM whose delay is d then
// reads whole words at position d - a + m: no shift, and 32 samples of one bit
// a word. T = 256 halves the staging per output but doubles the counters: with
// 2 DMs per wave they spilled, with 1 it measured 12.1 against 11.6 ms (2-bit,
// 512 ch x 4 beams x 1024 DMs, at an early stage of this kernel).
//
// Sums are bit-sliced counters: PL planes per position, plane l counting 2^l.
// CC channels are added at a time, level by level: a full adder takes two
// inputs of a level into its plane (sum, one three-input bit operation) and
// hands the carry (majority, another) to the next level; an odd input takes a
// half adder. Per channel and 32 samples that is 2.3 operations for 1-bit
// input (16 channels at a time), 4.8 for 2-bit (8), 10 for 4-bit and 18 for
// 8-bit (4), with NB words read from LDS. The packed-lane kernel takes two
// words and a funnel shift, then a mask, a shift and an addition per 4 samples.
// The counters hold the exact sums (the uint32 sums of
// src/tdd/dedisperse/dedisperse_kernel.cuh:151-193).
//
// What bounds it is the bit operations (half-rate) and the staging: every block
// of DMs fetches its windows of every channel, 26.6 GB a launch at the 4-bit
// size below (1.9 TB/s). Execute times, packed
// lanes (4-bit: runs layout) -> planes: 1-bit 512 ch x 200003 x 501 DMs 0.99 ->
// 0.35 ms; 2-bit 512 ch x 4 beams (2.4e6 samples) x 1024 DMs 21.8 -> 8.4 ms;
// 4-bit 1024 ch x 2^20 x 1167 DMs 22.9 -> 14.6 ms; 8-bit 1024 ch x 15625 x 3000
// DMs 1.92 -> 1.43 ms. Tried: 4 DMs per wave (spills),
// staging each position with two loads of its own (2-bit 11.6 ms), its scalar
// loads where they are used (10.0 ms), the carries of four chunks together (14 %
// fewer bit operations, 4-bit unchanged).
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "tdd_planes_stage.h"

namespace {

constexpr int T = DD_TDD_PLANES_T;     // positions per tile = run length (samples)
constexpr int G = T / 64;              // positions per lane
constexpr int TILE = 32 * T;           // output samples per tile

// (float)sum * out_range / (in_range * nchans) * factor with the rounded
// quotient (src/tdd/dedisperse/dedisperse_kernel.cuh:45-64) from the rounded
// reciprocal: num * rcp, then one correction with the exact remainder. Equal to
// the IEEE division for every sum <= den of 1-, 2-, 4- and 8-bit samples, 1 ..
// 8192 channels and the three output ranges (checked exhaustively), three
// operations instead of ten.
__device__ __forceinline__ float tdd_scale(float fsum, const dd_tdd_epilogue& ep, float rcp)
{
    const float num = fsum * ep.out_range;
    const float q = num * rcp;
    return fmaf(fmaf(-q, ep.den, num), rcp, q) * ep.factor;
}

__device__ __forceinline__ void tdd_store(uint8_t* row, size_t t, float scaled, const dd_tdd_epilogue& ep)
{
    if (ep.out_nbits == 32) {
        reinterpret_cast<float*>(row)[t] = scaled;
    } else {
        float v = fminf(fmaxf(scaled, 0.f), ep.out_range);  // clip, then truncate
        if (ep.out_nbits == 16) reinterpret_cast<uint16_t*>(row)[t] = (uint16_t)__float2uint_rz(v);
        else row[t] = (uint8_t)__float2uint_rz(v);
    }
}

// ---------------------------------------------------------------------------
// Transpose: time-major packed rows -> bit-plane rows
// ---------------------------------------------------------------------------
//
// A workgroup takes 32 positions x 32 runs of one tile (1024 sample rows) x 64
// bytes: staged in LDS (rows of 17 words, so that the 32 positions of one word
// fall into 32 banks), then a thread reads one word of the 32 runs at its
// position, transposes the 32 x 32 bit matrix in registers (five stages of
// shift and bitfield insert) and holds the plane words of 32/NB channels.

constexpr uint32_t low_blocks_mask(int sh)
{
    // the low sh bits of every 2*sh-bit group
    uint32_t m = 0;
    for (int b = 0; b < 32; ++b)
        if ((b / sh) % 2 == 0) m |= 1u << b;
    return m;
}

constexpr int TP_W = 16;   // words of a sample row per workgroup
constexpr int TP_P = 32;   // positions per workgroup

template <int NB>
__global__ __launch_bounds__(256) void tdd_transpose_planes_k(
    const uint8_t* __restrict__ in, size_t nsamps, size_t in_stride, size_t row_bytes, size_t nchans,
    uint32_t* __restrict__ out, size_t row_words)
{
    __shared__ uint32_t tile[32 * TP_P * (TP_W + 1)];
    const int tid = threadIdx.x;
    const size_t q = blockIdx.x / (T / TP_P);
    const size_t p0 = (size_t)(blockIdx.x % (T / TP_P)) * TP_P;
    const size_t b0 = (size_t)blockIdx.y * (TP_W * 4);
    const size_t tq = q * TILE + p0;  // sample of run 0, position p0
    const bool words = ((in_stride | reinterpret_cast<uintptr_t>(in)) & 3u) == 0;
    const int w = tid % TP_W, row0 = tid / TP_W;
    const size_t b = b0 + 4 * (size_t)w;
    if (words && (row_bytes % 4 == 0 || b0 + TP_W * 4 <= row_bytes) && tq + 31 * T + TP_P <= nsamps) {
        // whole words of whole rows: a thread's word lies in the row or beyond
        // it (zeros); 16 loads are issued before the first is waited on (rows
        // of odd bytes in a padded stride, in all but the last tile: 4108 2-bit
        // channels, stride 1028, 200000 samples 154 us, guarded throughout 282)
        for (int n0 = 0; n0 < 64; n0 += 16) {
            uint32_t v[16];
#pragma unroll
            for (int n = 0; n < 16; ++n) {
                const int row = row0 + 16 * (n0 + n);  // run row / 32, position row % 32
                const size_t t = tq + (size_t)(row / TP_P) * T + row % TP_P;
                v[n] = (b < row_bytes) ? *reinterpret_cast<const uint32_t*>(in + t * in_stride + b) : 0;
            }
#pragma unroll
            for (int n = 0; n < 16; ++n) tile[(row0 + 16 * (n0 + n)) * (TP_W + 1) + w] = v[n];
        }
    } else {
        for (int n = 0; n < 64; ++n) {
            const int row = row0 + 16 * n;
            const size_t t = tq + (size_t)(row / TP_P) * T + row % TP_P;
            uint32_t v = 0;
            if (t < nsamps) {
                if (words && b + 3 < row_bytes) {
                    v = *reinterpret_cast<const uint32_t*>(in + t * in_stride + b);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (b + k < row_bytes) v |= (uint32_t)in[t * in_stride + b + k] << (8 * k);
                }
            }
            tile[row * (TP_W + 1) + w] = v;
        }
    }
    __syncthreads();

    constexpr int CPW = 32 / NB;  // channels per word
    const int p = tid % TP_P;
#pragma unroll 1
    for (int wi = tid / TP_P; wi < TP_W; wi += 256 / TP_P) {
        const size_t c0 = (b0 / 4 + wi) * CPW;
        if (c0 >= nchans) break;
        uint32_t R[32];
#pragma unroll
        for (int r = 0; r < 32; ++r) R[r] = tile[(r * TP_P + p) * (TP_W + 1) + wi];
        // bit i of R[r] -> bit r of R[i]
#pragma unroll
        for (int B = 16; B >= 1; B /= 2) {
            const uint32_t m = low_blocks_mask(B);
#pragma unroll
            for (int r = 0; r < 32; ++r) {
                if (r & B) continue;
                const uint32_t x = R[r], y = R[r + B];
                R[r] = (x & m) | ((y << B) & ~m);
                R[r + B] = ((x >> B) & m) | (y & ~m);
            }
        }
        uint32_t* o = out + c0 * row_words + (q * T + p0 + p) * NB;
#pragma unroll
        for (int i = 0; i < CPW; ++i) {
            if (c0 + i < nchans) {
                uint32_t* d = o + i * row_words;
                if constexpr (NB == 1) {
                    d[0] = R[i];
                } else if constexpr (NB == 2) {
                    *reinterpret_cast<uint2*>(d) = make_uint2(R[2 * i], R[2 * i + 1]);
                } else {
#pragma unroll
                    for (int k = 0; k < NB; k += 4)
                        *reinterpret_cast<uint4*>(d + k) =
                            make_uint4(R[NB * i + k], R[NB * i + k + 1], R[NB * i + k + 2], R[NB * i + k + 3]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Channel sum
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}
__device__ __forceinline__ uint32_t majority(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0xe8);
}

// Level at which N samples of NB bits leave a single carry (what they add to
// the counter beyond its low planes).
constexpr int top_level(int NB, int N)
{
    for (int L = 0, NC = 0;; ++L) {
        const int NI = (L < NB ? N : 0) + NC;
        if (L >= NB && NI == 1) return L;
        NC = (NI + 1) / 2;
    }
}

__device__ __forceinline__ uint32_t full_add(uint32_t& acc, uint32_t a, uint32_t b)
{
    const uint32_t s = acc;
    acc = xor3(s, a, b);
    return majority(s, a, b);
}
__device__ __forceinline__ uint32_t half_add(uint32_t& acc, uint32_t a)
{
    const uint32_t s = acc;
    acc = s ^ a;
    return s & a;
}

// Level L of an addition to the counter: its inputs are plane L of the N
// samples (L < NB) and the NC carries of the level below. Returns the carry
// into level top_level(NB, N).
template <int NB, int N, int PL, int L, int NC>
__device__ __forceinline__ uint32_t add_level(uint32_t (&acc)[PL], const uint32_t (&x)[N][NB],
                                              const uint32_t (&c)[NC > 0 ? NC : 1])
{
    if constexpr (L == top_level(NB, N)) {
        return c[0];
    } else {
        constexpr int NX = (L < NB) ? N : 0, NI = NX + NC, NO = (NI + 1) / 2;
        auto in = [&](int i) -> uint32_t {
            if constexpr (L < NB) {
                if (i < NX) return x[i][L < NB ? L : 0];
            }
            return c[i - NX];
        };
        uint32_t carry[NO];
#pragma unroll
        for (int i = 0; i + 1 < NI; i += 2) carry[i / 2] = full_add(acc[L], in(i), in(i + 1));
        if constexpr (NI % 2) carry[NO - 1] = half_add(acc[L], in(NI - 1));
        return add_level<NB, N, PL, L + 1, NO>(acc, x, carry);
    }
}

// a into planes L, L+1, ... of the counter (the carry out of the last plane is
// zero: the counter holds the largest sum)
template <int PL>
__device__ __forceinline__ void ripple(uint32_t (&acc)[PL], int L, uint32_t a)
{
#pragma unroll
    for (int l = 0; l < PL; ++l)
        if (l >= L) a = half_add(acc[l], a);
}

// NB words (the planes of one position) at p, aligned to their size
template <int NB>
__device__ __forceinline__ void read_planes(const uint32_t* p, uint32_t (&v)[NB])
{
    if constexpr (NB == 1) {
        v[0] = p[0];
    } else if constexpr (NB == 2) {
        const uint2 u = *reinterpret_cast<const uint2*>(p);
        v[0] = u.x, v[1] = u.y;
    } else {
#pragma unroll
        for (int k = 0; k < NB; k += 4) {
            const uint4 u = *reinterpret_cast<const uint4*>(p + k);
            v[k] = u.x, v[k + 1] = u.y, v[k + 2] = u.z, v[k + 3] = u.w;
        }
    }
}
// the same from global memory (global loads, not flat ones, which the LDS
// counter would wait for)
typedef const __attribute__((address_space(1))) uint32_t gword;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <int NB>
__device__ __forceinline__ void load_planes(gword* p, uint32_t (&v)[NB])
{
    if constexpr (NB == 1) {
        v[0] = p[0];
    } else if constexpr (NB == 2) {
        const u32x2 u = *reinterpret_cast<const __attribute__((address_space(1))) u32x2*>(p);
        v[0] = u.x, v[1] = u.y;
    } else {
#pragma unroll
        for (int k = 0; k < NB; k += 4) {
            const u32x4 u = *reinterpret_cast<const __attribute__((address_space(1))) u32x4*>(p + k);
            v[k] = u.x, v[k + 1] = u.y, v[k + 2] = u.z, v[k + 3] = u.w;
        }
    }
}
template <int NB>
__device__ __forceinline__ void write_planes(uint32_t* p, const uint32_t (&v)[NB])
{
    if constexpr (NB == 1) {
        p[0] = v[0];
    } else if constexpr (NB == 2) {
        *reinterpret_cast<uint2*>(p) = make_uint2(v[0], v[1]);
    } else {
#pragma unroll
        for (int k = 0; k < NB; k += 4)
            *reinterpret_cast<uint4*>(p + k) = make_uint4(v[k], v[k + 1], v[k + 2], v[k + 3]);
    }
}

template <int V>
struct Phase {
    static constexpr int value = V;
};

// CC channels per staged chunk, PL counter planes, DPW DMs per wave, WAVES
// waves: a block of DPW * WAVES DMs. lds: CC windows of stride positions, then
// T positions of zeros.
template <int NB, int CC, int PL, int DPW, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 4) void tdd_planes_k(
    const uint32_t* __restrict__ rows, size_t row_words, const uint32_t* __restrict__ code,
    const uint32_t* __restrict__ wstart, const uint32_t* __restrict__ chunks, uint32_t nchunk, uint32_t ndm, uint32_t nsamps_out, uint32_t ndmblk, uint32_t stride,
    uint8_t* __restrict__ out, size_t out_stride, dd_tdd_epilogue ep, const dd_tdd_beam* __restrict__ beams,
    const uint32_t* __restrict__ tile_beam)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];

    // XCD-aware mapping: workgroups go round-robin over the 8 XCDs; each XCD
    // gets a contiguous range of (time tile, DM block) pairs, DM block fastest,
    // so the blocks sharing a tile's input run on the same L2.
    const uint32_t nb = gridDim.x, bid = blockIdx.x;
    const uint32_t xcd = bid & 7u, per = nb >> 3, rem = nb & 7u;
    const uint32_t L = xcd * per + min(xcd, rem) + (bid >> 3);
    const uint32_t tile_g = L / ndmblk, dblk = L % ndmblk;
    uint32_t tile = tile_g;
    if (beams) {
        const dd_tdd_beam bm = beams[tile_beam[tile_g]];
        tile = tile_g - bm.tile0;
        rows = bm.rows;
        row_words = bm.row_words;
        nsamps_out = bm.nsamps_out;
        out = bm.out;
        out_stride = bm.out_stride;
    }
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t dmb = dblk * (DPW * WAVES) + wave * DPW;

    uint32_t acc[DPW][G][PL];
#pragma unroll
    for (int i = 0; i < DPW; ++i)
#pragma unroll
        for (int k = 0; k < G; ++k)
#pragma unroll
            for (int l = 0; l < PL; ++l) acc[i][k][l] = 0;

    const uint2* desc = reinterpret_cast<const uint2*>(wstart) + (size_t)dblk * nchunk * CC;  // (start, channel)
    const uint32_t* pos = chunks + (size_t)dblk * nchunk;  // positions staged per channel
    const uint32_t* cod = code + ((size_t)dblk * WAVES + wave) * nchunk * (DPW * CC);

    // Staging: item (slot jj, group g) of a wave is the positions 64g .. 64g+63
    // (mod T) of one channel's window, however long it is: position s = u*T + p
    // of the rows is the runs r + u at p, so three words a lane (this tile's,
    // the next two's at the window's start) give the item's words of every u
    // by one funnel shift each. The words of the next chunk are loaded before
    // this chunk's sums and wait in registers.
    constexpr int ITEMS = CC * G, IPW = (ITEMS + WAVES - 1) / WAVES;
    uint32_t w[IPW][3][NB];
    auto item_of = [&](int n) -> uint32_t {
        return (ITEMS % WAVES) ? min(wave + WAVES * n, ITEMS - 1u) : wave + WAVES * n;
    };
    auto load_desc = [&](uint32_t ci, uint2 (&d)[IPW], uint32_t& P) {
#pragma unroll
        for (int n = 0; n < IPW; ++n) d[n] = desc[ci * CC + item_of(n) / G];
        P = pos[ci];
    };
    // The third word is needed (and lies in another tile's cache lines) only
    // where the window's runs pass the next tile's start. 4- and 8-bit input
    // loads the second again elsewhere (4-bit, 1024 ch x 2^20 x 1167 DMs: 21.4
    // instead of 39 GB fetched, 15.07 -> 14.55 ms); with the fewer bytes and
    // more items of 1- and 2-bit input finding out costs more (2-bit 8.30 ->
    // 8.63 ms).
    auto stage_load = [&](const uint2 (&d)[IPW], uint32_t P) {
#pragma unroll
        for (int n = 0; n < IPW; ++n) {
            gword* src = (gword*)rows + (size_t)d[n].y * row_words + ((size_t)tile + d[n].x / T / 32) * (T * NB) +
                         (64 * (item_of(n) % G) + lane) * NB;
            const uint32_t third = (NB < 4 || planes_needs_third(d[n].x, P)) ? 2 : 1;
            load_planes<NB>(src, w[n][0]);
            load_planes<NB>(src + T * NB, w[n][1]);
            load_planes<NB>(src + third * (T * NB), w[n][2]);
        }
    };
    auto stage_write = [&](const uint2 (&d)[IPW], uint32_t P) {
#pragma unroll
        for (int n = 0; n < IPW; ++n) {
            const uint32_t item = item_of(n);
            const uint32_t a = d[n].x, p = 64 * (item % G) + lane;
            const uint32_t first = planes_lds_first(item / G, stride, a, p, NB);
            planes_stage(a, P, p, [&](int k, uint32_t shift, uint32_t u, bool in) {
                uint32_t v[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) v[b] = __builtin_amdgcn_alignbit(w[n][k + 1][b], w[n][k][b], shift);
                if (in) write_planes<NB>(lds + planes_lds_word(first, u, NB), v);
            });
        }
    };

    // the window of the channels past the last one: zeros after the chunk's
    for (uint32_t i = threadIdx.x; i < T * NB; i += WAVES * 64) lds[CC * stride * NB + i] = 0;
    constexpr int LT = top_level(NB, CC);
    static_assert(LT < PL, "a chunk's carry has its plane");
    uint32_t pend[DPW][G];
    uint2 dc[IPW], dn[IPW];  // descriptors of this chunk's and the next one's items
    uint32_t Pc, Pn;
    load_desc(0, dc, Pc);
    stage_load(dc, Pc);
    // Chunk ci, ci % 2 = PH (the number of chunks is even). The carry of an even
    // chunk into plane LT waits for the odd one's (one full adder for both), so
    // that the half adders through the planes above run once in two chunks.
    auto chunk = [&](uint32_t ci, auto ph) __attribute__((always_inline)) {
        constexpr int PH = decltype(ph)::value;
        // scalar loads of the whole iteration up front, so that their latency
        // passes with the staging writes (scalar and LDS accesses share a
        // counter: the wait before the barrier covers both)
        uint32_t c[DPW][CC];  // wave-uniform window offsets (bytes)
        {
            const uint32_t* cp = cod + (size_t)ci * (DPW * CC);
#pragma unroll
            for (int i = 0; i < DPW; ++i)
#pragma unroll
                for (int jj = 0; jj < CC; ++jj) c[i][jj] = cp[i * CC + jj];
        }
        load_desc(min(ci + 1, nchunk - 1), dn, Pn);
        __syncthreads();  // the previous chunk's sums have read the windows
        stage_write(dc, Pc);
#pragma unroll
        for (int i = 0; i < DPW; ++i)
#pragma unroll
            for (int jj = 0; jj < CC; ++jj) asm volatile("" : "+s"(c[i][jj]));
#pragma unroll
        for (int n = 0; n < IPW; ++n) {
            asm volatile("" : "+s"(dn[n].x), "+s"(dn[n].y));
            dc[n] = dn[n];
        }
        asm volatile("" : "+s"(Pn));
        Pc = Pn;
        __syncthreads();
        stage_load(dc, Pc);  // (the last chunk's again after the last one)
        // all LDS words of a step first, so that their latencies overlap
        constexpr int KB = (NB < 4 && 2 * CC * NB <= 32) ? 2 : 1;
#pragma unroll
        for (int i = 0; i < DPW; ++i)
#pragma unroll
            for (int k0 = 0; k0 < G; k0 += KB) {
                uint32_t x[KB][CC][NB];
#pragma unroll
                for (int jj = 0; jj < CC; ++jj) {
                    const uint32_t* p =
                        reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(lds) + c[i][jj]) + lane * NB;
#pragma unroll
                    for (int k = 0; k < KB; ++k) read_planes<NB>(p + 64 * NB * (k0 + k), x[k][jj]);
                }
                __builtin_amdgcn_sched_barrier(0);
                const uint32_t none[1] = {0};
#pragma unroll
                for (int k = 0; k < KB; ++k) {
                    uint32_t(&cnt)[PL] = acc[i][k0 + k];
                    const uint32_t t = add_level<NB, CC, PL, 0, 0>(cnt, x[k], none);
                    if constexpr (PH == 0) pend[i][k0 + k] = t;
                    else ripple(cnt, LT + 1, full_add(cnt[LT], pend[i][k0 + k], t));
                }
            }
        // the sums end here (moved past the barrier, they cost copies of the counters)
#pragma unroll
        for (int i = 0; i < DPW; ++i)
#pragma unroll
            for (int k = 0; k < G; ++k)
#pragma unroll
                for (int l = 0; l <= PL; ++l) asm volatile("" : "+v"(l < PL ? acc[i][k][l < PL ? l : 0] : pend[i][k]));
    };
    for (uint32_t ci = 0; ci < nchunk; ci += 2) {
        chunk(ci, Phase<0>{});
        chunk(ci + 1, Phase<1>{});
    }

    // Epilogue: lane l owns positions l + 64k; run r of position m is sample
    // tile * TILE + r*T + m. Four planes make the nibbles of the runs 4n + s
    // (mask every fourth bit), two such words the bytes of runs 8n + s and 8n +
    // 4 + s, which convert to float one by one.
    constexpr int NG = (PL + 3) / 4, NY = (NG + 1) / 2;  // nibbles, bytes of a sum
    const uint32_t t0 = tile * TILE;
    const float rcp = 1.0f / ep.den;
#pragma unroll
    for (int i = 0; i < DPW; ++i) {
        const uint32_t dm = dmb + i;
        if (dm >= ndm) continue;
        uint8_t* orow = out + (size_t)dm * out_stride;
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const uint32_t m = lane + 64u * k;
#pragma unroll 1
            for (int s = 0; s < 4; ++s) {
                uint32_t nib[2 * NY];
#pragma unroll
                for (int g = 0; g < 2 * NY; ++g) {
                    nib[g] = 0;
#pragma unroll
                    for (int l = 0; l < 4; ++l)
                        if (4 * g + l < PL) nib[g] |= ((acc[i][k][4 * g + l < PL ? 4 * g + l : 0] >> s) & 0x11111111u) << l;
                }
                uint32_t byt[2][NY];
#pragma unroll
                for (int y = 0; y < NY; ++y) {
                    byt[0][y] = (nib[2 * y] & 0x0f0f0f0fu) | ((nib[2 * y + 1] & 0x0f0f0f0fu) << 4);
                    byt[1][y] = ((nib[2 * y] >> 4) & 0x0f0f0f0fu) | (nib[2 * y + 1] & 0xf0f0f0f0u);
                }
#pragma unroll
                for (int r8 = 0; r8 < 8; ++r8) {  // run 4 r8 + s
                    float sum = 0.f;
#pragma unroll
                    for (int y = NY - 1; y >= 0; --y)
                        sum = sum * 256.f + (float)((byt[r8 & 1][y] >> (8 * (r8 >> 1))) & 0xffu);  // exact
                    const uint32_t t = t0 + (uint32_t)(4 * r8 + s) * T + m;
                    if (t < nsamps_out) tdd_store(orow, t, tdd_scale(sum, ep, rcp), ep);
                }
            }
        }
    }
}

}  // namespace

extern "C" hipError_t dd_tdd_transpose_planes(const uint8_t* in, size_t nsamps, size_t in_stride, unsigned nbits,
                                              size_t nchans, uint32_t* out, size_t row_words, hipStream_t stream)
{
    const size_t row_bytes = (nchans * nbits + 7) / 8;
    const size_t rb = (in_stride < row_bytes) ? in_stride : row_bytes;
    if (row_words % ((size_t)T * nbits)) return hipErrorInvalidValue;
    const size_t nq = row_words / ((size_t)T * nbits);
    if (nq * (T / TP_P) >= (size_t(1) << 31)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(nq * (T / TP_P)), (unsigned)((row_bytes + TP_W * 4 - 1) / (TP_W * 4)));
#define DD_TP(NB)                                                                                             \
    hipLaunchKernelGGL(tdd_transpose_planes_k<NB>, grid, dim3(256), 0, stream, in, nsamps, in_stride, rb, nchans, \
                       out, row_words)
    switch (nbits) {
    case 1: DD_TP(1); break;
    case 2: DD_TP(2); break;
    case 4: DD_TP(4); break;
    case 8: DD_TP(8); break;
    default: return hipErrorInvalidValue;
    }
#undef DD_TP
    return hipGetLastError();
}

// Instantiated shapes: (nbits, channels per chunk, counter planes, DMs per wave, waves).
#define DD_PLANES(X) \
    X(1, 16, 10, 2, 8) X(1, 16, 14, 2, 8) X(1, 16, 10, 1, 8) X(1, 16, 14, 1, 8) \
    X(2, 8, 11, 2, 8) X(2, 8, 15, 2, 8) X(2, 8, 11, 1, 8) X(2, 8, 15, 1, 8) \
    X(4, 4, 14, 2, 8) X(4, 4, 17, 2, 8) X(4, 4, 14, 1, 8) X(4, 4, 17, 1, 8) \
    X(8, 4, 16, 1, 8) X(8, 4, 18, 1, 8) X(8, 4, 21, 1, 8)

extern "C" unsigned dd_tdd_planes_chunk(unsigned nbits, size_t nact, unsigned dms_per_wave, unsigned waves)
{
#define DD_FIND(NB, CC, PL, DPW, W)                                                  \
    if (nbits == NB && dms_per_wave == DPW && waves == W &&                          \
        (uint64_t)nact * ((1u << NB) - 1u) < (uint64_t(1) << PL))                    \
        return CC;
    DD_PLANES(DD_FIND)
#undef DD_FIND
    return 0;
}

extern "C" hipError_t dd_tdd_dedisperse_planes(const uint32_t* rows, size_t row_words, unsigned nbits,
                                               const uint32_t* code, const uint32_t* wstart, const uint32_t* chunks,
                                               unsigned nchunk, size_t nact, size_t ndm,
                                               size_t nsamps_out, uint8_t* out, size_t out_stride,
                                               dd_tdd_epilogue ep, dd_tdd_tiling tl, const dd_tdd_beam* beams,
                                               const uint32_t* tile_beam, size_t batch_tiles, hipStream_t stream)
{
    if (ndm == 0) return hipSuccess;
    const size_t ntiles = beams ? batch_tiles : (nsamps_out + TILE - 1) / TILE;
    if (ntiles == 0) return hipSuccess;
    const size_t dpb = (size_t)tl.dms_per_wave * tl.waves;
    if (dpb == 0 || tl.window_words % 64) return hipErrorInvalidValue;
    const size_t ndmblk = (ndm + dpb - 1) / dpb;
    const size_t nblocks = ntiles * ndmblk;
    if (nblocks >= (size_t(1) << 31)) return hipErrorInvalidValue;
#define DD_CALL(NB, CC, PL, DPW, W)                                                                             \
    if (nbits == NB && tl.dms_per_wave == DPW && tl.waves == W && tl.chunk_channels == CC &&                    \
        (uint64_t)nact * ((1u << NB) - 1u) < (uint64_t(1) << PL)) {                                             \
        if ((nact + 2 * CC - 1) / (2 * CC) * 2 != nchunk) return hipErrorInvalidValue;                          \
        const size_t bytes = ((size_t)CC * tl.window_words + T) * NB * 4;                                             \
        auto kern = tdd_planes_k<NB, CC, PL, DPW, W>;                                                           \
        if (bytes > DD_TDD_PLANES_LDS_MAX) return hipErrorInvalidValue;                                         \
        if (bytes > 64 * 1024) {                                                                                \
            /* the same limit from every thread: one plan's must not end below what another's is launched with */ \
            hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,   \
                                               DD_TDD_PLANES_LDS_MAX);                                          \
            if (e != hipSuccess) return e;                                                                      \
        }                                                                                                       \
        hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(W * 64), bytes, stream, rows, row_words, code,   \
                           wstart, chunks, (uint32_t)nchunk, (uint32_t)ndm,                                     \
                           (uint32_t)nsamps_out, (uint32_t)ndmblk, tl.window_words, out, out_stride, ep, beams, \
                           tile_beam);                                                                          \
        return hipGetLastError();                                                                               \
    }
    DD_PLANES(DD_CALL)
#undef DD_CALL
    return hipErrorInvalidValue;
}

extern "C" int dd_tdd_planes_tilings(unsigned nbits, dd_tdd_tiling* out, int max)
{
    int n = 0;
    dd_tdd_tiling shapes[8];  // (fewer per width)
#define DD_LIST(NB, CC, PL, DPW, W)                                                                     \
    if (nbits == NB) {                                                                                  \
        bool seen = false;                                                                              \
        for (int k = 0; k < n; ++k) seen |= shapes[k].dms_per_wave == DPW && shapes[k].waves == W;      \
        if (!seen) {                                                                                    \
            shapes[n] = dd_tdd_tiling{DD_TDD_PLANES_SPL, DPW, W, 16, 0};                                \
            if (n < max && out) out[n] = shapes[n];                                                     \
            ++n;                                                                                        \
        }                                                                                               \
    }
    DD_PLANES(DD_LIST)
#undef DD_LIST
    return n;
}
