// The tile kernel of the experts' products with many rows: out = x W[e]^T in bfloat16 with float32 sums, the
// rows of x being sorted by expert.
//
// A workgroup of four waves makes a tile of 64 TM rows of x by 64 TN rows of W, each wave a quarter
// (32 TM x 32 TN) with v_mfma_f32_32x32x16_bf16, formed transposed (A = W, B = x) so that a lane ends with
// four consecutive columns of one row.  (The 32 x 32 form reads half as many operand registers per flop as
// 16 x 16 x 32; under the chip's power limit a bare loop of it reaches 1.86 PFLOP/s on random operands
// against 1.65.)  K is walked in stages of 64, one 128-byte line per row, which are copied straight into
// shared memory (global_load_lds, 16 bytes a lane; a copy of sixteen half lines moves 67 KB a microsecond
// into a compute unit, one of eight lines 130), their 16-byte chunks swizzled by the row so that operand
// reads have no bank conflicts.
//
// What bounds it is how many bytes a workgroup has under way, not the way into a compute unit (130 KB a microsecond
// out of the XCD's cache, of which the tile of 256 x 256 takes 35) and, while W comes from memory, not the arithmetic:
// two buffers of 64 KB had some 35 KB under way at a time, 1 us of latency long.  Hence:
//  * x and W have rings of buffers of their own in the 160 KB: two of x, whose rows other workgroups of the XCD
//    read too, and three of W, which comes from memory and so is asked for two stages ahead (low tiles: three and
//    three, four and four; of two workgroups to a compute unit 128 x 128 two and three, 64 x 256 two and two, which are all that it
//    holds).  One round of the chip, 16 experts of 256, 192, 128, 64 rows, 4,096 x 4,096: 155, 120, 109, 102 us; with two buffers of
//    both, and lines of W asked for ahead, 163, 141, 123, 108; 128 x 128: 8 x 60, 4,096 -> 3,584 71 -> 51, 64 x 60, 2,048 -> 2,048 138 -> 125, though
//    where W alone bounds it now and then the slower way, by up to 4 % (32 x 40, 4,096 -> 3,584 186 to 197, 182 to 200);
//  * operands of the next 16 k are read between the products of this one, one read per two products, and
//    the one barrier of a stage stands before its last 16 k, so that nothing waits behind it;
//  * copies are spread over a stage's four steps instead of issued in a burst (a burst fills the
//    address unit and holds the products up), x's first, since copies land in order and x's are due sooner.
// 7,108 rows of 32 experts, sums, shares spread as exp(0.4 normal) and nearly equal: 4,096 -> 3,584 326 -> 271 us, 288 -> 256; 3,584 -> 4,096
// 318 -> 272, 270 -> 242.  With an activation in the epilogue, which nobody else's products hide, less or nothing: silu 349 -> 295, 289 -> 287;
// gelu, equal shares, 312 -> 310.  (The rows' gather through `order` costs nothing: 288 in order, 285 gathered.)  In a prompt of 1,777 tokens these two products
// took 341 on average and take 329, with gelu, and 268.  8,000 rows, 4,096 -> 2 x 2,048 363 -> 319, 2,048 -> 4,096 194 -> 172; 8,192 rows of one
// 4,096 x 4,096 228 -> 220 (1,250 TFLOP/s).
// The copies are written in asm because the compiler takes any operand read to depend on every copy in
// flight and waits for all of them; they have no output registers, and the waits below count them.
#pragma once
#include "common.h"
#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 pt_bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float pt_floatx16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float pt_floatx4_t;
union PtFrag {
    uint4 u;
    pt_bf16x8_t v;
};

enum PtMode {
    PT_ROWS = 0,        // bfloat16 rows [pairs, F] of the sums, or of act(sum)
    PT_GATE = 1,        // W: F gate rows, then F up rows; bfloat16 [pairs, F] of act(gate) * up
};

// act < 0: none; 0 silu, 1 gelu (tanh form), 3 gelu (exact); as a gate also 2: a sigmoid(1.702 a) (b + 1) of
// a cut off above and b cut off on both sides at `limit`
struct PtArgs {
    const bf16_t* x;
    const bf16_t* w;
    void* out;
    int F, K;                           // columns of out, a multiple of 8; a multiple of 64
    int act;
    float limit;
    // rows offsets[e] .. offsets[e + 1] - 1 are those of expert e, row p being row order[p] / top of x (or p),
    // W [E, F or 2 F, K]; tiles of rows do not cross experts
    const int* order;
    const int* offsets;
    int top, E;
};

// The activations of all kernels of the experts, so that a value does not depend on how many rows share its step.
// The gate of clamped experts: a <- min(a, limit), b <- b clamped to -limit .. limit, a sigmoid(1.702 a) (b + 1)
__device__ __forceinline__ float re_clamped_pair(float a, float b, float limit) {
    a = fminf(a, limit);
    b = fminf(fmaxf(b, -limit), limit);
    return a / (1.f + expf(-1.702f * a)) * (b + 1.f);
}

// 0 silu, 1 gelu (tanh form), 3 gelu (exact); the numbers of ops.kernels.ACTIVATIONS
__device__ __forceinline__ float re_activation(float z, int act) {
    if (act == 0) return z / (1.f + expf(-z));
    if (act == 1) return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    return 0.5f * z * (1.f + erff(z * 0.7071067811865476f));
}

// act of eight values, once for the whole launch.  (With the exponential and reciprocal instructions in place of the
// library's forms a product of 222 rows for each of 32 experts, 4,096 -> 2 x 3,584, took 606 us and not 623, but
// silu's error grew with its argument, from 1.2e-7 of the value to 3.5e-6 at -60.)
__device__ __forceinline__ void pt_act(float (&z)[8], int act) {
    if (act == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) z[i] = re_activation(z[i], 0);
    } else if (act == 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) z[i] = re_activation(z[i], 1);
    } else if (act == 3) {
#pragma unroll
        for (int i = 0; i < 8; ++i) z[i] = re_activation(z[i], 3);
    }
}
__device__ __forceinline__ void pt_gate(float (&a)[8], const float (&b)[8], int act, float limit) {
    if (act == 2) {
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = re_clamped_pair(a[i], b[i], limit);
        return;
    }
    pt_act(a, act);
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] *= b[i];
}

// f(std::integral_constant<int, I>) for I = A .. B - 1
template <int A, int B, typename Fn>
__device__ __forceinline__ void pt_copies(Fn f) {
    if constexpr (A < B) {
        f(std::integral_constant<int, A>{});
        pt_copies<A + 1, B>(f);
    }
}

// Tiles of up to BM rows that the experts' shares make, and the bm-th of them (expert, first row, the row behind the
// tile's last); every wave works it out for itself, an expert per lane.  EVEN: an expert's tiles are of equal
// height, in steps of 64, instead of all but the last full.
template <int BM>
__device__ __forceinline__ int pt_row_tiles(const int* __restrict__ offsets, int E) {
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int e = lane; e < E; e += 64) n += (offsets[e + 1] - offsets[e] + BM - 1) / BM;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    return __builtin_amdgcn_readfirstlane(n);
}
template <int BM, bool EVEN>
__device__ __forceinline__ void pt_find_tile(const int* __restrict__ offsets, int E, int bm, int& expert, int& m0,
                                             int& m1) {
    const int lane = threadIdx.x & 63;
    // EVEN: the experts whose tiles are highest come first
    for (int steps = EVEN ? BM / 64 : 1; steps > 0; --steps)
        for (int first = 0; first < E; first += 64) {
            const int e = first + lane;
            const int lo = e < E ? offsets[e] : 0, rows = e < E ? offsets[e + 1] - lo : 0;
            int own = (rows + BM - 1) / BM;
            const int high = EVEN ? (rows + 64 * (own > 0 ? own : 1) - 1) / (64 * (own > 0 ? own : 1)) : BM / 64;
            if (EVEN && high != steps) own = 0;
            int end = own;                                       // tiles up to and with this lane's
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int before = __shfl_up(end, o, 64);
                if (lane >= o) end += before;
            }
            const unsigned long long mine = __ballot(bm >= end - own && bm < end);
            if (mine) {
                const int at = __builtin_ctzll(mine);
                expert = first + at;
                const int height = __builtin_amdgcn_readlane(high, at) * 64;
                const int before = (bm - __builtin_amdgcn_readlane(end - own, at)) * height;
                const int left = __builtin_amdgcn_readlane(rows, at) - before;
                m0 = __builtin_amdgcn_readlane(lo, at) + before;
                m1 = m0 + (left < height ? left : height);
                return;
            }
            bm -= __builtin_amdgcn_readlane(end, 63);
        }
}

#define PT_WAVES 4
#define PT_RUN 4               // tiles of one row tile that an XCD takes together (1, 2, 4: alike; 7, 14: slower)
#define PT_AS3(p) ((__attribute__((address_space(3))) void*)(p))

// Buffers that a workgroup keeps for stages of x and of W, in `rows` lines of 128 bytes: of W, which comes from memory, one
// more than of x, which comes out of the XCD's cache, where there is room for it.  (Still more of W gain nothing:
// copies land in order, so those of x that the next stage needs wait for all of W asked for before them.)
struct PtRings {
    int x, w;
};
constexpr PtRings pt_rings(int rows, int bm, int bn) {
    PtRings best{0, 0};
    for (int n = 2; n <= 5 && n * (bm + bn) <= rows; ++n) best = {n, n * (bm + bn) + bn <= rows ? n + 1 : n};
    return best;
}

// One tile of up to 64 TM rows: rows m0 .. m1 - 1, all of expert e, columns from n0 on, within LDS bytes of shared
// memory.
template <int TM, int TN, int MODE, int LDS>
__device__ __forceinline__ void pt_tile(const PtArgs& g, char* lds, int e, int m0, int m1, int n0) {
    constexpr int BM = 64 * TM, BN = 64 * TN;
    constexpr int UX = BM / 32, UW = BN / 32, U = UX + UW;       // 1 KB copies (8 rows) of a wave and stage
    constexpr PtRings RING = pt_rings(LDS / 128, BM, BN);
    constexpr int NX = RING.x, NW = RING.w, XS = BM * 128, WS = BN * 128, W0 = NX * XS;
    static_assert(NX >= 2 && (NX - 1) * U + UW < 64, "stages under way, counted by the wait");
    const int F = g.F, N = MODE == PT_GATE ? 2 * F : F;          // columns of out, rows of an expert's W
    const int K = g.K;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave & 1, wc = wave >> 1;
    const bf16_t* we = g.w + (size_t)e * N * K;
    // row of x and row of W that row r of the tile stands for; beyond the last one it again, never stored
    auto x_row = [&](int r) {
        const int m = m0 + r < m1 ? m0 + r : m1 - 1;
        return g.order ? g.order[m] / g.top : m;
    };
    auto w_row = [&](int r) {
        if (MODE != PT_GATE) return n0 + r < F ? n0 + r : F - 1;
        const int n = n0 + (r >> 6) * 32 + (r & 31);             // 32 gate rows, then the same up rows
        return (n < F ? n : F - 1) + ((r >> 5) & 1) * F;
    };
#define PT_SWIZZLE(r) (((r) >> 1) & 7)
    const int T = K / 64;                                        // stages of the whole product
    // experts begin at different stages: their matrices are often a power of two apart, and walked in step from
    // the first one they meet in the same memory channels (32 experts of 4,096 x 4,096, 40 tokens: 266 -> 190 us).  By the
    // expert alone, so that a row's sums have one order in every tile of this file.  Groups of an expert's column tiles
    // with stages of their own, 128 or 256 columns wide as the tile, gained nothing behind the rings: 7,108 rows of 32, 4,096 -> 3,584
    // 294 us with, 295 without, 3,584 -> 4,096 271, 272; 16 x 250, 4,096 x 4,096 171, 175; 32 x 64, 4,096 -> 3,584 185, 183.
    const int turn = e * 8 % T;
    const char* xp[UX];
    uint32_t wo[UW];
#pragma unroll
    for (int i = 0; i < UX; ++i) {
        const int r = (wave + PT_WAVES * i) * 8 + (lane >> 3), c = (lane & 7) ^ PT_SWIZZLE(r);
        xp[i] = (const char*)(g.x + (size_t)x_row(r) * K) + c * 16;
    }
    const int wfirst = MODE == PT_GATE ? 0 : n0;
#pragma unroll
    for (int i = 0; i < UW; ++i) {
        const int r = (wave + PT_WAVES * i) * 8 + (lane >> 3), c = (lane & 7) ^ PT_SWIZZLE(r);
        wo[i] = (uint32_t)(w_row(r) - wfirst) * (uint32_t)(K * 2) + c * 16;
    }
    const char* wbase = (const char*)(we + (size_t)wfirst * K);
    const uint32_t lds_at = (uint32_t)(uintptr_t)PT_AS3(lds);
    // copy i of the wave (x first) into x's buffer bx or W's bw, of the stage NX or NW behind stage t; not beyond the last
#define PT_COPY(i, t, bx, bw) do { \
        constexpr bool X = (i) < UX; \
        const uint32_t to = __builtin_amdgcn_readfirstlane(lds_at + (X ? (bx) * XS : W0 + (bw) * WS) + \
                            (wave + PT_WAVES * (X ? (i) : (i) - UX)) * 1024); \
        const int stage = (t) + (X ? NX : NW) < T ? (t) + (X ? NX : NW) : T - 1; \
        const size_t at = (size_t)(uint32_t)__builtin_amdgcn_readfirstlane(stage + turn < T ? stage + turn : stage + turn - T) * 128; \
        if (X) \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" \
                         :: "s"(to), "v"(xp[X ? (i) : 0] + at) : "memory", "m0"); \
        else \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" \
                         :: "s"(to), "v"(wo[X ? 0 : (i) - UX]), "s"(wbase + at) : "memory", "m0"); \
    } while (0)

    const int hi = lane >> 5, swizzle = PT_SWIZZLE(lane & 31);
    const int x_at = (wr * TM * 32 + (lane & 31)) * 128, w_at = W0 + (wc * TN * 32 + (lane & 31)) * 128;
    int chunk[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) chunk[s] = ((2 * s + hi) ^ swizzle) * 16;
    pt_floatx16_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
    PtFrag a0[TN], b0[TM], a1[TN], b1[TM];
#define PT_READ(bx, bw, s, A, B, q) do { \
        if ((q) < TN) A[(q) < TN ? (q) : 0].u = *(const uint4*)(lds + (bw) * WS + w_at + chunk[s] + (q) * 4096); \
        else B[(q) < TN ? 0 : (q) - TN].u = *(const uint4*)(lds + (bx) * XS + x_at + chunk[s] + ((q) - TN) * 4096); \
    } while (0)
    // the products of operands A, B; between them the reads of the next 16 k (step s of buffers bx, bw) into NA, NB, and
    // copies C0 .. C1 - 1 of the stages behind t into buffers tx, tw
#define PT_STEP(A, B, READ, bx, bw, s, NA, NB, C0, C1, t, tx, tw) do { \
        _Pragma("unroll") for (int q = 0; q < TN * TM; ++q) { \
            acc[q / TM][q % TM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[q / TM].v, B[q % TM].v, acc[q / TM][q % TM], 0, 0, 0); \
            if (READ) { _Pragma("unroll") for (int r = 0; r < TN + TM; ++r) \
                if (r * (TN * TM) / (TN + TM) == q) PT_READ(bx, bw, s, NA, NB, r); } \
            pt_copies<C0, C1>([&](auto i) { \
                if ((i.value - (C0)) * (TN * TM) / ((C1) - (C0)) == q) PT_COPY(i.value, t, tx, tw); }); \
            __builtin_amdgcn_sched_barrier(0); \
        } \
    } while (0)
    // all but the newest n copies of every wave have landed, and every wave has read its operands
#define PT_SYNC(n) do { \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(n) : "memory"); \
        __builtin_amdgcn_s_barrier(); \
        asm volatile("" ::: "memory"); \
    } while (0)
    // The copies between two waits, x's first: those before CA in the last step of the stage whose buffers they take,
    // those before CB, CC, U in the first steps of the next.
    constexpr int CA = UX, CB = UX + UW / 3;
    // How many copies a wave may still have under way when it goes on to the next stage, R stages being left behind
    // this one: those behind the next stage's.  Between two waits x's copies of one stage come first, then W's of one
    // NW - NX stages later.
    auto left = [](int R) constexpr {
        int n = 0;
        for (int j = 0; j <= NX - 2; ++j) {
            if (j < NX - 2 && NX - 1 - j <= R) n += UX;
            if ((j < NX - 2 || NX < NW) && NW - 1 - j <= R) n += UW;
        }
        return n;
    };
    pt_copies<0, NW - 1>([&](auto s) {                           // as if the waits before the first stage had been
        constexpr int t = s.value - (NW - 1);
        if constexpr (t + NX - 1 >= 0) pt_copies<0, UX>([&](auto i) { PT_COPY(i.value, t - 1, t + NX - 1, 0); });
        pt_copies<UX, U>([&](auto i) { PT_COPY(i.value, t - 1, 0, s.value); });
    });
    pt_copies<0, CA>([&](auto i) { PT_COPY(i.value, -1, NX - 1, NW - 1); });
    PT_SYNC(left(NW) + CA);
#pragma unroll
    for (int r = 0; r < TN + TM; ++r) PT_READ(0, 0, 0, a0, b0, r);
    int t = 0, bx = 0, bw = 0;                                   // the stage, its buffers: t modulo NX, NW
    // stage t, R stages behind it (NW: or more), whose copies alone are asked for: first what is left of the copies
    // between the last wait and this stage's, then those behind it
#define PT_STAGE(R) do { \
        constexpr bool X1 = (R) >= NX - 1, W1 = (R) >= NW - 1, X2 = (R) >= NX, W2 = (R) >= NW; \
        constexpr int END = W1 ? U : X1 ? UX : 0, E2 = W2 ? U : X2 ? UX : 0; \
        constexpr int S0 = CA < END ? CA : END, S1 = CB < END ? CB : END; \
        constexpr int S2 = (CB + U) / 2 < END ? (CB + U) / 2 : END, S3 = CA < E2 ? CA : E2; \
        const int px = bx == 0 ? NX - 1 : bx - 1, pw = bw == 0 ? NW - 1 : bw - 1; \
        const int nx = bx == NX - 1 ? 0 : bx + 1, nw = bw == NW - 1 ? 0 : bw + 1; \
        PT_STEP(a0, b0, true, bx, bw, 1, a1, b1, S0, S1, t - 1, px, pw); \
        PT_STEP(a1, b1, true, bx, bw, 2, a0, b0, S1, S2, t - 1, px, pw); \
        PT_STEP(a0, b0, true, bx, bw, 3, a1, b1, S2, END, t - 1, px, pw); \
        if constexpr ((R) > 0) PT_SYNC(left(R)); \
        PT_STEP(a1, b1, (R) > 0, nx, nw, 0, a0, b0, 0, S3, t, bx, bw); \
        bx = nx; \
        bw = nw; \
    } while (0)
    for (; t < T - NW; ++t) PT_STAGE(NW);
    pt_copies<0, NW>([&](auto i) {                               // the last NW
        constexpr int R = NW - 1 - i.value;
        if (R < T) {
            t = T - 1 - R;
            PT_STAGE(R);
        }
    });
    PT_SYNC(0);

    // The tile leaves through shared memory as float32, 32 rows of a wave at a time, so that what follows is a
    // short loop that stores whole rows of the wave's columns.  (Unrolled over the accumulators, with every
    // activation, the code was 200 KB; fetching it took longer than the products of a tile.)
    constexpr int PITCH = TN * 128 + 16;
    constexpr int WN = (MODE == PT_GATE ? TN / 2 : TN) * 32, UNITS = WN / 8;     // columns of a wave, eight a unit
    char* mine = lds + wave * 32 * PITCH;
    const int c0 = n0 + wc * WN;
#pragma unroll 1
    for (int j = 0; j < TM; ++j) {
        pt_copies<0, TM>([&](auto J) {
            if (j == J.value)
#pragma unroll
                for (int i = 0; i < TN; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *(pt_floatx4_t*)(mine + (lane & 31) * PITCH + (i * 32 + 8 * q + 4 * hi) * 4) =
                            pt_floatx4_t{acc[i][J.value][4 * q], acc[i][J.value][4 * q + 1],
                                         acc[i][J.value][4 * q + 2], acc[i][J.value][4 * q + 3]};
        });
        __builtin_amdgcn_wave_barrier();                         // a wave's own accesses are in order
#pragma unroll 1
        for (int u = lane; u < 32 * UNITS; u += 64) {
            const int row = u / UNITS, unit = u % UNITS;
            const int m = m0 + (wr * TM + j) * 32 + row, n = c0 + unit * 8;
            if (m >= m1 || n >= F) continue;                     // F is a multiple of eight
            const char* from = mine + row * PITCH + (MODE == PT_GATE ? (unit / 4) * 256 + (unit % 4) * 32 : unit * 32);
            float z[8];
            *(pt_floatx4_t*)z = *(const pt_floatx4_t*)from;
            *(pt_floatx4_t*)(z + 4) = *(const pt_floatx4_t*)(from + 16);
            if (MODE == PT_GATE) {
                float up[8];
                *(pt_floatx4_t*)up = *(const pt_floatx4_t*)(from + 128);
                *(pt_floatx4_t*)(up + 4) = *(const pt_floatx4_t*)(from + 144);
                pt_gate(z, up, g.act, g.limit);
            } else {
                pt_act(z, g.act);
            }
            *(uint4*)((bf16_t*)g.out + (size_t)m * F + n) =
                make_uint4((uint32_t)float_to_bf16(z[0]) | ((uint32_t)float_to_bf16(z[1]) << 16),
                           (uint32_t)float_to_bf16(z[2]) | ((uint32_t)float_to_bf16(z[3]) << 16),
                           (uint32_t)float_to_bf16(z[4]) | ((uint32_t)float_to_bf16(z[5]) << 16),
                           (uint32_t)float_to_bf16(z[6]) | ((uint32_t)float_to_bf16(z[7]) << 16));
        }
        __builtin_amdgcn_wave_barrier();
    }
#undef PT_COPY
#undef PT_READ
#undef PT_STEP
#undef PT_STAGE
#undef PT_SYNC
#undef PT_SWIZZLE
}

template <int TM, int TN, int MODE>
__global__ __launch_bounds__(PT_WAVES * 64, (TM + TN) * 64 * 256 <= 80 * 1024 ? 2 : 1)
void prompt_tile_kernel(const PtArgs g) {
    constexpr int BM = 64 * TM, BN = 64 * TN;
    // Tall tiles are as high as their rows: an expert's rest is often far below 256, and a tile of 64, 128 or 192
    // rows takes fewer copies and products; the highest go first, so that the last round is one of low tiles.
    // Whole prompts, all tiles 256 high, heights by the rows, and highest first: 1,777 tokens of 32 experts of
    // 2 x 4,096 x 3,584 13.06, 12.84, 12.27 ms; 2,048 tokens 13.85, 13.50, 13.20; eight prompts of 100 to 500 18.5, 18.1,
    // 17.6; of gated experts of 3 x 4,096 x 2,048 four of 600 to 1,000 20.55, 20.55, 20.2, one of 2,048 14.1, 13.9, 13.95.
    constexpr bool EVEN = TM == 4;
    constexpr int G = 4;                                         // row tiles that run through the columns together
    constexpr int LDS = ((TM + TN) * 64 * 256 <= 80 * 1024 ? 80 : 160) * 1024;     // two workgroups to a compute unit, or one
    __shared__ __attribute__((aligned(1024))) char lds[LDS];

    const int F = g.F;
    constexpr int CN = MODE == PT_GATE ? BN / 2 : BN;            // columns of out that a tile makes
    const int mt = pt_row_tiles<BM>(g.offsets, g.E), nt = (F + CN - 1) / CN;
    const int total = mt * nt, turn = blockIdx.x >> 3;
    int bm, bn;
    if (EVEN) {
        // the XCDs (every eighth workgroup each) take runs of columns of a row tile in turn, so that each gets its
        // share of every height and the highest begin first
        const int work = ((turn / PT_RUN) * 8 + (blockIdx.x & 7)) * PT_RUN + turn % PT_RUN;
        if (work >= total) return;                               // the whole workgroup
        bm = work / nt;
        bn = work - bm * nt;
    } else {
        // the workgroups of one XCD take consecutive tiles
        const int per = (total + 7) / 8, work = (blockIdx.x & 7) * per + turn;
        if (turn >= per || work >= total) return;
        const int group = work / (G * nt), in_group = work - group * G * nt;
        const int group_rows = mt - group * G < G ? mt - group * G : G;
        bm = group * G + in_group % group_rows;
        bn = in_group / group_rows;
    }
    int m0 = 0, m1 = 0, e = 0;
    pt_find_tile<BM, EVEN>(g.offsets, g.E, bm, e, m0, m1);
    if constexpr (EVEN) {
        if (m1 - m0 <= 64) return pt_tile<1, TN, MODE, LDS>(g, lds, e, m0, m1, bn * CN);
        if (m1 - m0 <= 128) return pt_tile<2, TN, MODE, LDS>(g, lds, e, m0, m1, bn * CN);
        if (m1 - m0 <= 192) return pt_tile<3, TN, MODE, LDS>(g, lds, e, m0, m1, bn * CN);
    }
    pt_tile<TM, TN, MODE, LDS>(g, lds, e, m0, m1, bn * CN);
}
