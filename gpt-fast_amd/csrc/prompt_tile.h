// The tile kernel of the experts' products with many rows: out = x W[e]^T in bfloat16 with float32 sums, the
// rows of x being sorted by expert.
//
// A workgroup of four waves makes a tile of 64 TM rows of x by 64 TN rows of W, each wave a quarter
// (32 TM x 32 TN) with v_mfma_f32_32x32x16_bf16, formed transposed (A = W, B = x) so that a lane ends with
// four consecutive columns of one row.  (The 32 x 32 form reads half as many operand registers per flop as
// 16 x 16 x 32; under the chip's power limit a bare loop of it reaches 1.86 PFLOP/s on random operands
// against 1.65.)  K is walked in pieces of 64, one 128-byte line per row, which are copied straight into
// shared memory (global_load_lds, 16 bytes a lane) two buffers deep, their 16-byte chunks swizzled by the
// row so that operand reads have no bank conflicts.
//
// What bounds it is the path into a compute unit, not the arithmetic: at 256 x 256 a piece takes 2,048
// cycles of the matrix units and 64 KB of copies.  Hence:
//  * operands of the next 16 k are read between the products of this one, one read per two products, and
//    the one barrier of a piece stands before its last 16 k, so that nothing waits behind it;
//  * copies are spread over three of a piece's four steps instead of issued in a burst (a burst fills the
//    address unit and holds the products up);
//  * in the tile that fills a compute unit by itself, the lines of W are asked for two pieces before they are
//    copied (one dword of 64 lines per instruction, into shared memory that nobody reads), so that the copies find
//    them in the XCD's cache.
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

// One tile of up to 64 TM rows: rows m0 .. m1 - 1, all of expert e, columns from n0 on.  ASK: the lines of W are
// asked for ahead.
template <int TM, int TN, int MODE, bool ASK>
__device__ __forceinline__ void pt_tile(const PtArgs& g, char* lds, int e, int m0, int m1, int n0) {
    constexpr int BM = 64 * TM, BN = 64 * TN;
    constexpr int UX = BM / 32, UW = BN / 32, U = UX + UW;       // 1 KB copies (8 rows) of a wave and piece
    constexpr int XB = BM * 128, BUF = (BM + BN) * 128;
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
    const int T = K / 64;                                        // pieces
    // experts begin at different pieces: their matrices are often a power of two apart, and walked in step from
    // the first piece they meet in the same memory channels (32 experts of 4,096 x 4,096, 40 tokens: 266 -> 190 us)
    const int turn = (e * 8) % T;
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

    // the line (of the pieces to come) that this lane asks for: one of the tile's rows of W
    const char* line = nullptr;
    if (ASK) {
        static_assert(BN / PT_WAVES <= 64, "a lane asks for one line");
        line = (const char*)(we + (size_t)w_row(wave * (BN / PT_WAVES) + lane % (BN / PT_WAVES)) * K);
    }
    const uint32_t lds_at = (uint32_t)(uintptr_t)PT_AS3(lds);
    // copy i of the wave (x first) of piece t into buffer b
#define PT_COPY(i, t, b) do { \
        constexpr bool X = (i) < UX; \
        const uint32_t to = __builtin_amdgcn_readfirstlane(lds_at + (b) * BUF + (X ? 0 : XB) + \
                            (wave + PT_WAVES * (X ? (i) : (i) - UX)) * 1024); \
        const size_t at = (size_t)(uint32_t)__builtin_amdgcn_readfirstlane((t) + turn < T ? (t) + turn : (t) + turn - T) * 128; \
        if (X) \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" \
                         :: "s"(to), "v"(xp[X ? (i) : 0] + at) : "memory", "m0"); \
        else \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" \
                         :: "s"(to), "v"(wo[X ? 0 : (i) - UX]), "s"(wbase + at) : "memory", "m0"); \
    } while (0)
#define PT_ASK(t) do { if (ASK) { \
        const int piece = ((t) < T ? (t) : T - 1) + turn; \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" \
                     :: "s"(__builtin_amdgcn_readfirstlane(lds_at + 2 * BUF + wave * 256)), \
                        "v"(line + (size_t)(piece < T ? piece : piece - T) * 128) : "memory", "m0"); \
    } } while (0)

    const int hi = lane >> 5, swizzle = PT_SWIZZLE(lane & 31);
    const int x_at = (wr * TM * 32 + (lane & 31)) * 128, w_at = XB + (wc * TN * 32 + (lane & 31)) * 128;
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
#define PT_READ(b, s, A, B, q) do { \
        if ((q) < TN) A[(q) < TN ? (q) : 0].u = *(const uint4*)(lds + (b) * BUF + w_at + chunk[s] + (q) * 4096); \
        else B[(q) < TN ? 0 : (q) - TN].u = *(const uint4*)(lds + (b) * BUF + x_at + chunk[s] + ((q) - TN) * 4096); \
    } while (0)
    // the products of operands A, B; between them the reads of the next 16 k (step s of buffer b) into NA, NB
    // and copies C0 .. C1 - 1 of piece t into buffer to
#define PT_STEP(A, B, b, s, NA, NB, C0, C1, t, to) do { \
        _Pragma("unroll") for (int q = 0; q < TN * TM; ++q) { \
            acc[q / TM][q % TM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[q / TM].v, B[q % TM].v, acc[q / TM][q % TM], 0, 0, 0); \
            _Pragma("unroll") for (int r = 0; r < TN + TM; ++r) \
                if (r * (TN * TM) / (TN + TM) == q) PT_READ(b, s, NA, NB, r); \
            pt_copies<C0, C1>([&](auto i) { \
                if ((i.value - (C0)) * (TN * TM) / ((C1) - (C0)) == q) PT_COPY(i.value, t, to); }); \
            __builtin_amdgcn_sched_barrier(0); \
        } \
    } while (0)
    // everything but the newest request (the line asked for ahead) has landed, in every wave
#define PT_SYNC(n) do { \
        asm volatile("s_waitcnt vmcnt(" #n ") lgkmcnt(0)" ::: "memory"); \
        __builtin_amdgcn_s_barrier(); \
        asm volatile("" ::: "memory"); \
    } while (0)
    constexpr int C0 = (U * 5 + 15) / 16, C1 = (U * 10 + 15) / 16;      // copies of the first, first two steps
    pt_copies<0, U>([&](auto i) { PT_COPY(i.value, 0, 0); });
    PT_ASK(1);
    if (ASK) PT_SYNC(1); else PT_SYNC(0);
    int t1 = T > 1 ? 1 : 0;                                       // the piece whose copies are under way
    pt_copies<0, C0>([&](auto i) { PT_COPY(i.value, t1, 1); });
#pragma unroll
    for (int r = 0; r < TN + TM; ++r) PT_READ(0, 0, a0, b0, r);
    for (int t = 0; t < T; ++t) {
        const int b = t & 1;
        PT_STEP(a0, b0, b, 1, a1, b1, C0, C1, t1, b ^ 1);
        PT_STEP(a1, b1, b, 2, a0, b0, C1, U, t1, b ^ 1);
        PT_ASK(t + 2);
        PT_STEP(a0, b0, b, 3, a1, b1, U, U, 0, 0);
        if (ASK) PT_SYNC(1); else PT_SYNC(0);
        // behind the last piece: its copies once more, and operands that nothing multiplies
        t1 = t + 2 < T ? t + 2 : T - 1;
        PT_STEP(a1, b1, b ^ 1, 0, a0, b0, 0, C0, t1, b);
    }
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
#undef PT_ASK
#undef PT_READ
#undef PT_STEP
#undef PT_SYNC
}

template <int TM, int TN, int MODE>
__global__ __launch_bounds__(PT_WAVES * 64, (TM + TN) * 64 * 256 <= 80 * 1024 ? 2 : 1)
void prompt_tile_kernel(const PtArgs g) {
    constexpr int BM = 64 * TM, BN = 64 * TN, BUF = (BM + BN) * 128;
    // asking ahead pays where no second workgroup shares the compute unit (1,777 tokens of 32 experts, W 3,584 x
    // 4,096: tiles of 256 x 256 374 -> 368 us, 256 x 128 409 -> 384, but 128 x 128 368 -> 432)
    constexpr bool ASK = (BM + BN) * 256 > 80 * 1024;
    // Tall tiles are as high as their rows: an expert's rest is often far below 256, and a tile of 64, 128 or 192
    // rows takes fewer copies and products; the highest go first, so that the last round is one of low tiles.
    // Whole prompts, all tiles 256 high, heights by the rows, and highest first: 1,777 tokens of 32 experts of
    // 2 x 4,096 x 3,584 13.06, 12.84, 12.27 ms; 2,048 tokens 13.85, 13.50, 13.20; eight prompts of 100 to 500 18.5, 18.1,
    // 17.6; of gated experts of 3 x 4,096 x 2,048 four of 600 to 1,000 20.55, 20.55, 20.2, one of 2,048 14.1, 13.9, 13.95.
    constexpr bool EVEN = TM == 4;
    constexpr int G = 4;                                         // row tiles that run through the columns together
    __shared__ __attribute__((aligned(1024))) char lds[2 * BUF + (ASK ? PT_WAVES * 256 : 0)];

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
    if (EVEN && m1 - m0 <= 64) pt_tile<1, TN, MODE, ASK>(g, lds, e, m0, m1, bn * CN);
    else if (EVEN && m1 - m0 <= 128) pt_tile<2, TN, MODE, ASK>(g, lds, e, m0, m1, bn * CN);
    else if (EVEN && m1 - m0 <= 192) pt_tile<3, TN, MODE, ASK>(g, lds, e, m0, m1, bn * CN);
    else pt_tile<TM, TN, MODE, ASK>(g, lds, e, m0, m1, bn * CN);
}
