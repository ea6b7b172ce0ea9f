// Plain decoder layers over a few rows (decoding, short prompts) in one launch whose workgroups stay on their
// compute units through all layers.  Every layer has the phases
//   0  q/k/v projection, rotation, cache write      3  gate product
//   1  attention over the paged cache               4  second feed-forward product, into the stream
//   2  output projection, into the stream
// of h = x + wo attention(norm(x)), out = h + w2 (act(w1 norm(h)) * (w3 norm(h))) (model.py:161-227), the norms in two
// halves as in gemm_bf16.hip: the product in front leaves bfloat16(stream * weight) and shares of the rows' sums of
// squares, the one behind scales its result.
//
// What bounds it is the stream of the weights.  Launched one by one (gemm_bf16.hip), every phase loses 4 to 5 us of it: the
// last workgroups of a kernel finish, the next one starts and asks for its first weights, and a few compute units
// work alone while attention runs.  But the weights depend on nothing.  So eight waves of every workgroup (streamers) do
// nothing but read weights and multiply.  While a product's x is there each has RL_RING blocks of 16 rows x 128 columns
// (16 KB) under way in registers, across the ends of tiles; behind its last tile it asks for the next product's first
// blocks, RL_PACE at a time: a chip's worth of loads in flight makes every store, counter and poll of the phases' meeting
// wait behind it, and asking for all of them at once, or more into the second-level cache, measured slower (8B, 1 row,
// 16 counters: 2741 us a step; two at a time 2820, all at once 2830, three more blocks into the cache 3000).  The other four waves: one
// waits for the phase before and finishes the products (sum over the streamers, norm, rotation, gate, residual,
// stores), three bring x into shared memory and work on attention.
//
// Loads of 4 rows x 256 bytes, past the caches, stream at 7.0 TB/s, 16 rows x 64 bytes (the
// order of the matrix cores' operands) at 6.0: so the blocks pass through a piece of shared memory of the wave's own.
//
// Measured, us a decode step, five launches a layer -> this: 110M shape (12 layers, 768 wide) 1 row 333 -> 286,
// 8 rows of 200 keys 375 -> 317; 8B shape 1 row of 200 keys 2990 -> 2660 (its weights take 2150 at 7.0 TB/s, the head's with
// them), 8 rows 3090 -> 2896; 8 new tokens of one sequence behind 6000 keys 10300 -> 3710 (the
// attention of prompts has too few workgroups there).  What is left over the stream is the meetings, 1 to 4 us each under
// load, and attention, 5 and its own meeting.
//
// Between phases: results are stored through to memory (agent scope), and once they are there the workgroup adds
// one to one of 128 counters in lines of their own; the next phase polls all of them, two a lane.  Additions to a line wait for one
// another, longer the more loads are under way: with 8, 16, 32, 64, 128 counters a step of the 110M shape takes 323, 306, 293, 286,
// 286 us at 1 row and 376, 352, 336, 321, 317 at 8 rows, of the 8B shape 2800, 2746, 2700, 2676, 2660 and 3084, 2998, 2952, 2917, 2896; lines of 128 and 512
// bytes take as long as these of 256.  (256 workgroups that do nothing else meet in 1.3 us with 16, 3.9 with one, 2.2 to 3.2
// with a flag each.)  What a phase leaves is read at agent scope
// like the counters, and lies in memory that this launch has not read before: every layer has its own buffers.  Workgroups of several dies
// write parts of one line (of a norm's shares, four bytes each), and a cache that holds such a line after its own part was stored through may
// not be believed about the others.  That order between workgroups is the hardware's (stores at agent scope, vmcnt(0), an addition;
// a poll that sees it, then loads at agent scope), not the language's, whose fences write back and drop second-level caches that
// hold nothing of this: us a step, 110M shape 1 row, 8B shape 1 and 8 rows: 256, 2492, 2723 without; with the acquiring
// fences 315, 2631, 2840, with both 527, 4120, 4346; reading at agent scope instead of through the caches costs nothing, 257, 2482, 2706.
// The counters only grow: nothing arrives for a phase before the one in front of it is complete.
//
// Waiting cannot lock up, whatever part of the grid the chip has room for: nothing is waited for but workgroups that
// run.  A phase's work is cut into as many parts as the grid has workgroups.  They are counted at the start: if all are there,
// workgroup b takes part b of every phase.  If some are not there after a while (another launch holds their place), those that
// run close the list and share all parts among themselves, worker v of V taking parts v, v + V, ...; what starts later
// waits for the next layer, in front of which the list is made anew, until all are there.  So a launch that begins on a busy chip has the
// rest of it as soon as it is free, and every result has the same bits whoever worked it out.
#include "few_row_layers.h"
#include <cstring>

#define AGENT __HIP_MEMORY_SCOPE_AGENT
#define RL_STREAMERS 8                // waves that read weights
#define RL_THREADS 768                // and four others
#define RL_RING 4                     // blocks of weights that a streamer has under way
#define RL_PACE 1                     // blocks that a streamer has under way between two products
#define RL_MAX_LAYERS 32              // of one launch: their pointers are kernel arguments
#define RL_MAX_ROWS 16
#define RL_PIECE 128                  // columns of a block: 16 rows x 256 bytes
#define RL_PITCH 272                  // bytes of a block's row in shared memory: 16 more, against conflicts
#define RL_STAGE (16 * RL_PITCH)
#define RL_X_BYTES (88 * 1024)        // x: whole if it fits, else two halves in turn
#define RL_X_HALF (RL_X_BYTES / 2)
#define RL_SHARE 8                    // blocks of 32 keys that a share of a context has at least, and
#define RL_SHARE_COST 6               // blocks that a share costs beside its own
#define RL_SUMS (RL_STREAMERS * 2 * 64)   // floatx4 of a tile's partial sums
#define RL_COUNTERS 128
#define RL_LINE 64                    // ints from one counter to the next
#define RL_AT_AGENT 16                // cache policy of a load (sc1): as an atomic load at agent scope
#define RL_NOWHERE 0xfffff000u        // an offset behind every matrix: reads as zero
#define RL_MOST_BYTES 0xffff0000l
#define RL_MOST_COLUMNS (1 << 23)     // of a row of x: sixteen of them, and all buffers of a layer, have 32-bit offsets

typedef unsigned int rl_u4 __attribute__((ext_vector_type(4)));
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;

union RlFrag {
    rl_u4 u;
    bf16x8_t v;
    bf16_t e[8];
};

// What differs from phase to phase lies in tables by the phase (entry 1, attention, unused).  A chain of choices between
// fields instead (phase == 0 ? wqkv : phase == 2 ? ...) was compiled wrongly (clang 20, ROCm 7.2): the last alternative's address was
// never copied, so that one matrix was read with another one's size.
struct ResidentLayer {
    const bf16_t* w[5];
    const float* norm[5];                 // weights of the norm that the phase's result goes into (2, 4; null: none)
    bf16_t *k_pages, *v_pages;
    const int* table;
};

struct ResidentArgs {
    ResidentLayer layer[RL_MAX_LAYERS];
    int N[5], K[5], gate[5];              // rows and columns of W; rows between a column's two rows, or 0
    unsigned off_in[5];                   // rows that the phase's product multiplies
    unsigned off_out[5], off_share[5];    // 2, 4: the next norm's first half and the shares of its sums of squares; of 4 in the next layer
    unsigned off_sums[5];                 // 0, 3: those of the norm in front
    float eps[5];
    const float* norm_first;              // of the norm before the first layer
    float* residual;                      // [M, D], updated in place
    const float* freqs;
    const int *tok_seq, *tok_pos, *start_pos;
    int* words;                           // zero at the start: RlWords below
    char* work;                           // per layer work_stride bytes: the buffers below
    size_t work_stride;
    unsigned off_q;
    size_t off_po, off_pml;               // sums of the contexts' shares, behind the layers' buffers: one place for all layers,
                                          // read past the caches, written again only when the layer that read them is complete
    int n_layers, M, D, I, H, Hkv, hd, rot, table_stride, window, pad, gate_mode;
    int start_polls, seal_polls;          // polls before the list of workers is closed, and then the first layer's
    float scale_log2;
};

// The words of a launch, in ints: [0] groups of workgroups that are there and the closed bit, then the groups' and the phases'
// counters, per layer its list of workers (how many, how many of them worked on the layer before, the closed bit), then one word
// per (token, kv head) for its shares.
#define RL_CLOSED (1 << 30)
#define RL_BEFORE (1 << 15)
#define RL_COUNT (RL_BEFORE - 1)
#define RL_GROUPS 16
#define RL_LIST 16                    // ints from one list to the next
#define RL_AT_GROUPS RL_LINE
#define RL_AT_COUNTERS (RL_AT_GROUPS + RL_GROUPS * RL_LINE)
#define RL_AT_LISTS (RL_AT_COUNTERS + RL_COUNTERS * RL_LINE)
#define RL_AT_SPLITS (RL_AT_LISTS + RL_MAX_LAYERS * RL_LIST)
#define RL_MAX_POLLS (1 << 22)        // seconds: a wait that runs out leaves NaN

typedef const __attribute__((address_space(4))) ResidentArgs RlArgs;
typedef const __attribute__((address_space(4))) ResidentLayer RlLayer;

template <typename T> __device__ __forceinline__ void rl_put(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, AGENT); }
__device__ __forceinline__ void rl_put8(void* p, unsigned a, unsigned b) {
    __hip_atomic_store((unsigned long long*)p, (unsigned long long)b << 32 | a, __ATOMIC_RELAXED, AGENT);
}
template <typename T> __device__ __forceinline__ T rl_get(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, AGENT); }
__device__ __forceinline__ float2 rl_get8(const float* p) {
    const unsigned long long v = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, AGENT);
    return make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
}
__device__ __forceinline__ rl_u4 rl_get16(const void* p) {
    const float2 lo = rl_get8((const float*)p), hi = rl_get8((const float*)p + 2);
    return rl_u4{__float_as_uint(lo.x), __float_as_uint(lo.y), __float_as_uint(hi.x), __float_as_uint(hi.y)};
}
__device__ __forceinline__ void rl_all_landed() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);                    // vmcnt(0)
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ unsigned rl_two(float a, float b) {
    return (unsigned)float_to_bf16(a) | (unsigned)float_to_bf16(b) << 16;
}

// One part of a product of a layer.
struct RlProduct {
    const bf16_t* w;
    unsigned bytes;
    int K, gate;                          // gate: rows between a column's two rows of W, or 0
    int base, rows;                       // the part's rows of W, in tiles of sixteen; both multiples of four
    int pieces;                           // of 128 columns: those of the streamer that has the most
    int chunk, chunks;                    // pieces of x that lie in shared memory at a time; 1 chunk: all of x, as it is
};

// What is the same in every layer, worked out once and kept in shared memory.
struct RlPlan {
    int N, share, K, gate;                // share: rows of a part
    int pieces, chunk, chunks, arrivals;  // arrivals: parts that have rows
    unsigned bytes, off_in, off_out, off_share;
    unsigned off_sums, unused[3];
};

template <typename Args>
__device__ __forceinline__ void rl_make_plan(const Args& a, RlPlan* plan, int phase, int parts) {
    RlPlan t = {};
    const int N = a.N[phase], share = ((N >> 2) + parts - 1) / parts * 4;
    t.N = N;
    t.share = share;
    t.K = a.K[phase];
    t.gate = a.gate[phase];
    t.bytes = (unsigned)(N + t.gate) * (unsigned)t.K * 2u;
    t.arrivals = share > 0 ? (N + share - 1) / share : 0;
    const int T = (t.K + RL_PIECE - 1) / RL_PIECE;
    t.pieces = (T + RL_STREAMERS - 1) / RL_STREAMERS;
    if (T * RL_PIECE * 2 * a.pad <= RL_X_BYTES) {
        t.chunk = t.pieces;
        t.chunks = 1;
    } else {
        t.chunk = RL_X_HALF / (RL_STREAMERS * RL_PIECE * 2 * a.pad);
        if (a.pad < 4) t.chunk &= -(4 / a.pad);            // whole KB of every streamer
        t.chunks = (t.pieces + t.chunk - 1) / t.chunk;
    }
    t.off_in = a.off_in[phase];
    t.off_out = a.off_out[phase];
    t.off_share = a.off_share[phase];
    t.off_sums = a.off_sums[phase];
    plan[phase] = t;
}

__device__ __forceinline__ int rl_same(int x) { return __builtin_amdgcn_readfirstlane(x); }

template <typename Args>
__device__ __forceinline__ RlProduct rl_product(const Args& a, const RlPlan* plan, int layer, int phase, int part) {
    RlProduct p;
    const bool is = layer < a.n_layers;                    // behind the last layer: a product without rows
    p.w = a.layer[is ? layer : 0].w[phase];
    const RlPlan t = plan[phase];
    p.bytes = rl_same(t.bytes);
    p.K = rl_same(t.K);
    p.gate = rl_same(t.gate);
    const int share = rl_same(t.share), left = rl_same(t.N) - part * share;
    p.base = part * share;
    p.rows = !is || left <= 0 ? 0 : left < share ? left : share;
    p.pieces = rl_same(t.pieces);
    p.chunk = rl_same(t.chunk);
    p.chunks = rl_same(t.chunks);
    return p;
}
// First piece of streamer s.
__device__ __forceinline__ int rl_first_piece(int K, int s) {
    return s * ((K + RL_PIECE - 1) / RL_PIECE) / RL_STREAMERS;
}

// The place of the next block to ask for.
struct RlCursor {
    RlProduct p;
    int first, own;                       // this streamer's pieces
    int row, left, piece, set;            // first row of the tile, rows left, piece within them, row set (gate)
};

__device__ __forceinline__ void rl_seek(RlCursor& c, const RlProduct& p, int streamer) {
    c.p = p;
    c.first = rl_first_piece(p.K, streamer);
    c.own = rl_first_piece(p.K, streamer + 1) - c.first;
    c.row = p.base;
    c.left = p.rows;
    c.piece = 0;
    c.set = 0;
}

// Asks for the block at the cursor and moves it on.  Rows beyond the worker's and columns beyond K read as zero and cost no
// traffic; so do blocks behind the last one.
__device__ __forceinline__ void rl_ask(RlCursor& c, rl_u4 (&regs)[4], int lane) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)c.p.w, 0, (int)c.p.bytes, 0x27000);
    const int k = (c.first + c.piece) * RL_PIECE + (lane & 15) * 8;
    const int left = c.piece < c.own ? c.left : 0;
    const unsigned off = ((unsigned)(c.row + c.set + (lane >> 4)) * (unsigned)c.p.K + (unsigned)k) * 2u;
    const unsigned step = (unsigned)c.p.K * 8u;
#pragma unroll
    for (int j = 0; j < 4; ++j)                            // 2: not kept in the caches
        regs[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, k < c.p.K && 4 * j < left ? off + j * step : RL_NOWHERE, 0, 2);
    if (c.p.gate != 0 && c.set == 0) {
        c.set = c.p.gate;
    } else {
        c.set = 0;
        if (++c.piece == c.p.pieces) {
            c.piece = 0;
            c.row += 16;
            c.left -= 16;
        }
    }
}

// A streamer's way through one product.  Meets the other waves at: what the phase reads is complete; x is in shared memory;
// every end of a chunk (with the tile's sums in shared memory at its last one).  The blocks go to two sums in turn: the
// gate's two sets of rows, or two partial sums of the same rows.
__device__ __forceinline__ void rl_stream(const RlProduct& p, const RlProduct& next, RlCursor& c, rl_u4 (&ring)[RL_RING][4],
                                          int streamer, int lane, int pad, const char* x_lds, char* stage, floatx4_t* sums) {
    if (p.rows > 0) {
        lds_barrier();
        lds_barrier();
    }
    const int fi = lane & 15, fg = lane >> 4;
    const int first = rl_first_piece(p.K, streamer), own = rl_first_piece(p.K, streamer + 1) - first;
    const bool gate = p.gate != 0;
    const int blocks = ((p.rows + 15) >> 4) * p.pieces * (gate ? 2 : 1);
    const int piece_bytes = RL_PIECE * 2 * pad;
    const char* x_own = x_lds + (p.chunks == 1 ? first : streamer * p.chunk) * piece_bytes + (fg * pad + (fi & (pad - 1))) * 16;
    char* put = stage + (lane >> 4) * RL_PITCH + (lane & 15) * 16;
    const char* get = stage + fi * RL_PITCH + fg * 16;
    floatx4_t acc[2] = {floatx4_t{0.f, 0.f, 0.f, 0.f}, floatx4_t{0.f, 0.f, 0.f, 0.f}};
    int tile = 0, piece = 0, chunk_begin = 0, half = 0;
    auto take = [&](int i) {                               // the block in slot i, into its piece of shared memory
#pragma unroll
        for (int j = 0; j < 4; ++j) *(rl_u4*)(put + 4 * j * RL_PITCH) = ring[i][j];
    };
    auto multiply = [&](int i) {
        __builtin_amdgcn_wave_barrier();                   // what other lanes wrote is read: not in front of the writes
        const char* xp = x_own + half + (piece - chunk_begin) * piece_bytes;
        RlFrag w[4], x[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) x[s].u = *(const rl_u4*)(xp + s * 64 * pad);
#pragma unroll
        for (int s = 0; s < 4; ++s) w[s].u = *(const rl_u4*)(get + s * 64);
        if ((first + piece + 1) * RL_PIECE > p.K) {        // columns beyond K: zeros, whatever lies there
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if ((first + piece) * RL_PIECE + s * 32 + fg * 8 >= p.K) x[s].u = rl_u4{0, 0, 0, 0};
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s].v, x[s].v, acc[i & 1], 0, 0, 0);
    };
    auto next_block = [&](int i) {
        if (gate && !(i & 1)) return;
        ++piece;
        if (piece == p.pieces || piece == chunk_begin + p.chunk) {
            if (piece == p.pieces) {
                floatx4_t* mine = sums + (tile & 1) * RL_SUMS + streamer * 128 + lane;
                mine[0] = gate ? acc[0] : acc[0] + acc[1];
                if (gate) mine[64] = acc[1];
                acc[0] = acc[1] = floatx4_t{0.f, 0.f, 0.f, 0.f};
                piece = 0;
                ++tile;
            }
            lds_barrier();
            chunk_begin = piece;
            if (p.chunks > 1) half ^= RL_X_HALF;
        }
    };
    int at = 0;
    for (; at + RL_RING < blocks; at += RL_RING) {
#pragma unroll
        for (int i = 0; i < RL_RING; ++i) {
            const bool live = piece < own;
            if (live) take(i);
            rl_ask(c, ring[i], lane);
            if (live) multiply(i);
            next_block(i);
        }
    }
    // The last blocks are worked on as they come, and only then the next product's are asked for: asking waits
    // until the memory takes it, which is as long as reading it, and others wait for these sums.
#pragma unroll
    for (int i = 0; i < RL_RING; ++i)
        if (at + i < blocks) {
            if (piece < own) {
                take(i);
                multiply(i);
            }
            next_block(i);
        }
    // And a few at a time: what others store, count and read between the phases would stand behind all of them.
    rl_seek(c, next, streamer);
#pragma unroll
    for (int i = 0; i < RL_RING; ++i) {
        if (i >= RL_PACE) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0f70 | (4 * (RL_PACE - 1)));   // vmcnt: all but the last RL_PACE - 1 blocks are here
            asm volatile("" ::: "memory");
        }
        rl_ask(c, ring[i], lane);
    }
}

// ---------------------------------------------------------------------------- the other waves

// x of one product, or a chunk of it, into shared memory, by three waves: copies that pass through no registers, all
// of them under way at once.  Of a chunk every streamer has its part.
__device__ __forceinline__ void rl_bring(const RlProduct& p, const char* x, int pad, int chunk_begin, char* to, int third, int lane) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, p.K * 2 * pad, 0x27000);
    const int piece_bytes = RL_PIECE * 2 * pad, T = (p.K + RL_PIECE - 1) / RL_PIECE;
    const int part = (p.chunks == 1 ? T * piece_bytes + 1023 : p.chunk * piece_bytes) >> 10;   // KB; whole ones (rl_product)
    const int all = p.chunks == 1 ? part : part * RL_STREAMERS;
#pragma unroll 1
    for (int n = third; n < all; n += 3) {
        int from = n << 10;
        if (p.chunks > 1) {
            // a streamer that has fewer pieces: what it does not multiply may be anything of x
            const int s = n / part;
            from = (rl_first_piece(p.K, s) + chunk_begin) * piece_bytes + ((n - s * part) << 10);
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(to + (n << 10)), 16, from + lane * 16, 0, 0, RL_AT_AGENT);
    }
    rl_all_landed();
}

// Attention of one token, one key/value head and one share of the context: three waves take its 32-key
// blocks in turn, with the operands and the arithmetic of attention_mfma_kernel (attention_bf16.hip) at one tile
// of rows, the heads of the group.
struct RlItem {
    int index, g, token, pair, split, splits;
    // first: shares of the tokens in front of each
    template <typename Args> __device__ __forceinline__ RlItem(const Args& a, const int* first, int item) {
        const int at = item / a.Hkv, lane = threadIdx.x & 63;
        index = item;
        g = item - at * a.Hkv;
        token = rl_same(__popcll(__ballot(lane < a.M && first[(lane & 15) + 1] <= at)));
        split = at - rl_same(first[token]);
        splits = rl_same(first[token + 1]) - rl_same(first[token]);
        pair = token * a.Hkv + g;
    }
};

// Shares of the tokens' contexts, all of one size: the smallest that makes one share a workgroup and kv head, or two if that is
// clearly less work for the one that has most, since one context may be far longer than the others.  By a wave, which
// sees the contexts as they are at this step: 8B, 8 rows of which one has 16000 keys, 4958 us with as many shares of
// each, 3740 so; contexts of one length take as long either way.
template <typename Args>
__device__ __forceinline__ void rl_make_shares(const Args& a, int* first, int lane) {
    const int t = lane & 15;
    int blocks = 0;
    if (t < a.M) {
        const int pos = a.tok_pos[t], lo = (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
        blocks = (pos >> 5) - (lo >> 5) + 1;
        blocks = blocks > 1 ? blocks : 1;
    }
    auto all = [&](int x) {
#pragma unroll
        for (int d = 8; d > 0; d >>= 1) x += __shfl_xor(x, d, GFA_WAVE);
        return rl_same(x);
    };
    int longest = blocks;
#pragma unroll
    for (int d = 8; d > 0; d >>= 1) {
        const int other = __shfl_xor(longest, d, GFA_WAVE);
        longest = longest > other ? longest : other;
    }
    // joining costs about as much a share as a block does: no more shares of a context than a share has blocks
    // (8B, 1 row: 2000 keys 3035 us in shares of 16, 2964 of 8; 6000 keys 3184 of 16, 3245 of 8, 3165 of 14)
    int least = RL_SHARE;
    for (const int n = rl_same(longest); least * least < n;) ++least;
    const int total = all(blocks);
    int most = (int)gridDim.x / a.Hkv;
    most = most > a.M ? most : a.M;
    auto size_for = [&](int n) {                           // ends: with one share a token there are M
        int size = (total + n - 1) / n;
        size = size > least ? size : least;
        while (all((blocks + size - 1) / size) > n) size += 1 + size / 16;
        return size;
    };
    const int once = size_for(most), twice = size_for(2 * most);
    const int size = 2 * twice + RL_SHARE_COST < once ? twice : once;
    int behind = (blocks + size - 1) / size;
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
        const int before = __shfl(behind, (lane & 48) | ((t - d) & 15), GFA_WAVE);
        if (t >= d) behind += before;
    }
    if (lane < 16) first[t + 1] = behind;
    if (lane == 0) first[0] = 0;
}

// FULL: heads of DS * 32 dims, no more and no fewer.
// A wave's part (wave 1, 2, 3): leaves its heads' maxima, sums and results in shared memory.  `ready` returns when the phase may begin.
template <int DS, bool FULL, typename Args, typename LayerT, typename Ready>
__device__ __forceinline__ void rl_attend(const Args& a, const LayerT& L, const char* work, const RlItem& it, char* smem,
                                          int wave, Ready&& ready) {
    constexpr int DT = DS * 2;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));                         // offsets worked out anew for every layer, not kept beside the rest
    const int li = lane & 15, lg = lane >> 4;
    const int hd = FULL ? DS * 32 : a.hd, R = a.H / a.Hkv, g = it.g;
    const int pos = a.tok_pos[it.token], seq = a.tok_seq[it.token];
    const int* pages = L.table + (size_t)seq * a.table_stride;
    const int lo = (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
    const int kb_lo = lo >> 5, nkb = (pos >> 5) - kb_lo + 1;
    const int kb_begin = kb_lo + it.split * nkb / it.splits;
    const int kb_end = kb_lo + (it.split + 1) * nkb / it.splits;
    const bool valid = li < R;
    // Nothing of this token's products is needed to find the pages, nor for blocks of keys that lie wholly in front of this
    // step's tokens: the first block is asked for before what this phase waits for is complete.
    RlFrag kf[2][DS], vf[DT];
    const int key_lane = lg * 512 + li * 16, value_lane = lane * 16;   // bytes
    auto region = [&](bf16_t* pages_of, int page) {
        return __builtin_amdgcn_make_buffer_rsrc(pages_of + cache_region(rl_same(page), g, a.Hkv, hd), 0, GFA_PAGE * hd * 2, 0x27000);
    };
    auto ask_keys = [&](int page, int kb) {                // dims beyond the head read as zero
        const auto rs = region(L.k_pages, page);
        const int at = (kb & 1) * 64 * hd;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int ds = 0; ds < DS; ++ds)
                kf[kt][ds].u = __builtin_amdgcn_raw_buffer_load_b128(
                    rs, FULL || ds * 32 + lg * 8 < hd ? key_lane + ds * 2048 + kt * 256 : (int)RL_NOWHERE, at, RL_AT_AGENT);
    };
    auto ask_values = [&](int page, int kb) {
        const auto rs = region(L.v_pages, page);
        const int at = (kb & 1) * 1024;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            vf[dt].u = __builtin_amdgcn_raw_buffer_load_b128(rs, FULL || dt * 16 < hd ? value_lane + dt * 2048 : (int)RL_NOWHERE, at, RL_AT_AGENT);
    };
    int kb = kb_begin + wave - 1;
    int page = kb < kb_end ? pages[kb >> 1] : 0, page_behind = kb + 3 < kb_end ? pages[(kb + 3) >> 1] : 0;
    const bool early = kb < kb_end && kb * 32 + 32 <= a.start_pos[seq];
    if (early) {
        ask_keys(page, kb);
        ask_values(page, kb);
    }
    ready();
    RlFrag qf[DS];
    {
        const bf16_t* q = (const bf16_t*)(work + a.off_q) + ((size_t)it.token * a.H + g * R + (valid ? li : 0)) * hd;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const int d = ds * 32 + lg * 8;
            qf[ds].u = (valid && (FULL || d < hd)) ? rl_get16(q + d) : rl_u4{0, 0, 0, 0};
        }
    }
    if (kb < kb_end && !early) {
        ask_keys(page, kb);
        ask_values(page, kb);
    }
    float m = -INFINITY, l = 0.f;
    floatx4_t o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    for (; kb < kb_end; kb += 3) {
        const bool more = kb + 3 < kb_end;
        floatx4_t s[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            s[kt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ds = 0; ds < DS; ++ds)
                s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kt][ds].v, qf[ds].v, s[kt], 0, 0, 0);
        }
        if (more) {                                        // the next block's keys come in while this one's scores are worked on
            page = page_behind;
            page_behind = kb + 6 < kb_end ? pages[(kb + 6) >> 1] : 0;
            ask_keys(page, kb + 3);
        }
        const int key0 = kb * 32 + lg * 8;                 // this lane's keys: key0 .. key0 + 7
        if (kb * 32 + 31 > pos) {                          // slots beyond the newest key hold no data yet
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (key0 + e > pos) vf[dt].e[e] = 0;
        }
        float sv[8], mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int key = key0 + e;
            sv[e] = (valid && key <= pos && key >= lo) ? s[e >> 2][e & 3] : -INFINITY;
            mx = fmaxf(mx, sv[e]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, GFA_WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, GFA_WAVE)) * a.scale_log2;
        const float m_new = fmaxf(m, mx);
        const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;   // no key so far: -inf - -inf must not be formed
        const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
        RlFrag pf;
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float p = __builtin_amdgcn_exp2f(fmaf(sv[e], a.scale_log2, -m_safe));
            sum += p;
            pf.e[e] = float_to_bf16(p);
        }
        l = l * alpha + sum;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt].v, pf.v, o[dt], 0, 0, 0);
        if (more) ask_values(page, kb + 3);
    }
    l += __shfl_xor(l, 16, GFA_WAVE);
    l += __shfl_xor(l, 32, GFA_WAVE);
    float* sm_ml = (float*)smem;                           // [4][16][2]
    floatx4_t* sm_o = (floatx4_t*)(smem + 4 * 16 * 2 * sizeof(float));   // [4][DT][64]
    if (lg == 0) {
        sm_ml[(wave * 16 + li) * 2] = m;
        sm_ml[(wave * 16 + li) * 2 + 1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) sm_o[(wave * DT + dt) * 64 + lane] = o[dt];
}

// Then all four waves, a quarter of the dims each: the three parts added in the waves' order, and where some token's context
// has shares (`shared`) their sums by the workgroup that comes last.  Meets the streamers RL_ITEM_MEETINGS times less the
// two before it.  Returns whether the pair's result is complete, and then it has landed.
#define RL_ITEM_MEETINGS(shared) ((shared) ? 5 : 3)
template <int DS, bool FULL, typename Args>
__device__ __forceinline__ bool rl_join_heads(const Args& a, char* work, const RlItem& it, int layer, const char* smem, int wave,
                                              bool shared, int* flag) {
    constexpr int DT = DS * 2, DQ = DT / 4;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int li = lane & 15, lg = lane >> 4, d0 = wave * DQ * 16;
    const int hd = FULL ? DS * 32 : a.hd, R = a.H / a.Hkv;
    const float* sm_ml = (const float*)smem;
    const floatx4_t* sm_o = (const floatx4_t*)(smem + 4 * 16 * 2 * sizeof(float));
    float m = -INFINITY, l = 0.f;
    floatx4_t o[DQ];
#pragma unroll
    for (int q = 0; q < DQ; ++q) o[q] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto merge = [&](float mw, float lw, const floatx4_t (&other)[DQ]) {
        if (mw == -INFINITY && lw == 0.f) return;          // saw no key; scores that are no numbers leave lw NaN, and that stays
        const float m_new = fmaxf(m, mw);
        const float keep = __builtin_amdgcn_exp2f(m - m_new), add = __builtin_amdgcn_exp2f(mw - m_new);
        l = l * keep + lw * add;
        m = m_new;
#pragma unroll
        for (int q = 0; q < DQ; ++q) o[q] = o[q] * keep + other[q] * add;
    };
#pragma unroll
    for (int w = 1; w < 4; ++w) {
        floatx4_t other[DQ];
#pragma unroll
        for (int q = 0; q < DQ; ++q) other[q] = sm_o[(w * DT + wave * DQ + q) * 64 + lane];
        merge(sm_ml[(w * 16 + li) * 2], sm_ml[(w * 16 + li) * 2 + 1], other);
    }
    bool complete = true;
    if (shared) {
        // [item][R][hd] and [item][R][2], this lane's dims of its head
        const int row = li < R ? li : 0;
        float* po = (float*)(a.work + a.off_po);
        float* pml = (float*)(a.work + a.off_pml);
        if (it.splits > 1 && li < R) {
#pragma unroll
            for (int q = 0; q < DQ; ++q)
                if (FULL || d0 + q * 16 < hd) {
                    float* at = po + ((size_t)it.index * R + row) * hd + d0 + q * 16 + lg * 4;
                    rl_put8(at, __float_as_uint(o[q][0]), __float_as_uint(o[q][1]));
                    rl_put8(at + 2, __float_as_uint(o[q][2]), __float_as_uint(o[q][3]));
                }
            if (wave == 0 && lg == 0) rl_put8(pml + (it.index * R + row) * 2, __float_as_uint(m), __float_as_uint(l));
        }
        rl_all_landed();
        lds_barrier();
        if (wave == 0 && lane == 0)                        // the words count all layers
            *flag = it.splits == 1 ||
                    __hip_atomic_fetch_add(a.words + RL_AT_SPLITS + it.pair, 1, __ATOMIC_RELAXED, AGENT) == (layer + 1) * it.splits - 1;
        lds_barrier();
        complete = rl_same(*flag) != 0;
        if (complete && it.splits > 1) {
            m = -INFINITY;
            l = 0.f;
#pragma unroll
            for (int q = 0; q < DQ; ++q) o[q] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
            for (int sp = 0; sp < it.splits; ++sp) {
                const int item = it.index + (sp - it.split) * a.Hkv;
                const float2 ml = rl_get8(pml + (item * R + row) * 2);
                floatx4_t other[DQ];
#pragma unroll
                for (int q = 0; q < DQ; ++q) {
                    const float* at = po + ((size_t)item * R + row) * hd + (FULL || d0 + q * 16 < hd ? d0 + q * 16 : 0) + lg * 4;
                    const float2 u = rl_get8(at), w = rl_get8(at + 2);
                    other[q] = floatx4_t{u.x, u.y, w.x, w.y};
                }
                merge(ml.x, ml.y, other);
            }
        }
    }
    if (complete && li < R) {
        const float inv = 1.f / l;
        bf16_t* y = (bf16_t*)(work + a.off_in[2]);
#pragma unroll
        for (int q = 0; q < DQ; ++q)
            if (FULL || d0 + q * 16 < hd)
                rl_put8(y + chunked_elem(it.token, (it.g * R + li) * hd + d0 + q * 16 + lg * 4, a.pad), rl_two(o[q][0] * inv, o[q][1] * inv),
                        rl_two(o[q][2] * inv, o[q][3] * inv));
    }
    rl_all_landed();
    lds_barrier();                                         // and the shared memory is free again
    return complete;
}

// What is waited for: cumulative counts of the counters, lane c holding those of counters c and 64 + c.
struct RlWait {
    int* counters;
    int need, lane;
    bool lost;
    int need1 = 0;                        // of the second counter
    __device__ __forceinline__ void expect(int arrivals) {
        need += (unsigned)(arrivals + RL_COUNTERS - 1 - lane) / RL_COUNTERS;
        need1 += (unsigned)(arrivals + RL_COUNTERS - 1 - 64 - lane) / RL_COUNTERS;
    }
    __device__ __forceinline__ void all() {
        if (lost) return;
        int polls = 0;
        for (;;) {
            const int seen = rl_get(counters + lane * RL_LINE), seen1 = rl_get(counters + (64 + lane) * RL_LINE);
            if (__all(seen >= need && seen1 >= need1)) break;
            if (++polls == RL_MAX_POLLS) {
                lost = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        asm volatile("" ::: "memory");
    }
    // what this wave stored has landed: one more of this phase's arrivals
    __device__ __forceinline__ void arrive(int index) {
        rl_all_landed();
        if (lane == 0) __hip_atomic_fetch_add(counters + (index % RL_COUNTERS) * RL_LINE, 1, __ATOMIC_RELAXED, AGENT);
    }
};

// The place of a workgroup: worker v of V, from a layer on; v < 0: nothing to do.
struct RlPlace {
    int v, V, layer;
};

// Into the list of the first layer from `layer` on that is not closed yet, and waits until it is.  By one lane.
__device__ __forceinline__ RlPlace rl_enlist(int* lists, int layer, int n_layers) {
    for (; layer < n_layers; ++layer) {
        int* list = lists + layer * RL_LIST;
        int seen = rl_get(list);
        while (!(seen & RL_CLOSED))
            if (__hip_atomic_compare_exchange_strong(list, &seen, seen + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED, AGENT)) {
                const int v = seen & RL_COUNT;
                while (!((seen = rl_get(list)) & RL_CLOSED)) __builtin_amdgcn_s_sleep(2);
                return {v, seen & RL_COUNT, layer};
            }
    }
    return {-1, 0, 0};
}

// Who works at the start.  By one lane.  Those that are here wait for the others about as long as a layer would take them, a tenth
// of start_polls for all of the grid (8B: 76 us, 100 polls): a long wait is lost if nobody comes, a layer by few workers if they
// come soon.
__device__ __forceinline__ RlPlace rl_join(int* words, int n_layers, int start_polls, int seal_polls) {
    const int b = blockIdx.x, n = gridDim.x, group = b % RL_GROUPS;
    const int groups = n < RL_GROUPS ? n : RL_GROUPS, of_group = (n - group + RL_GROUPS - 1) / RL_GROUPS;
    int* lists = words + RL_AT_LISTS;
    int state = 0;
    if (__hip_atomic_fetch_add(words + RL_AT_GROUPS + group * RL_LINE, 1, __ATOMIC_RELAXED, AGENT) == of_group - 1) {
        state = rl_get(words);                             // the last of its group: the group is there
        while (!(state & RL_CLOSED) &&
               !__hip_atomic_compare_exchange_strong(words, &state, state + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED, AGENT)) {}
    }
    int polls = 0;
    for (;;) {
        state = rl_get(words);
        if (state == groups) return {b, n, 0};             // all are there
        if (state & RL_CLOSED) return rl_enlist(lists, 0, n_layers);
        if (++polls >= start_polls) {
            int here = 0;
            for (int i = 0; i < groups; ++i) here += rl_get(words + RL_AT_GROUPS + i * RL_LINE);
            if (10 * here * polls >= start_polls * n &&
                __hip_atomic_compare_exchange_strong(words, &state, state | RL_CLOSED, __ATOMIC_RELAXED, __ATOMIC_RELAXED, AGENT))
                break;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    // some are not: those that come here before the first layer's list is closed share the work
    const int v = __hip_atomic_fetch_add(lists, 1, __ATOMIC_RELAXED, AGENT);
    for (int i = 0; i < seal_polls; ++i) __builtin_amdgcn_s_sleep(2);
    return {v, __hip_atomic_fetch_or(lists, RL_CLOSED, __ATOMIC_RELAXED, AGENT), 0};
}

// Who works on the next layer: the V that worked on the one before, the last of which closes the list, and those that came
// before that.  By one lane.
__device__ __forceinline__ int2 rl_join_again(int* list, int V) {
    int seen = __hip_atomic_fetch_add(list, RL_BEFORE + 1, __ATOMIC_RELAXED, AGENT);
    const int v = seen & RL_COUNT;
    if (seen / RL_BEFORE + 1 == V) return make_int2(v, __hip_atomic_fetch_or(list, RL_CLOSED, __ATOMIC_RELAXED, AGENT) & RL_COUNT);
    while (!((seen = rl_get(list)) & RL_CLOSED)) __builtin_amdgcn_s_sleep(2);
    return make_int2(v, seen & RL_COUNT);
}

__device__ __forceinline__ float rl_gate(int mode, float a) {
    if (mode == 6) return 0.5f * a * (1.f + tanhf(0.7978845608028654f * (a + 0.044715f * a * a * a)));
    return a / (1.f + expf(-a));
}

// Lane i of every sixteen gets the value of lane (i + n) % 16.
#define RL_TURNED(x, n) __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), 0x120 + 16 - (n), 0xf, 0xf, false))

// A worker's way through the layers.  WHOLE: all workgroups are there, and every part of a phase has one worker from the first
// layer to the last.  In a body of its own: in one body for both forms more is alive than there are registers for, and a step of the 8B
// shape takes 2,880 us instead of 2,667 at 1 row, 3,108 instead of 2,892 at 8.
template <int DS, bool FULL, bool WHOLE, typename Args>
__device__ __forceinline__ void rl_work(const Args& a, char* smem, int v, int V, int first_layer) {
    char* x_lds = smem;
    char* stages = smem + RL_X_BYTES;
    floatx4_t* sums = (floatx4_t*)(stages + RL_STREAMERS * RL_STAGE);
    int* place = (int*)(sums + 2 * RL_SUMS);
    const int* first = place + 16;
    const RlPlan* plan = (RlPlan*)(first + 32);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), parts = gridDim.x;
    if (WHOLE) first_layer = 0;
    // where some are missing all waves meet twice between layers: the new list is there; all have read it
    auto new_list = [&] {
        lds_barrier();
        v = rl_same(place[0]);
        V = rl_same(place[1]);
        lds_barrier();
    };
    const int pad = a.pad, pairs = a.M * a.Hkv;
    const int items = rl_same(first[a.M]) * a.Hkv;
    const bool shared = items > pairs;
    if (wave < RL_STREAMERS) {
        rl_u4 ring[RL_RING][4];
        RlCursor c;
        char* stage = stages + wave * RL_STAGE;
        int layer = first_layer, phase = 0, part = v;
        RlProduct p = rl_product(a, plan, layer, 0, v);
        rl_seek(c, p, wave);
#pragma unroll
        for (int i = 0; i < RL_RING; ++i) rl_ask(c, ring[i], lane);
#pragma unroll 1
        while (layer < a.n_layers) {
            bool part_left = false;
            if (!WHOLE) {
                part_left = part + V < parts;
                part = part_left ? part + V : v;
            }
            const int next_phase = part_left ? phase : phase == 0 ? 2 : phase == 4 ? 0 : phase + 1;
            const int next_layer = layer + (phase == 4 && !part_left);
            const bool other_list = !WHOLE && next_layer != layer && V < parts;   // the next part is not known yet
            RlProduct next = rl_product(a, plan, other_list ? a.n_layers : next_layer, next_phase, part);
            rl_stream(p, next, c, ring, wave, lane, pad, x_lds, stage, sums);
            if (phase == 0 && !part_left)                  // attention: the other waves'
                for (int item = v; item < items; item += V)
                    for (int i = 0; i < RL_ITEM_MEETINGS(shared); ++i) lds_barrier();
            if (other_list && next_layer < a.n_layers) {
                new_list();
                part = v;
                next = rl_product(a, plan, next_layer, 0, v);
                rl_seek(c, next, wave);
#pragma unroll
                for (int i = 0; i < RL_RING; ++i) rl_ask(c, ring[i], lane);
            }
            p = next;
            phase = next_phase;
            layer = next_layer;
        }
        return;
    }

    if (wave > RL_STREAMERS) {                             // bring x, and work on attention
        const int aux = wave - RL_STREAMERS;
        __builtin_amdgcn_s_setprio(2);
#pragma unroll 1
        for (int at = 5 * first_layer; at < 5 * a.n_layers; ++at) {
            const int layer = at / 5, phase = at - 5 * layer;
            char* work = a.work + (size_t)layer * a.work_stride;
            if (phase == 1) {
                for (int item = v; item < items; item += V) {
                    const RlItem it(a, first, item);
                    rl_attend<DS, FULL>(a, a.layer[layer], work, it, x_lds, aux, [] { lds_barrier(); });
                    lds_barrier();
                    rl_join_heads<DS, FULL>(a, work, it, layer, x_lds, aux, shared, place + 3);
                }
                continue;
            }
            int part = v;
            do {
                const RlProduct p = rl_product(a, plan, layer, phase, part);
                if (p.rows == 0) break;
                const char* x = work + (unsigned)rl_same(plan[phase].off_in);
                lds_barrier();
                int chunk_begin = 0;
                for (int n = 0, of = ((p.rows + 15) >> 4) * p.chunks; n <= of; ++n) {
                    if (n == 0 || (p.chunks > 1 && n < of))
                        rl_bring(p, x, pad, chunk_begin, x_lds + (n & 1) * RL_X_HALF, aux - 1, lane);
                    chunk_begin += p.chunk;
                    if (chunk_begin >= p.pieces) chunk_begin = 0;
                    lds_barrier();
                }
            } while (!WHOLE && (part += V) < parts);
            if (!WHOLE && phase == 4 && V < parts && layer + 1 < a.n_layers) new_list();
        }
        return;
    }

    // the one that waits for the phase before and finishes products and attention
    const int fi = lane & 15, fg = lane >> 4;
    const int with_d = rl_same(plan[2].arrivals);
    RlWait wait = {a.words + RL_AT_COUNTERS, 0, lane, false};

    // four columns n.. of the stream: their normed half; returns the sum of their squares
    auto leave_normed = [&](int n, const float4& r, const float4& g, char* x) {
        rl_put8((bf16_t*)x + chunked_elem(fi, n, pad), rl_two(r.x * g.x, r.y * g.y), rl_two(r.z * g.z, r.w * g.w));
        return fmaf(r.x, r.x, fmaf(r.y, r.y, fmaf(r.z, r.z, r.w * r.w)));
    };
    // a part's share of the rows' sums of squares
    auto leave_share = [&](float sum, char* s, int part) {
        sum += __shfl_xor(sum, 16, GFA_WAVE);
        sum += __shfl_xor(sum, 32, GFA_WAVE);
        if (fg == 0 && fi < pad) rl_put((float*)s + (size_t)part * pad + fi, sum);
    };
    // four columns of the stream: one worker's from the first layer to the last, or another one's in every layer
    auto stream_at = [&](int n) {
        const float* at = a.residual + (size_t)fi * a.D + n;
        if (WHOLE) return *(const float4*)at;
        const float2 lo = rl_get8(at), hi = rl_get8(at + 2);
        return make_float4(lo.x, lo.y, hi.x, hi.y);
    };
    // What finishing the first tile of a product needs beside the sums stays here: the stream's columns, and of the rotation
    // what is the same in every layer.
    float4 stream0 = make_float4(0.f, 0.f, 0.f, 0.f);
    float cs0[2] = {1.f, 1.f}, sn0[2] = {0.f, 0.f};
    int pos = 0;
    auto angles = [&](int n, float (&cs)[2], float (&sn)[2]) {
        const int head = n / a.hd, d = n - head * a.hd;
        cs[0] = cs[1] = 1.f;
        sn[0] = sn[1] = 0.f;
        if (head < a.H + a.Hkv)
#pragma unroll
            for (int pr = 0; pr < 2; ++pr)
                if (d + 2 * pr < a.rot) sincosf((float)pos * a.freqs[(d + 2 * pr) >> 1], &sn[pr], &cs[pr]);
    };
    {
        __builtin_amdgcn_s_setprio(3);                     // others wait for what this wave does
        for (int part = v; part < with_d && first_layer == 0; part += WHOLE ? with_d : V) {   // the norm before the first layer
            const RlProduct d = rl_product(a, plan, 0, 2, part);
            float sum = 0.f;
            for (int n = d.base + fg * 4; n < d.base + d.rows; n += 16)
                if (fi < a.M) {
                    const float4 r = *(const float4*)(a.residual + (size_t)fi * a.D + n);
                    sum += leave_normed(n, r, *(const float4*)(a.norm_first + n), a.work + a.off_in[0]);
                    if (n < d.base + 16) stream0 = r;
                }
            leave_share(sum, a.work + a.off_sums[0], part);
            wait.arrive(part);
        }
        wait.expect(with_d);
        for (int n = 0; n < first_layer; ++n) {            // what others have done
            wait.expect(rl_same(plan[0].arrivals));
            wait.expect(pairs);
            for (int phase = 2; phase < 5; ++phase) wait.expect(rl_same(plan[phase].arrivals));
        }
        if (fi < a.M) pos = a.tok_pos[fi];
        const int n = v * rl_same(plan[0].share) + fg * 4;
        if (fi < a.M && n < a.N[0]) angles(n, cs0, sn0);
    }

    for (int layer = first_layer; layer < a.n_layers; ++layer) {
        const auto& L = a.layer[layer];
        char* work = a.work + (size_t)layer * a.work_stride;
#pragma unroll 1
        for (int phase = 0; phase < 5; ++phase) {
            if (phase == 1) {
                for (int item = v; item < items; item += V) {
                    const RlItem it(a, first, item);
                    if (item == v) wait.all();
                    lds_barrier();
                    lds_barrier();
                    if (rl_join_heads<DS, FULL>(a, work, it, layer, x_lds, 0, shared, place + 3)) wait.arrive(it.pair);
                }
                wait.expect(pairs);
                continue;
            }
            int part = v;
            do {
                const RlProduct p = rl_product(a, plan, layer, phase, part);
                if (p.rows == 0) break;
                const int tiles = (p.rows + 15) >> 4;
                {
                    const float* norm = L.norm[phase];
                    float4 res = stream0, g = make_float4(0.f, 0.f, 0.f, 0.f);
                    float cs[2] = {cs0[0], cs0[1]}, sn[2] = {sn0[0], sn0[1]};
                    int page = 0, n = 0;
                    bool mine = false;
                    // the rest of it, of the first tile before this phase may begin, of the others while they are worked out
                    auto ask_operands = [&](int j) {
                        n = p.base + j * 16 + fg * 4;
                        mine = fi < a.M && j * 16 + fg * 4 < p.rows;
                        if (mine) {
                            if (phase == 0) {
                                if (n >= a.H * a.hd) page = L.table[(size_t)a.tok_seq[fi] * a.table_stride + pos / GFA_PAGE];
                                if (j > 0 || !WHOLE) angles(n, cs, sn);
                            } else if (phase != 3) {
                                if (j > 0) res = stream_at(n);
                                if (norm) g = *(const float4*)(norm + n);
                            }
                        }
                    };
                    ask_operands(0);
                    wait.all();
                    if (!WHOLE && mine && (phase == 2 || phase == 4)) res = stream_at(n);
                    lds_barrier();
                    // the norm's other half: all workers' shares, sixteen bytes a lane, all of them under way at once;
                    // lane l's numbers are of rows 4 l + e: of every fourth row, or of two or all rows in turn
                    const bool normed = phase == 0 || phase == 3;
                    float e[4] = {0.f, 0.f, 0.f, 0.f};
                    if (normed) {
                        const char* s = work + (unsigned)rl_same(plan[phase].off_sums);
                        const int all = with_d * pad * 4;
                        const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)s, 0, all, 0x27000);
#pragma unroll 1
                        for (int at = 0; at < all; at += 8192) {
                            rl_u4 shares[8];
#pragma unroll
                            for (int i = 0; i < 8; ++i) shares[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at + (i * 64 + lane) * 16, 0, RL_AT_AGENT);
#pragma unroll
                            for (int i = 0; i < 8; ++i)
#pragma unroll
                                for (int j = 0; j < 4; ++j) e[j] += __uint_as_float(shares[i][j]);
                        }
                    }
                    lds_barrier();
                    float rs = 1.f;
                    if (normed) {
                        if (pad == 1) e[0] = e[1] = e[2] = e[3] = (e[0] + e[1]) + (e[2] + e[3]);
                        if (pad == 2) { e[0] = e[2] = e[0] + e[2]; e[1] = e[3] = e[1] + e[3]; }
                        // over the lanes whose numbers are of the same rows: turns within sixteen lanes, then their groups
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            e[j] += RL_TURNED(e[j], 8);
                            e[j] += RL_TURNED(e[j], 4);
                            if (pad <= 8) e[j] += RL_TURNED(e[j], 2);
                            if (pad <= 4) e[j] += RL_TURNED(e[j], 1);
                        }
                        // row fi: number fi % 4 of lane (fi % pad) / 4
                        const int from = (lane & 48) | ((fi & (pad - 1)) >> 2);
                        float own[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) own[j] = __shfl(e[j], from, GFA_WAVE);
                        float ssq = (fi & 2) ? ((fi & 1) ? own[3] : own[2]) : ((fi & 1) ? own[1] : own[0]);
                        ssq += __shfl_xor(ssq, 16, GFA_WAVE);
                        ssq += __shfl_xor(ssq, 32, GFA_WAVE);
                        rs = rsqrtf(ssq / (float)a.D + a.eps[phase]);
                    }
                    if (wait.lost) rs = __builtin_nanf("");
                    const unsigned out = rl_same(plan[phase].off_out);
                    float squares = 0.f;
                    for (int j = 0; j < tiles; ++j) {
                        const bool last = j + 1 == tiles;
                        for (int c = 0; c < p.chunks; ++c) lds_barrier();
                        const floatx4_t* sum = sums + (j & 1) * RL_SUMS + lane;
                        floatx4_t v0 = sum[0], v1 = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int s = 1; s < RL_STREAMERS; ++s) v0 += sum[s * 128];
                        v0 *= rs;
                        if (phase == 3) {
                            v1 = sum[64];
#pragma unroll
                            for (int s = 1; s < RL_STREAMERS; ++s) v1 += sum[s * 128 + 64];
                            v1 *= rs;
                        }
                        if (mine) {
                            if (phase == 0) {              // two rotary pairs of one head
                                const int head = n / a.hd, d = n - head * a.hd;
                                float o[4] = {v0[0], v0[1], v0[2], v0[3]};
                                if (head < a.H + a.Hkv) {
#pragma unroll
                                    for (int pr = 0; pr < 2; ++pr)
                                        if (d + 2 * pr < a.rot) {
                                            const float p0 = o[2 * pr], p1 = o[2 * pr + 1];
                                            o[2 * pr] = p0 * cs[pr] - p1 * sn[pr];
                                            o[2 * pr + 1] = p1 * cs[pr] + p0 * sn[pr];
                                        }
                                }
                                const unsigned lo = rl_two(o[0], o[1]), hi = rl_two(o[2], o[3]);
                                const int off = pos % GFA_PAGE;
                                if (head < a.H) {
                                    rl_put8((bf16_t*)(work + a.off_q) + ((size_t)fi * a.H + head) * a.hd + d, lo, hi);
                                } else if (head < a.H + a.Hkv) {
                                    rl_put8(L.k_pages + key_elem(page, head - a.H, off, d, a.Hkv, a.hd), lo, hi);
                                } else {
#pragma unroll
                                    for (int e = 0; e < 4; ++e)
                                        rl_put(L.v_pages + value_elem(page, head - a.H - a.Hkv, d + e, off, a.Hkv, a.hd), float_to_bf16(o[e]));
                                }
                            } else if (phase == 3) {
                                float h[4];
#pragma unroll
                                for (int e = 0; e < 4; ++e) h[e] = rl_gate(a.gate_mode, v0[e]) * v1[e];
                                rl_put8((bf16_t*)(work + a.off_in[4]) + chunked_elem(fi, n, pad), rl_two(h[0], h[1]), rl_two(h[2], h[3]));
                            } else {
                                res.x += v0[0]; res.y += v0[1]; res.z += v0[2]; res.w += v0[3];
                                if (norm) squares += leave_normed(n, res, g, work + out);
                            }
                        }
                        float* out_stream = a.residual + (size_t)fi * a.D + n;
                        if (!WHOLE && mine && (phase == 2 || phase == 4)) {
                            rl_put8(out_stream, __float_as_uint(res.x), __float_as_uint(res.y));
                            rl_put8(out_stream + 2, __float_as_uint(res.z), __float_as_uint(res.w));
                        }
                        if (last) {
                            if (norm) leave_share(squares, work + (unsigned)rl_same(plan[phase].off_share), part);
                            wait.arrive(part);
                        }
                        // the stream itself is this wave's alone, and of the first tile it stays in registers
                        if (WHOLE && (phase == 2 || phase == 4)) {
                            if (j == 0) stream0 = res;
                            if (mine && (j > 0 || layer + 1 == a.n_layers)) *(float4*)out_stream = res;
                        }
                        if (!last) ask_operands(j + 1);
                    }
                }
            } while (!WHOLE && (part += V) < parts);
            wait.expect(rl_same(plan[phase].arrivals));
        }
        if (!WHOLE && V < parts && layer + 1 < a.n_layers) {
            if (lane == 0) {
                const int2 w = rl_join_again(a.words + RL_AT_LISTS + (layer + 1) * RL_LIST, V);
                place[0] = w.x;
                place[1] = w.y;
            }
            new_list();
        }
    }
}

template <int DS, bool FULL>
__global__ __launch_bounds__(RL_THREADS) void resident_layers_kernel(const ResidentArgs) {
    RlArgs& a = *(RlArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    extern __shared__ __attribute__((aligned(128))) char smem[];
    int* place = (int*)(smem + RL_X_BYTES + RL_STREAMERS * RL_STAGE + 2 * RL_SUMS * 16);
    int* first = place + 16;
    RlPlan* plan = (RlPlan*)(first + 32);
    if (threadIdx.x == 0) {
        const RlPlace w = rl_join(a.words, a.n_layers, a.start_polls, a.seal_polls);
        place[0] = w.v;
        place[1] = w.V;
        place[2] = w.layer;
    }
    lds_barrier();
    const int v = rl_same(place[0]), V = rl_same(place[1]), first_layer = rl_same(place[2]);
    if (v < 0) return;
    if (threadIdx.x < 5) rl_make_plan(a, plan, threadIdx.x, gridDim.x);
    if (rl_same(threadIdx.x >> 6) == 1) rl_make_shares(a, first, threadIdx.x & 63);
    lds_barrier();
    if (V == (int)gridDim.x && first_layer == 0) rl_work<DS, FULL, true>(a, smem, v, V, 0);
    else rl_work<DS, FULL, false>(a, smem, v, V, first_layer);
}

__global__ __launch_bounds__(256) void resident_zero_kernel(int* words, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) words[i] = 0;
}

static int rl_rows_kept(int M) { return M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : M <= 8 ? 8 : 16; }

static int rl_units() {
    int dev = 0, units = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    return units;
}

// The buffers of a launch: sizes and places.  Returns the bytes of all of them: 32 layers of the 8B shape 3 MB at 1 row, 19 at 8 (36 and
// 52 with partial sums in every layer).
static size_t rl_lay_out(ResidentArgs& a, int units) {
    const size_t pad = a.pad, D = a.D, heads = (size_t)a.H * a.hd;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t at = off; off = (off + bytes + 255) / 256 * 256; return at; };
    a.off_in[0] = take(pad * D * 2);
    a.off_sums[0] = take((D + 3) / 4 * pad * 4);
    a.off_q = take((size_t)a.M * heads * 2);
    a.off_in[2] = take(pad * heads * 2);
    a.off_in[3] = take(pad * D * 2);
    a.off_sums[3] = take((D + 3) / 4 * pad * 4);
    a.off_in[4] = take(pad * (size_t)a.I * 2);
    a.work_stride = off;
    a.off_out[2] = a.off_in[3];
    a.off_share[2] = a.off_sums[3];
    a.off_out[4] = (unsigned)off + a.off_in[0];
    a.off_share[4] = (unsigned)off + a.off_sums[0];
    off *= a.n_layers;
    const long pairs = (long)a.M * a.Hkv, of_token = (a.table_stride * 2 + RL_SHARE - 1) / RL_SHARE;
    const long most = 2l * (units > pairs ? units : pairs);
    const size_t partials = of_token > 1 ? (most < pairs * of_token ? most : pairs * of_token) * (a.H / a.Hkv) : 0;
    a.off_po = take(partials * a.hd * 4);
    a.off_pml = take(partials * 2 * 4);
    return off;
}

static size_t rl_word_bytes(int M, int Hkv) { return ((size_t)(RL_AT_SPLITS + M * Hkv) * 4 + 255) / 256 * 256; }

template <int DS, bool FULL>
static int rl_launch(const ResidentArgs& a, int grid, int shared, hipStream_t stream) {
    const int rc = (int)hipFuncSetAttribute((const void*)resident_layers_kernel<DS, FULL>, hipFuncAttributeMaxDynamicSharedMemorySize, shared);
    if (rc) return rc;
    resident_layers_kernel<DS, FULL><<<grid, RL_THREADS, shared, stream>>>(a);
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_resident_layers_max() { return RL_MAX_LAYERS; }

// Bytes of work memory that gfa_resident_layers_bf16 needs for these layers.
extern "C" long gfa_resident_work_bytes(int n_layers, int M, int D, int I, int H, int Hkv, int hd, int table_stride) {
    ResidentArgs a = {};
    a.n_layers = n_layers; a.M = M; a.D = D; a.I = I; a.H = H; a.Hkv = Hkv; a.hd = hd; a.table_stride = table_stride;
    a.pad = rl_rows_kept(M);
    return (long)(rl_word_bytes(M, Hkv) + rl_lay_out(a, rl_units()));
}

// layers' residual [M, D] in place, as gfa_few_row_layers_bf16 (gemm_bf16.hip) but from the stream on: the first norm
// is part of it.  `workgroups`, `start_polls`: 0 for what the device has and the usual patience.
extern "C" int gfa_resident_layers_bf16(const FewRowLayer* layers, int n_layers, const FewRowStep* step, int workgroups, int start_polls,
                                        hipStream_t stream) {
    const FewRowStep& s = *step;
    const int units = rl_units();
    if (n_layers <= 0 || n_layers > RL_MAX_LAYERS || s.M <= 0 || s.M > RL_MAX_ROWS || s.D <= 0 || s.D % 8 || s.I <= 0 || s.I % 8 ||
        s.H <= 0 || s.Hkv <= 0 || s.H % s.Hkv || s.H / s.Hkv > 16 || s.hd <= 0 || s.hd % 16 || s.hd > 128 || s.rot < 0 || s.rot % 2 ||
        s.rot > s.hd || s.table_stride <= 0 || (s.gate_mode != 3 && s.gate_mode != 6) || units <= 0 ||
        s.D >= RL_MOST_COLUMNS || s.I >= RL_MOST_COLUMNS || (long)s.H * s.hd >= RL_MOST_COLUMNS || (long)s.D * s.I * 4 >= RL_MOST_BYTES || (long)s.D * (s.H + 2 * s.Hkv) * s.hd * 2 >= RL_MOST_BYTES)
        return (int)hipErrorInvalidValue;
    ResidentArgs a = {};
    for (int i = 0; i < n_layers; ++i) {
        const FewRowLayer& L = layers[i];
        a.layer[i] = {{(const bf16_t*)L.wqkv, nullptr, (const bf16_t*)L.wo, (const bf16_t*)L.w13, (const bf16_t*)L.w2},
                      {nullptr, nullptr, L.norm_ffn, nullptr, i + 1 < n_layers ? layers[i + 1].norm_mixer : nullptr},
                      (bf16_t*)L.k_pages, (bf16_t*)L.v_pages, L.table};
    }
    const int heads = s.H * s.hd;
    const int N[5] = {(s.H + 2 * s.Hkv) * s.hd, 0, s.D, s.I, s.D}, K[5] = {s.D, 0, heads, s.D, s.I};
    for (int i = 0; i < 5; ++i) {
        a.N[i] = N[i];
        a.K[i] = K[i];
    }
    a.gate[3] = s.I;
    a.eps[0] = s.eps_mixer;
    a.eps[3] = s.eps_ffn;
    a.norm_first = layers[0].norm_mixer;
    a.residual = s.residual;
    a.freqs = s.freqs;
    a.tok_seq = s.tok_seq;
    a.tok_pos = s.tok_pos;
    a.start_pos = s.start_pos;
    a.n_layers = n_layers; a.M = s.M; a.D = s.D; a.I = s.I; a.H = s.H; a.Hkv = s.Hkv; a.hd = s.hd; a.rot = s.rot;
    a.table_stride = s.table_stride;
    a.window = s.window;
    a.pad = rl_rows_kept(s.M);
    a.gate_mode = s.gate_mode;
    a.scale_log2 = s.scale * 1.4426950408889634f;
    a.start_polls = start_polls > 0 && start_polls < 1000 ? start_polls : 1000;
    a.seal_polls = a.start_polls < 100 ? 2 * a.start_polls : 200;
    a.words = (int*)s.work;
    a.work = (char*)s.work + rl_word_bytes(s.M, s.Hkv);
    rl_lay_out(a, units);
    const int grid = workgroups > 0 && workgroups < units ? workgroups : units;
    const int words = RL_AT_SPLITS + s.M * s.Hkv;
    resident_zero_kernel<<<(words + 255) / 256, 256, 0, stream>>>(a.words, words);
    const int shared = RL_X_BYTES + RL_STREAMERS * RL_STAGE + 2 * RL_SUMS * 16 + (16 + 32) * 4 + 5 * (int)sizeof(RlPlan);
    return s.hd == 64   ? rl_launch<2, true>(a, grid, shared, stream)
           : s.hd == 128 ? rl_launch<4, true>(a, grid, shared, stream)
           : s.hd < 64   ? rl_launch<2, false>(a, grid, shared, stream)
                         : rl_launch<4, false>(a, grid, shared, stream);
}
