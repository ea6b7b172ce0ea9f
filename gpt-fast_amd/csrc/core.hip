// Plain kernels for every op of a decoder step.
//
// These are the reference kernels of the library: simple, one workgroup per row or per
// (token, head), all arithmetic in float.  The float32 engine runs on them alone; the
// bfloat16 engine uses them where no faster kernel exists, and the faster kernels are
// tested against them.  In each kernel the order of floating-point additions that
// produce one output element depends only on that element's own inputs (its row, its
// position), never on the number of rows or on the other sequences of the launch, so a
// float32 result is the same however the tokens were cut into steps or batched.
#include "few_row_layers.h"
#include <type_traits>

// --------------------------------------------------------------------------------------
// embedding gather: out[n, :] = float(table[tokens[n], :])          (model.py:140)
template <typename T>
__global__ void embed_kernel(const T* __restrict__ table, const int* __restrict__ tokens,
                             float* __restrict__ out, int dim) {
    const int n = blockIdx.x;
    const T* row = table + (size_t)tokens[n] * dim;
    float* o = out + (size_t)n * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) o[d] = load_as_float(row + d);
}

extern "C" int gfa_embed(const void* table, int table_bf16, const int* tokens, float* out,
                         int n_tokens, int dim, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (table_bf16)
        embed_kernel<bf16_t><<<n_tokens, 256, 0, stream>>>((const bf16_t*)table, tokens, out, dim);
    else
        embed_kernel<float><<<n_tokens, 256, 0, stream>>>((const float*)table, tokens, out, dim);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// RMS norm: out[i, :] = x[r, :] * rsqrt(mean(x[r, :]^2) + eps) * w[:],  r = rows ? rows[i] : i
// (model.py:236-241; statistics in float, one rounding at the store)
template <typename T>
__global__ void rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                               const int* __restrict__ rows, T* __restrict__ out, int dim,
                               float eps) {
    __shared__ float scratch[16];
    const int i = blockIdx.x;
    const int r = rows ? rows[i] : i;
    const float* xr = x + (size_t)r * dim;
    float ss = 0.f;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) {
        const float v = xr[d];
        ss = fmaf(v, v, ss);
    }
    ss = block_sum(ss, scratch);
    const float rs = rsqrtf(ss / (float)dim + eps);
    T* o = out + (size_t)i * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) store_from_float(o + d, xr[d] * rs * w[d]);
}

// The same for rows of up to 1024 * VPT elements (a multiple of 4): the row is read once
// with 16-byte loads, kept in registers between the sum and the scaling.
template <typename T, int VPT, int THREADS>
__global__ __launch_bounds__(THREADS) void rmsnorm_vec_kernel(
        const float* __restrict__ x, const float* __restrict__ w, const int* __restrict__ rows,
        T* __restrict__ out, int dim, float eps) {
    __shared__ float scratch[16];
    const int i = blockIdx.x;
    const int r = rows ? rows[i] : i;
    const float4* xr = (const float4*)(x + (size_t)r * dim);
    const float4* w4 = (const float4*)w;
    const int n4 = dim >> 2;
    float4 v[VPT];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        v[j] = idx < n4 ? xr[idx] : make_float4(0.f, 0.f, 0.f, 0.f);
        ss = fmaf(v[j].x, v[j].x, ss);
        ss = fmaf(v[j].y, v[j].y, ss);
        ss = fmaf(v[j].z, v[j].z, ss);
        ss = fmaf(v[j].w, v[j].w, ss);
    }
    ss = block_sum(ss, scratch);
    const float rs = rsqrtf(ss / (float)dim + eps);
    T* o = out + (size_t)i * dim;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            const float4 g = w4[idx];
            store_from_float(o + 4 * idx + 0, v[j].x * rs * g.x);
            store_from_float(o + 4 * idx + 1, v[j].y * rs * g.y);
            store_from_float(o + 4 * idx + 2, v[j].z * rs * g.z);
            store_from_float(o + 4 * idx + 3, v[j].w * rs * g.w);
        }
    }
}

template <typename T>
static bool launch_rmsnorm_vec(const float* x, const float* w, const int* rows, T* out, int n_rows,
                               int dim, float eps, hipStream_t stream) {
    if (dim % 4 != 0 || dim > 8192) return false;
    // one float4 per thread where the row allows it: the kernel is a chain of latencies
    if (dim <= 1024) rmsnorm_vec_kernel<T, 1, 256><<<n_rows, 256, 0, stream>>>(x, w, rows, out, dim, eps);
    else if (dim <= 4096) rmsnorm_vec_kernel<T, 1, 1024><<<n_rows, 1024, 0, stream>>>(x, w, rows, out, dim, eps);
    else rmsnorm_vec_kernel<T, 2, 1024><<<n_rows, 1024, 0, stream>>>(x, w, rows, out, dim, eps);
    return true;
}

extern "C" int gfa_rmsnorm(const float* x, const float* w, const int* rows, void* out,
                           int out_bf16, int n_rows, int dim, float eps, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (out_bf16 ? launch_rmsnorm_vec<bf16_t>(x, w, rows, (bf16_t*)out, n_rows, dim, eps, stream)
                 : launch_rmsnorm_vec<float>(x, w, rows, (float*)out, n_rows, dim, eps, stream))
        return GFA_LAUNCH_RESULT();
    if (out_bf16)
        rmsnorm_kernel<bf16_t><<<n_rows, 256, 0, stream>>>(x, w, rows, (bf16_t*)out, dim, eps);
    else
        rmsnorm_kernel<float><<<n_rows, 256, 0, stream>>>(x, w, rows, (float*)out, dim, eps);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// The sum that completes a block and the norm that opens the next, one pass over each row:
// res[i, :] += float(y[i, :]);  out[i, :] = rmsnorm(res[i, :]) in bfloat16
// (model.py:162-163 followed by 236-241; the sum and the statistics in float)
__global__ void add_rmsnorm_kernel(float* __restrict__ res, const bf16_t* __restrict__ y,
                                   const float* __restrict__ w, bf16_t* __restrict__ out, int dim,
                                   float eps) {
    __shared__ float scratch[16];
    const int i = blockIdx.x;
    float* xr = res + (size_t)i * dim;
    const bf16_t* yr = y + (size_t)i * dim;
    float ss = 0.f;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) {
        const float v = xr[d] + bf16_to_float(yr[d]);
        xr[d] = v;                                       // read back by this thread only
        ss = fmaf(v, v, ss);
    }
    ss = block_sum(ss, scratch);
    const float rs = rsqrtf(ss / (float)dim + eps);
    bf16_t* o = out + (size_t)i * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) store_from_float(o + d, xr[d] * rs * w[d]);
}

// rows of up to 1024 * VPT elements (a multiple of 4), kept in registers
template <int VPT, int THREADS>
__global__ __launch_bounds__(THREADS) void add_rmsnorm_vec_kernel(
        float* __restrict__ res, const bf16_t* __restrict__ y, const float* __restrict__ w,
        bf16_t* __restrict__ out, int dim, float eps) {
    __shared__ float scratch[16];
    const int i = blockIdx.x;
    float4* xr = (float4*)(res + (size_t)i * dim);
    const uint2* yr = (const uint2*)(y + (size_t)i * dim);
    const float4* w4 = (const float4*)w;
    const int n4 = dim >> 2;
    float4 v[VPT];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (idx < n4) {
            v[j] = xr[idx];
            const uint2 a = yr[idx];
            v[j].x += __uint_as_float(a.x << 16);
            v[j].y += __uint_as_float(a.x & 0xffff0000u);
            v[j].z += __uint_as_float(a.y << 16);
            v[j].w += __uint_as_float(a.y & 0xffff0000u);
            xr[idx] = v[j];
        }
        ss = fmaf(v[j].x, v[j].x, ss);
        ss = fmaf(v[j].y, v[j].y, ss);
        ss = fmaf(v[j].z, v[j].z, ss);
        ss = fmaf(v[j].w, v[j].w, ss);
    }
    ss = block_sum(ss, scratch);
    const float rs = rsqrtf(ss / (float)dim + eps);
    uint2* o = (uint2*)(out + (size_t)i * dim);
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            const float4 g = w4[idx];
            bf16_t e[4];
            e[0] = float_to_bf16(v[j].x * rs * g.x);
            e[1] = float_to_bf16(v[j].y * rs * g.y);
            e[2] = float_to_bf16(v[j].z * rs * g.z);
            e[3] = float_to_bf16(v[j].w * rs * g.w);
            o[idx] = make_uint2((unsigned)e[0] | ((unsigned)e[1] << 16),
                                (unsigned)e[2] | ((unsigned)e[3] << 16));
        }
    }
}

extern "C" int gfa_add_rmsnorm(float* res, const void* y, const float* w, void* out, int n_rows,
                               int dim, float eps, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    const bf16_t* yp = (const bf16_t*)y;
    bf16_t* op = (bf16_t*)out;
    const bool vec = dim % 4 == 0 && dim <= 8192 && (uintptr_t)res % 16 == 0 &&
                     (uintptr_t)y % 8 == 0 && (uintptr_t)out % 8 == 0 && (uintptr_t)w % 16 == 0;
    if (!vec) add_rmsnorm_kernel<<<n_rows, 256, 0, stream>>>(res, yp, w, op, dim, eps);
    else if (dim <= 1024) add_rmsnorm_vec_kernel<1, 256><<<n_rows, 256, 0, stream>>>(res, yp, w, op, dim, eps);
    else if (dim <= 4096) add_rmsnorm_vec_kernel<1, 1024><<<n_rows, 1024, 0, stream>>>(res, yp, w, op, dim, eps);
    else add_rmsnorm_vec_kernel<2, 1024><<<n_rows, 1024, 0, stream>>>(res, yp, w, op, dim, eps);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// float32 matrix products: out[b][m, n] (+)= sum_k a[b][m, k] * w[b][n, k], element (m, k) of a[b] at
// a + b sab + m sam + k, element (n, k) of w[b] at w + b swb + n swn + k swk, element (m, n) of out[b] at
// out + b sob + m som + n.
//
// v_mfma_f32_16x16x4_f32: true float32 products and sums, at the vector units' peak rate but without
// their operand traffic.  The four waves of a workgroup take the same 16 MT x 16 NT tile and every
// fourth block of 32 k each, so that even a 16-column tile of one row keeps four waves' loads in flight.
// An output's sum is therefore four chains, added as (0 + 1) + (2 + 3), whose
// order depends on K alone (the k within a block are taken in an order that is the same for a and w): every kernel here,
// every tile size and every M gives the same bits, and a row's result does not
// depend on the other rows (a float32 logit is the same however tokens are cut into steps).
// gf_product picks the kernel and the tile.  Few rows are bound by latency and the weights (1 x 32,000 x 768 20 us, 5 TB/s),
// many by the matrix units (2,048 x 4,096 x 4,096 494 us, 139 of the 155 TFLOP/s that a loop of the instruction alone reaches).
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gf_floatx4_t;

// out's tile at (m0, n0) from the waves' sums, ((0 + 1) + (2 + 3)); lane: four columns of a row
template <int MT, int NT>
__device__ __forceinline__ void gf_store(const gf_floatx4_t (*sums)[MT * NT][64], float* __restrict__ out, int M,
                                         int N, int m0, int n0, long long som, int accumulate) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool quad = som % 4 == 0 && (uintptr_t)out % 16 == 0;
    for (int t = wave; t < MT * NT; t += 4) {
        const gf_floatx4_t v = (sums[0][t][lane] + sums[1][t][lane]) + (sums[2][t][lane] + sums[3][t][lane]);
        const int m = m0 + 16 * (t / NT) + (lane & 15), n = n0 + 16 * (t % NT) + 4 * (lane >> 4);
        if (m >= M || n >= N) continue;
        float* o = out + (size_t)m * som + n;
        if (quad && n + 4 <= N) {
            gf_floatx4_t* o4 = (gf_floatx4_t*)o;
            *o4 = accumulate ? *o4 + v : v;
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (n + q < N) o[q] = accumulate ? o[q] + v[q] : v[q];
        }
    }
}

// Operands of any strides, element by element: a lane's loads are four k of one row of a or w and land in operand order, so nothing
// goes through shared memory but the four sums at the end.
template <int MT, int NT>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(
        const float* __restrict__ a, const float* __restrict__ w, float* __restrict__ out,
        int M, int N, int K, long long sab, long long sam, long long swb, long long swn,
        long long swk, long long sob, long long som, int accumulate) {
    constexpr int AHEAD = MT * NT == 1 ? 4 : MT * NT <= 4 ? 2 : 1;   // blocks asked for ahead
    __shared__ gf_floatx4_t sums[4][MT * NT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int m0 = blockIdx.y * (16 * MT), n0 = blockIdx.x * (16 * NT);
    a += (size_t)blockIdx.z * sab;
    w += (size_t)blockIdx.z * swb;
    out += (size_t)blockIdx.z * sob;
    const float *ar[MT], *wr[NT];                  // rows beyond the last read it again, never stored
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = m0 + 16 * i + li;
        ar[i] = a + (size_t)(m < M ? m : M - 1) * sam;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n = n0 + 16 * j + li;
        wr[j] = w + (size_t)(n < N ? n : N - 1) * swn;
    }
    gf_floatx4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = gf_floatx4_t{0.f, 0.f, 0.f, 0.f};

    struct Block {
        gf_floatx4_t a[2][MT], w[2][NT];
    };
    // the lane's elements of block b (its k: 32 b + 16 h + 4 lg + 0..3); zero beyond K.  Every load is made,
    // at a place that is there: loads under a condition would not stay in flight
    auto load = [&](int b, Block& r) {
        const bool whole = 32 * b + 32 <= K;       // the same for the whole wave
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 32 * b + 16 * h + 4 * lg;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int at = k + q < K ? k + q : 0;
#pragma unroll
                for (int i = 0; i < MT; ++i) r.a[h][i][q] = ar[i][at];
#pragma unroll
                for (int j = 0; j < NT; ++j) r.w[h][j][q] = wr[j][(size_t)at * swk];
            }
            if (!whole) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (k + q >= K) {
#pragma unroll
                        for (int i = 0; i < MT; ++i) r.a[h][i][q] = 0.f;
#pragma unroll
                        for (int j = 0; j < NT; ++j) r.w[h][j][q] = 0.f;
                    }
            }
        }
    };
    auto multiply = [&](const Block& r) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)   // transposed: a lane ends with four columns of a row
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.w[h][j][q], r.a[h][i][q],
                                                                         acc[i][j], 0, 0, 0);
    };
    const int blocks = (K + 31) / 32;
    Block ring[AHEAD + 1];
    if (blocks > 0) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) load(wave + 4 * u, ring[u]);
    }
    for (int b = wave; b < blocks; b += 4 * (AHEAD + 1)) {
#pragma unroll
        for (int u = 0; u <= AHEAD; ++u) {
            if (b + 4 * u >= blocks) break;
            load(b + 4 * (u + AHEAD), ring[(u + AHEAD) % (AHEAD + 1)]);
            multiply(ring[u]);
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sums[wave][i * NT + j][lane] = acc[i][j];
    __syncthreads();
    gf_store<MT, NT>(sums, out, M, N, m0, n0, som, accumulate);
}

// How the staged kernel gets a row's 32 k of a block: in 16-byte loads at multiples of 16, in 16-byte loads at any
// float, or as elements `swk` apart, where the lanes take neighbouring rows (those of a matrix that lies transposed).
enum GfLoads { GF_WIDE, GF_ALONG, GF_ACROSS };
typedef gf_floatx4_t gf_loose4_t __attribute__((aligned(4)));

// The same arithmetic for many rows whose operands are not both 16-byte rows: a 64 x 64 tile whose waves copy their blocks
// through shared memory of their own (no barrier while K is walked).  A load instruction then takes whole lines, eight rows of 128 bytes (across:
// 64 rows of one k), where the operand order above takes sixteen rows of 64 bytes, which the compute unit's cache
// looks up piece by piece: 2,048 x 4,096 x 1,022 (rows at odd
// addresses) took 616 us without it against 168, 32 x 1,000 x 512 x 128 with the second operand
// transposed, as latent attention has it, 161 against 65.
#define GS_PITCH 144                              // bytes per staged row of 32 k: 128 + pad against conflicts
template <GfLoads AL, GfLoads WL>
__global__ __launch_bounds__(256, 2) void gemm_f32_staged_kernel(
        const float* __restrict__ a, const float* __restrict__ w, float* __restrict__ out,
        int M, int N, int K, long long sab, long long sam, long long swb, long long swn, long long swk,
        long long sob, long long som, int accumulate) {
    __shared__ __attribute__((aligned(16))) char lds[4 * 128 * GS_PITCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    a += (size_t)blockIdx.z * sab;
    w += (size_t)blockIdx.z * swb;
    out += (size_t)blockIdx.z * sob;
    const int row = lane >> 3, chunk = lane & 7;   // of eight rows, their 16-byte chunks
    const float *ar[8], *wr[WL == GF_ACROSS ? 1 : 8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int m = m0 + 8 * i + row, n = n0 + (WL == GF_ACROSS ? lane : 8 * i + row);
        ar[i] = a + (size_t)(m < M ? m : M - 1) * sam;
        if (WL != GF_ACROSS || i == 0) wr[i] = w + (size_t)(n < N ? n : N - 1) * swn;
    }
    gf_floatx4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = gf_floatx4_t{0.f, 0.f, 0.f, 0.f};
    gf_floatx4_t av[8], wv[8];
    auto load = [&](int b) {
        const bool whole = 32 * b + 32 <= K;       // the same for the whole wave
        const int k = 32 * b + 4 * chunk;
        // eight times four k, the row's first ones again beyond K
        auto eight = [&](auto row_of, auto k_of, GfLoads how, gf_floatx4_t (&v)[8]) {
            if (how == GF_ALONG && whole) {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = *(const gf_loose4_t*)(row_of(i) + k_of(i));
                return;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (how == GF_WIDE) {
                    v[i] = *(const gf_floatx4_t*)(row_of(i) + (k_of(i) < K ? k_of(i) : 0));
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int at = k_of(i) + q < K ? k_of(i) + q : 0;
                        v[i][q] = how == GF_ACROSS ? row_of(i)[(size_t)at * swk] : row_of(i)[at];
                    }
                }
            }
        };
        eight([&](int i) { return ar[i]; }, [&](int) { return k; }, AL, av);
        eight([&](int i) { return wr[WL == GF_ACROSS ? 0 : i]; }, [&](int i) { return WL == GF_ACROSS ? 32 * b + 4 * i : k; }, WL, wv);
        if (!whole) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (k + q >= K) av[i][q] = 0.f;
                    if ((WL == GF_ACROSS ? 32 * b + 4 * i : k) + q >= K) wv[i][q] = 0.f;
                }
        }
    };
    char* as = lds + wave * 128 * GS_PITCH;
    char* ws = as + 64 * GS_PITCH;
    const int put = row * GS_PITCH + chunk * 16, get = li * GS_PITCH + lg * 16;
    const int blocks = (K + 31) / 32;
    if (wave < blocks) load(wave);
    for (int b = wave; b < blocks; b += 4) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            *(gf_floatx4_t*)(as + put + 8 * i * GS_PITCH) = av[i];
            *(gf_floatx4_t*)(ws + (WL == GF_ACROSS ? lane * GS_PITCH + 16 * i : put + 8 * i * GS_PITCH)) = wv[i];
        }
        if (b + 4 < blocks) load(b + 4);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            gf_floatx4_t af[4], wf[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                af[i] = *(const gf_floatx4_t*)(as + get + 16 * i * GS_PITCH + 64 * h);
                wf[i] = *(const gf_floatx4_t*)(ws + get + 16 * i * GS_PITCH + 64 * h);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j][q], af[i][q], acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
    gf_floatx4_t (*sums)[16][64] = (gf_floatx4_t (*)[16][64])lds;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) sums[wave][i * 4 + j][lane] = acc[i][j];
    __syncthreads();
    gf_store<4, 4>(sums, out, M, N, m0, n0, som, accumulate);
}

// The same where all loads are 16 bytes at multiples of 16, the form of a model's products: each wave's blocks go through
// shared memory of its own, and every load, write and read of it is issued between two products.  A wave issues in order: in the
// staged kernel above the 16 loads, 16 writes and 16 reads of a block stand in a row, some 1,000 cycles in which the wave
// starts no product, and two waves of a SIMD fall into step (the matrix units were busy 56 to 63 % of the time).  Here, while
// a block's first half multiplies, its second half is read; while that multiplies, the next block is written, its first half
// read, and block + 1 + AHEAD asked for.
//
// The wave's whole blocks of `at` (16 MT rows) and `wt` (16 NT rows, the second half of them from `wt2`) into acc; from: the lane's bytes
// from there to its rows, eight a load.  ready() runs once the first AHEAD blocks are asked for.  NORMED: elements of `at` times
// their row's rs, then times g.
template <int MT, int NT, int AHEAD, bool NORMED, class Offset, class Ready>
__device__ __forceinline__ void gf_piped(const char* at, const char* wt, const char* wt2, const Offset (&from)[2 * (MT + NT)],
                                         const float* g, const float (&rs)[2 * MT], int K, char* own, gf_floatx4_t (&acc)[MT][NT], Ready ready) {
    constexpr int S = MT + NT, HALF = 4 * MT * NT;         // operands of a half block, its products
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane >> 3, chunk = lane & 7;           // of eight rows, their 16-byte chunks
    const int put = row * GS_PITCH + chunk * 16, get = (lane & 15) * GS_PITCH + (lane >> 4) * 16;
    gf_floatx4_t v[AHEAD][2 * S], gv[AHEAD], f[2][S];
    auto base = [&](int i) { return i < 2 * MT ? at : i < 2 * MT + NT ? wt : wt2; };
    auto ask = [&](int j, int slot) {                      // this wave's whole block j
        const size_t k = (size_t)(wave + 4 * j) * 128;
#pragma unroll
        for (int i = 0; i < 2 * S; ++i) v[slot][i] = *(const gf_floatx4_t*)(base(i) + k + from[i]);
        if (NORMED) gv[slot] = *(const gf_floatx4_t*)((const char*)g + k + 16 * chunk);
    };
    auto write = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 2 * S; ++i) {
            gf_floatx4_t x = v[slot][i];
            if (NORMED && i < 2 * MT)
#pragma unroll
                for (int q = 0; q < 4; ++q) x[q] = x[q] * rs[i < 2 * MT ? i : 0] * gv[slot][q];
            *(gf_floatx4_t*)(own + put + 8 * i * GS_PITCH) = x;
        }
    };
    auto read = [&](int h) {
#pragma unroll
        for (int i = 0; i < S; ++i) f[h][i] = *(const gf_floatx4_t*)(own + get + 16 * i * GS_PITCH + 64 * h);
    };
    auto multiply = [&](int h) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[h][MT + j][q], f[h][i][q], acc[i][j], 0, 0, 0);
    };
// `times` of the kind `what`, each in front of `each` products
#define GP_ORDER(what, times, each)                                                  \
    _Pragma("unroll") for (int u = 0; u < (times); ++u) {                            \
        __builtin_amdgcn_sched_group_barrier(what, 1, 0);                            \
        __builtin_amdgcn_sched_group_barrier(GP_PRODUCT, (each), 0);                 \
    }
#define GP_PRODUCT 0x008
#define GP_ASK 0x020
#define GP_READ 0x100
#define GP_WRITE 0x200
    const int whole = K / 32;
    const int count = wave < whole ? (whole - wave + 3) / 4 : 0;   // this wave's whole blocks
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
        if (u < count) ask(u, u);
    ready();
    if (count > 0) {
        write(0);
        read(0);
        if (AHEAD < count) ask(AHEAD, 0);
        // block j multiplies, j + 1 is written, j + 1 + AHEAD asked for
        auto step = [&](int j, int slot, auto more) {
            read(1);
            multiply(0);
            write(slot);
            read(0);
            if (decltype(more)::value) ask(j + 1 + AHEAD, slot);
            multiply(1);
            if (HALF > 4) {
                GP_ORDER(GP_READ, S, HALF / 2 / S)
                __builtin_amdgcn_sched_group_barrier(GP_PRODUCT, HALF - S * (HALF / 2 / S), 0);
                GP_ORDER(GP_WRITE, 2 * S, HALF / 4 / S)
                GP_ORDER(GP_READ, S, HALF / 4 / S)
                if (decltype(more)::value) GP_ORDER(GP_ASK, 2 * S, 1)
            }
        };
        int j = 0;
        for (; j + 2 * AHEAD < count; j += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) step(j + u, (u + 1) % AHEAD, std::true_type());
        }
#pragma unroll
        for (int u = 0; u < 2 * AHEAD; ++u) {              // the last 2 AHEAD blocks at most
            if (j + u + 1 >= count) break;
            if (u < AHEAD && j + u + 1 + AHEAD < count) step(j + u, (u + 1) % AHEAD, std::true_type());
            else step(j + u, (u + 1) % AHEAD, std::false_type());
        }
        read(1);
        multiply(0);
        multiply(1);
    }
#undef GP_ORDER
#undef GP_PRODUCT
#undef GP_ASK
#undef GP_READ
#undef GP_WRITE
    if (K % 32 && whole % 4 == wave) {                     // the rest behind the whole blocks, zero beyond K, a multiple of four
        const bool in = 32 * whole + 4 * chunk < K;
        const size_t k = (size_t)whole * 128;
        const int back = in ? 0 : 16 * chunk;
        if (NORMED) gv[0] = *(const gf_floatx4_t*)((const char*)g + k + 16 * chunk - back);
#pragma unroll
        for (int i = 0; i < 2 * S; ++i) {
            v[0][i] = *(const gf_floatx4_t*)(base(i) + k + from[i] - back);
            if (!in) v[0][i] = gf_floatx4_t{0.f, 0.f, 0.f, 0.f};
        }
        if (NORMED && !in) gv[0] = gf_floatx4_t{0.f, 0.f, 0.f, 0.f};
        write(0);
        read(0);
        read(1);
        multiply(0);
        multiply(1);
    }
}

// The product on it in tiles of 16 MT x 16 NT, us before (the two kernels above) and now: 2,048 x 4,096 x 4,096 704 -> 490
// (140 TFLOP/s), 717 x 4,096 x 768 71 -> 43, 717 x 768 x 2,048 41 -> 24, 60 x 768 x 2,048 19 -> 12, 4 x 32,000 x 768 32.5 -> 20,
// 4 x 768 x 2,048 10 -> 7.3, 16 x 28,672 x 4,096 142 -> 96.  A 1 x 1 tile with one block ahead takes 78 us for 4 x 4,096 x 14,336, with
// two 60, with four 45 (before: 55); 2 x 2 tiles with two ahead hold more registers and are slower (29.7, 31.5 at 717 x 768 x 2,048).
// Offset: of the bytes from a tile's first row to its others.
template <int MT, int NT, int AHEAD, class Offset = unsigned>
__global__ __launch_bounds__(256, 2) void gemm_f32_piped_kernel(
        const float* __restrict__ a, const float* __restrict__ w, float* __restrict__ out, int M, int N, int K,
        long long sab, long long sam, long long swb, long long swn, long long sob, long long som, int accumulate) {
    constexpr int S = MT + NT;
    __shared__ __attribute__((aligned(16))) char lds[4 * 16 * S * GS_PITCH];
    static_assert(4 * MT * NT * 1024 <= 4 * 16 * S * GS_PITCH, "the waves' sums take the blocks' place");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = blockIdx.y * (16 * MT), n0 = blockIdx.x * (16 * NT);
    Offset from[2 * S];                            // rows beyond the last read it again, never stored
#pragma unroll
    for (int i = 0; i < 2 * S; ++i) {
        const int r = 8 * (i < 2 * MT ? i : i - 2 * MT) + (lane >> 3), most = (i < 2 * MT ? M - m0 : N - n0) - 1;
        from[i] = (Offset)(r < most ? r : most) * (Offset)(4 * (i < 2 * MT ? sam : swn)) + 16 * (lane & 7);
    }
    gf_floatx4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = gf_floatx4_t{0.f, 0.f, 0.f, 0.f};
    const char* wt = (const char*)(w + (size_t)blockIdx.z * swb + (size_t)n0 * swn);
    const float none[2 * MT] = {};
    gf_piped<MT, NT, AHEAD, false>((const char*)(a + (size_t)blockIdx.z * sab + (size_t)m0 * sam), wt, wt, from, nullptr, none, K,
                                   lds + wave * 16 * S * GS_PITCH, acc, [] {});
    __syncthreads();
    gf_floatx4_t (*sums)[MT * NT][64] = (gf_floatx4_t (*)[MT * NT][64])lds;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sums[wave][i * NT + j][lane] = acc[i][j];
    __syncthreads();
    gf_store<MT, NT>(sums, out + (size_t)blockIdx.z * sob, M, N, m0, n0, som, accumulate);
}

// Side of a 16-byte product's tile by rows, columns and inner size, in sixteens.  Up to 16 rows 1 x 1, which spreads the weights over the
// most waves.  Else a tile's products take the matrix units of one of 256 compute units for as long as it has pieces of 16 x 16, and
// smaller tiles read more for each: tiles a unit, times pieces, times 1, 1.08, 1.09, 1.17 (2,048 x 4,096 x 4,096: 494, 549, 569,
// 600 us at 128, 132, 135, 128 pieces a unit; 717 rows of K = 768, us by 4 x 4, 3 x 4, 3 x 3, 2 x 2: N = 4,096 42, 44, 49, 45; 2,304 29.5, 33, 26.5,
// 27.4; 768 16.3, 13.7, 12.4, 13.6; 200 rows, N = 768, K = 2,048 35, 29, 23, 12).  Of 2 x 2 tiles
//  * four share a unit where of the others two do, which counts for more than what they read while a wave has a block or two: times 0.95 up to
//    K = 192 (2,498 x 14,713 x 16 by 4 x 4 and 2 x 2 130, 110; 705 x 2,220 x 116 12.3, 12.0; 60 times 218 x 1,319 x 16 68, 58);
//  * what is read again is no longer in the caches where operands are larger than these and rows long: times 1.40 (26 times 361 x 390 x 7,876
//    852, 1,389; 43 times 289 x 219 x 8,668 608, 1,197; but 2,131 x 565 x 1,380, 15 MB, 56, 41).
// Over 6,942 products of 17 to 2,500 rows, alone and up to 64 at a time, what it picks is 0.9 % off the fastest tile on average (without these two 3.4 %),
// and 0.5 % of them are more than 3 % slower than in the two kernels above with 16-byte loads, which this one replaced (1.9 %).
static int gf_piped_tile(int B, int M, int N, int K) {
    if (M <= 16) return 11;
    int best = 44;
    double least = INFINITY;
    const int small = K <= 192 ? 95 : K >= 1024 && ((double)M + N) * K * B * 4 > 32e6 ? 140 : 117;
    const int tiles[4][3] = {{4, 4, 100}, {3, 4, 108}, {3, 3, 109}, {2, 2, small}};
    for (const auto& t : tiles) {
        if ((M + 16 * t[0] - 1) / (16 * t[0]) > 65535) continue;     // rows of a grid
        const double n = (double)B * ((M + 16 * t[0] - 1) / (16 * t[0])) * ((N + 16 * t[1] - 1) / (16 * t[1]));
        const double cost = ceil(n / 256) * t[0] * t[1] * t[2];
        if (cost < least) least = cost, best = 10 * t[0] + t[1];
    }
    return best;
}

// Other forms.  Up to 16 rows: one 16 x 16 tile a workgroup.  More rows: 64 x 64 where these tiles are at least 100, else 32 x 32.
static int gf_product(const float* a, const float* w, float* out, int B, int M, int N, int K,
                      long long sab, long long sam, long long swb, long long swn, long long swk,
                      long long sob, long long som, int accumulate, hipStream_t stream) {
    if (B <= 0 || M <= 0 || N <= 0) return 0;
    // 16-byte loads: whole groups of four k, at addresses that are multiples of 16
    const bool a_wide = K % 4 == 0 && sam % 4 == 0 && sab % 4 == 0 && (uintptr_t)a % 16 == 0;
    const bool w_wide = swk == 1 && K % 4 == 0 && swn % 4 == 0 && swb % 4 == 0 && (uintptr_t)w % 16 == 0;
    if (a_wide && w_wide) {
        // Rows whose offsets within a tile of 64 have no 32 bits: the same with 64, by the tiles that they had in front of this kernel
        const bool far = sam < 0 || swn < 0 || sam >= 1 << 23 || swn >= 1 << 23;
        const long long tiles = (long long)((M + 63) / 64) * ((N + 63) / 64) * B;
        const int tile = !far ? gf_piped_tile(B, M, N, K) : M <= 16 ? 11 : tiles < 100 ? 22 : 44, mt = tile / 10 * 16, nt = tile % 10 * 16;
        if ((M + mt - 1) / mt > 65535 || B > 65535) return (int)hipErrorInvalidValue;
        const dim3 grid((N + nt - 1) / nt, (M + mt - 1) / mt, B);
#define GP_GO(...) gemm_f32_piped_kernel<__VA_ARGS__><<<grid, 256, 0, stream>>>(a, w, out, M, N, K, sab, sam, swb, swn, sob, som, accumulate)
        if (far && tile == 11) GP_GO(1, 1, 4, long long);
        else if (far && tile == 22) GP_GO(2, 2, 1, long long);
        else if (far) GP_GO(4, 4, 1, long long);
        else if (tile == 11) GP_GO(1, 1, 4);
        else if (tile == 22) GP_GO(2, 2, 1);
        else if (tile == 33) GP_GO(3, 3, 1);
        else if (tile == 34) GP_GO(3, 4, 1);
        else GP_GO(4, 4, 1);
#undef GP_GO
        return GFA_LAUNCH_RESULT();
    }
    const int tile = M <= 16 ? 16 : (long long)((M + 63) / 64) * ((N + 63) / 64) * B < 100 ? 32 : 64;
    if ((M + tile - 1) / tile > 65535 || B > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid((N + tile - 1) / tile, (M + tile - 1) / tile, B);
#define GF_GO(...) __VA_ARGS__<<<grid, 256, 0, stream>>>(a, w, out, M, N, K, sab, sam, swb, swn, swk, sob, som, accumulate)
    if (tile == 16) GF_GO(gemm_f32_kernel<1, 1>);
    else if (tile == 32) GF_GO(gemm_f32_kernel<2, 2>);
    else if (swk != 1 && a_wide) GF_GO(gemm_f32_staged_kernel<GF_WIDE, GF_ACROSS>);
    else if (swk != 1) GF_GO(gemm_f32_staged_kernel<GF_ALONG, GF_ACROSS>);
    else GF_GO(gemm_f32_staged_kernel<GF_ALONG, GF_ALONG>);
#undef GF_GO
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_gemm_f32(const float* a, const float* w, float* out, int M, int N, int K,
                            int lda, int ldo, int accumulate, hipStream_t stream) {
    return gf_product(a, w, out, 1, M, N, K, 0, lda, 0, K, 1, 0, ldo, accumulate, stream);
}

extern "C" int gfa_gemm_f32_strided(const float* a, const float* w, float* out, int B, int M, int N,
                                    int K, long long sab, long long sam, long long swb,
                                    long long swn, long long swk, long long sob, long long som,
                                    hipStream_t stream) {
    return gf_product(a, w, out, B, M, N, K, sab, sam, swb, swn, swk, sob, som, 0, stream);
}

// --------------------------------------------------------------------------------------
// Rotary position encoding of q and k, and the write of k and v into the paged cache.
// qkv: [N, (H + 2*Hkv) * hd] rows of q heads, k heads, v heads (model.py:195-199).
// Pair i of a head is (2i, 2i+1) if layout == 0 (model.py:281-293) or (i, i + rot/2) if
// layout == 1; it is rotated by angle = float(position) * freqs[i], cos and sin in float.
// Elements beyond `rot` pass through.  q goes to q_out [N, H, hd]; k and v of token n go
// to page table[seq(n)][pos / PAGE], offset pos % PAGE (model.py:91-100, 206-207); keys as
// rows [offset, hd], values transposed [hd, offset] (see common.h).
template <typename T>
__global__ __launch_bounds__(256) void rope_cache_kernel(
        const T* __restrict__ qkv, T* __restrict__ q_out, T* __restrict__ k_pages,
        T* __restrict__ v_pages, const float* __restrict__ freqs, const int* __restrict__ tok_seq,
        const int* __restrict__ tok_pos, const int* __restrict__ table, int table_stride, int H,
        int Hkv, int hd, int rot, int layout) {
    // one thread per pair of elements: q and k heads first (rotated or passed through), then
    // the pairs of v; blockIdx.y walks the token's pairs in groups of 256
    const int n = blockIdx.x;
    const int half = hd / 2;
    const int rot_pairs = rot / 2;
    const int qk_slots = (H + Hkv) * half, v_slots = Hkv * half;
    const int pos = tok_pos[n];
    // cos and sin of this token's angles, once per workgroup
    extern __shared__ float cs[];                          // [rot_pairs][2]
    if (blockIdx.y * 256 < qk_slots) {
        for (int i = threadIdx.x; i < rot_pairs; i += 256)
            sincosf((float)pos * freqs[i], &cs[2 * i + 1], &cs[2 * i]);
        __syncthreads();
    }
    const int e = blockIdx.y * 256 + threadIdx.x;
    if (e >= qk_slots + v_slots) return;
    const T* row = qkv + (size_t)n * (H + 2 * Hkv) * hd;
    int page = 0;
    if (k_pages) page = table[(size_t)tok_seq[n] * table_stride + pos / GFA_PAGE];
    const int off = pos % GFA_PAGE;
    if (e < qk_slots) {
        const int head = e / half, i = e - head * half;
        const T* src = row + (size_t)head * hd;
        if (head >= H && !k_pages) return;
        // where element d of this head goes: a row of q_out, or the key's place in its page
        T* const dst = head < H ? q_out + ((size_t)n * H + head) * hd
                                : k_pages + cache_region(page, head - H, Hkv, hd);
        auto place = [&](int d) { return head < H ? d : key_offset(off, d, hd); };
        if (i < rot_pairs) {
            const int ia = layout == 0 ? 2 * i : i;
            const int ib = layout == 0 ? 2 * i + 1 : i + rot_pairs;
            const float a = load_as_float(src + ia), b = load_as_float(src + ib);
            const float c = cs[2 * i], s = cs[2 * i + 1];
            store_from_float(dst + place(ia), a * c - b * s);
            store_from_float(dst + place(ib), b * c + a * s);
        } else {
            const int d0 = rot + 2 * (i - rot_pairs);      // elements rot .. hd-1 are copied
            dst[place(d0)] = src[d0];
            dst[place(d0 + 1)] = src[d0 + 1];
        }
    } else if (v_pages) {
        const int ev = e - qk_slots;
        const int g = ev / half, d = 2 * (ev - g * half);
        const T* vsrc = row + (size_t)(H + Hkv + g) * hd + d;
        v_pages[value_elem(page, g, d, off, Hkv, hd)] = vsrc[0];
        v_pages[value_elem(page, g, d + 1, off, Hkv, hd)] = vsrc[1];
    }
}

// (a, b) <- (a c - b s, b c + a s) of pair p of eight elements.  Which of the two products is rounded before it is
// added is written out, because compilers choose it by what surrounds the expression: a key has to have the same
// bits whether its prompt comes whole (rope_cache_rows_kernel) or in portions of few tokens.
template <bool SLICED>
__device__ __forceinline__ void rope_turn(float& a, float& b, float c, float s, int p) {
    const float x = SLICED || p % 2 == 0 ? fmaf(a, c, -(b * s)) : fmaf(-b, s, a * c);
    b = SLICED ? fmaf(b, c, a * s) : fmaf(a, s, b * c);
    a = x;
}

// The rotation and cache write for bfloat16 with interleaved pairs, eight elements (four pairs) per thread:
// 16-byte loads and stores for q and k.  Needs hd and rot to be multiples of 8.
__global__ __launch_bounds__(256) void rope_cache_bf16x8_kernel(
        const bf16_t* __restrict__ qkv, bf16_t* __restrict__ q_out, bf16_t* __restrict__ k_pages,
        bf16_t* __restrict__ v_pages, const float* __restrict__ freqs,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
        const int* __restrict__ table, int table_stride, int H, int Hkv, int hd, int rot) {
    const int n = blockIdx.x;
    const int per_head = hd / 8;
    const int qk_chunks = (H + Hkv) * per_head, v_chunks = Hkv * per_head;
    const int pos = tok_pos[n];
    extern __shared__ float cs[];                          // [rot / 2][2]
    if (blockIdx.y * 256 < qk_chunks) {
        for (int i = threadIdx.x; i < rot / 2; i += 256)
            sincosf((float)pos * freqs[i], &cs[2 * i + 1], &cs[2 * i]);
        __syncthreads();
    }
    const int c = blockIdx.y * 256 + threadIdx.x;
    if (c >= qk_chunks + v_chunks) return;
    const int head = c / per_head, d0 = (c - head * per_head) * 8;
    union { uint4 u; bf16_t e[8]; } in, out;
    in.u = *(const uint4*)(qkv + ((size_t)n * (H + 2 * Hkv) + head) * hd + d0);
    int page = 0;
    if (k_pages && head >= H) page = table[(size_t)tok_seq[n] * table_stride + pos / GFA_PAGE];
    const int off = pos % GFA_PAGE;
    if (head < H + Hkv) {
        if (d0 < rot) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                float a = bf16_to_float(in.e[2 * p]), b = bf16_to_float(in.e[2 * p + 1]);
                rope_turn<false>(a, b, cs[d0 + 2 * p], cs[d0 + 2 * p + 1], p);
                out.e[2 * p] = float_to_bf16(a);
                out.e[2 * p + 1] = float_to_bf16(b);
            }
        } else {
            out.u = in.u;
        }
        if (head < H) {
            *(uint4*)(q_out + ((size_t)n * H + head) * hd + d0) = out.u;
        } else if (k_pages) {
            *(uint4*)(k_pages + key_elem(page, head - H, off, d0, Hkv, hd)) = out.u;   // one chunk of 8 dims
        }
    } else if (v_pages) {
        const int g = head - H - Hkv;
#pragma unroll
        for (int j = 0; j < 8; ++j) v_pages[value_elem(page, g, d0 + j, off, Hkv, hd)] = in.e[j];
    }
}

// The same with the rows given as float partial sums of a sliced product, part [S, N, width]:
// the slices are added in order (the sum a kernel of its own would form), rotated and stored,
// so that the product's second kernel is this one.  The rotation then works on the float sums
// instead of their bfloat16 rounding.
__global__ __launch_bounds__(256) void rope_cache_sliced_bf16x8_kernel(
        const float* __restrict__ part, int S, size_t slice, bf16_t* __restrict__ q_out,
        bf16_t* __restrict__ k_pages, bf16_t* __restrict__ v_pages, const float* __restrict__ freqs,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
        const int* __restrict__ table, int table_stride, int H, int Hkv, int hd, int rot) {
    const int n = blockIdx.x;
    const int per_head = hd / 8;
    const int qk_chunks = (H + Hkv) * per_head, v_chunks = Hkv * per_head;
    const int pos = tok_pos[n];
    extern __shared__ float cs[];                          // [rot / 2][2]
    if (blockIdx.y * 256 < qk_chunks) {
        for (int i = threadIdx.x; i < rot / 2; i += 256)
            sincosf((float)pos * freqs[i], &cs[2 * i + 1], &cs[2 * i]);
        __syncthreads();
    }
    const int c = blockIdx.y * 256 + threadIdx.x;
    if (c >= qk_chunks + v_chunks) return;
    const int head = c / per_head, d0 = (c - head * per_head) * 8;
    const float* src = part + ((size_t)n * (H + 2 * Hkv) + head) * hd + d0;
    float v[8];
    {
        const float4 a = *(const float4*)src, b = *(const float4*)(src + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
    for (int s = 1; s < S; ++s) {
        const float4 a = *(const float4*)(src + s * slice), b = *(const float4*)(src + s * slice + 4);
        v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w; v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
    }
    int page = 0;
    if (k_pages && head >= H) page = table[(size_t)tok_seq[n] * table_stride + pos / GFA_PAGE];
    const int off = pos % GFA_PAGE;
    union { uint4 u; bf16_t e[8]; } out;
    if (head < H + Hkv) {
        if (d0 < rot) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                rope_turn<true>(v[2 * p], v[2 * p + 1], cs[d0 + 2 * p], cs[d0 + 2 * p + 1], p);
                out.e[2 * p] = float_to_bf16(v[2 * p]);
                out.e[2 * p + 1] = float_to_bf16(v[2 * p + 1]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) out.e[j] = float_to_bf16(v[j]);
        }
        if (head < H) {
            *(uint4*)(q_out + ((size_t)n * H + head) * hd + d0) = out.u;
        } else if (k_pages) {
            *(uint4*)(k_pages + key_elem(page, head - H, off, d0, Hkv, hd)) = out.u;
        }
    } else if (v_pages) {
        const int g = head - H - Hkv;
#pragma unroll
        for (int j = 0; j < 8; ++j) v_pages[value_elem(page, g, d0 + j, off, Hkv, hd)] = float_to_bf16(v[j]);
    }
}

// Both for prompts.  The first `qk_blocks` rows of the grid rotate and store q and k, RC_TOKENS tokens per
// workgroup, so that all its threads work out angles.  The others write values: in a page these lie as groups
// of eight keys per dim, so where the eight tokens of a group are all there one thread takes eight dims of
// them and stores 16 bytes per dim; other tokens' values leave element by element.  As 2-byte stores, a token
// at a time, the values took more than half of the kernel: neighbouring tokens' workgroups run on different
// XCDs, which then all write the same lines.  Heads as in the 8B shape, before and now: 401 tokens 7.3 -> 6.3 us,
// 2,048 21.5 -> 15.9 (50 MB), 7,491 65 -> 42, six prompts of 2,696 tokens together 26.2 -> 18.5; two slices of
// 640 12.4 -> 11.1, of 2,048 30.4 -> 27.3.
// eight elements of a row at `at`: the slices added in order (SLICED), or the bfloat16 values as floats
template <bool SLICED>
__device__ __forceinline__ void rope_eight(const void* __restrict__ qkv, int S, size_t slice, size_t at, float (&v)[8]) {
    if (SLICED) {
        const float* src = (const float*)qkv + at;
        const float4 a = *(const float4*)src, b = *(const float4*)(src + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        for (int s = 1; s < S; ++s) {
            const float4 c = *(const float4*)(src + s * slice), d = *(const float4*)(src + s * slice + 4);
            v[0] += c.x; v[1] += c.y; v[2] += c.z; v[3] += c.w; v[4] += d.x; v[5] += d.y; v[6] += d.z; v[7] += d.w;
        }
    } else {
        const uint4 u = *(const uint4*)((const bf16_t*)qkv + at);
        const uint32_t* w = (const uint32_t*)&u;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            v[2 * p] = __uint_as_float(w[p] << 16);
            v[2 * p + 1] = __uint_as_float(w[p] & 0xffff0000u);
        }
    }
}
__device__ __forceinline__ uint4 rope_pack(const float (&v)[8]) {
    uint32_t o[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) o[p] = (uint32_t)float_to_bf16(v[2 * p]) | ((uint32_t)float_to_bf16(v[2 * p + 1]) << 16);
    return make_uint4(o[0], o[1], o[2], o[3]);
}
// the same eight as bfloat16; what was bfloat16 before is copied bit by bit
template <bool SLICED>
__device__ __forceinline__ uint4 rope_copy(const void* __restrict__ qkv, int S, size_t slice, size_t at) {
    if (!SLICED) return *(const uint4*)((const bf16_t*)qkv + at);
    float v[8];
    rope_eight<SLICED>(qkv, S, slice, at, v);
    return rope_pack(v);
}

#define RC_TOKENS 4
#define RC_VALUE_TOKENS 2
template <bool SLICED>
__global__ __launch_bounds__(256) void rope_cache_rows_kernel(
        const void* __restrict__ qkv, int S, size_t slice, bf16_t* __restrict__ q_out,
        bf16_t* __restrict__ k_pages, bf16_t* __restrict__ v_pages, const float* __restrict__ freqs,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
        const int* __restrict__ table, int table_stride, int n_tokens, int H, int Hkv, int hd, int rot, int qk_blocks) {
    const int per_head = hd / 8;
    const size_t width = (size_t)(H + 2 * Hkv) * hd;
    if ((int)blockIdx.y >= qk_blocks) {
        const int v_chunks = Hkv * per_head;
        const int teams = v_chunks < 256 ? 256 / v_chunks : 1;   // groups of threads that take tokens of their own
        const int team = threadIdx.x / (v_chunks < 256 ? v_chunks : 256);
        if (team >= teams) return;
        const int block = (blockIdx.x * (gridDim.y - qk_blocks) + blockIdx.y - qk_blocks) * RC_VALUE_TOKENS;
        for (int n = block + team; n < block + RC_VALUE_TOKENS && n < n_tokens; n += teams) {
            const int pos = tok_pos[n], seq = tok_seq[n];
            // a group of eight keys that is there whole is its first token's
            const int first = n - pos % 8;
            bool whole = first >= 0 && first + 7 < n_tokens && hd % 16 == 0 && (uintptr_t)v_pages % 16 == 0;
            for (int t = 0; whole && t < 8; ++t)
                whole = tok_seq[first + t] == seq && tok_pos[first + t] == pos - pos % 8 + t;
            if (whole && n != first) continue;
            const int page = table[(size_t)seq * table_stride + pos / GFA_PAGE], off = pos % GFA_PAGE;
            for (int c = threadIdx.x - team * v_chunks; c < v_chunks; c += 256) {
                const int g = c / per_head, d0 = (c - g * per_head) * 8;
                const size_t at = (size_t)n * width + (size_t)(H + Hkv + g) * hd + d0;
                if (whole) {
                    uint4 row[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t) row[t] = rope_copy<SLICED>(qkv, S, slice, at + t * width);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        uint32_t o[4];
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const uint32_t lo = ((const uint32_t*)&row[2 * t])[j / 2], hi = ((const uint32_t*)&row[2 * t + 1])[j / 2];
                            o[t] = j % 2 ? (lo >> 16) | (hi & 0xffff0000u) : (lo & 0xffffu) | (hi << 16);
                        }
                        *(uint4*)(v_pages + value_elem(page, g, d0 + j, off, Hkv, hd)) = make_uint4(o[0], o[1], o[2], o[3]);
                    }
                } else {
                    const uint4 row = rope_copy<SLICED>(qkv, S, slice, at);
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        v_pages[value_elem(page, g, d0 + j, off, Hkv, hd)] = (bf16_t)(((const uint32_t*)&row)[j / 2] >> (j % 2 * 16));
                }
            }
        }
        return;
    }
    const int n0 = blockIdx.x * RC_TOKENS;
    const int qk_chunks = (H + Hkv) * per_head;
    const int c = blockIdx.y * 256 + threadIdx.x;
    extern __shared__ float cs[];                          // [RC_TOKENS][rot / 2][2]
    for (int i = threadIdx.x; i < RC_TOKENS * (rot / 2); i += 256) {
        const int t = i / (rot / 2);
        const int n = n0 + t < n_tokens ? n0 + t : n_tokens - 1;
        sincosf((float)tok_pos[n] * freqs[i - t * (rot / 2)], &cs[2 * i + 1], &cs[2 * i]);
    }
    __syncthreads();
    if (c >= qk_chunks) return;
    const int head = c / per_head, d0 = (c - head * per_head) * 8;
    uint4 row[RC_TOKENS];
    float v[RC_TOKENS][8];
#pragma unroll
    for (int t = 0; t < RC_TOKENS; ++t) {
        const size_t at = (size_t)(n0 + t < n_tokens ? n0 + t : n_tokens - 1) * width + (size_t)head * hd + d0;
        if (d0 < rot) rope_eight<SLICED>(qkv, S, slice, at, v[t]);
        else row[t] = rope_copy<SLICED>(qkv, S, slice, at);
    }
#pragma unroll
    for (int t = 0; t < RC_TOKENS; ++t) {
        const int n = n0 + t;
        if (n >= n_tokens) break;
        if (d0 < rot) {
            const float* at = cs + t * rot + d0;
#pragma unroll
            for (int p = 0; p < 4; ++p) rope_turn<SLICED>(v[t][2 * p], v[t][2 * p + 1], at[2 * p], at[2 * p + 1], p);
            row[t] = rope_pack(v[t]);
        }
        if (head < H) {
            *(uint4*)(q_out + ((size_t)n * H + head) * hd + d0) = row[t];
        } else if (k_pages) {                              // one chunk of 8 dims
            const int pos = tok_pos[n], page = table[(size_t)tok_seq[n] * table_stride + pos / GFA_PAGE];
            *(uint4*)(k_pages + key_elem(page, head - H, pos % GFA_PAGE, d0, Hkv, hd)) = row[t];
        }
    }
}

// The kernel above wins by its stores of values, where these are many and whole groups of eight keys are the rule:
// by the values of a step and the tokens per sequence on average (rows of the page table).  Microseconds of the kernel of
// few tokens and of this one, values of a token in brackets: 401 tokens (256) 3.3, 4.4; 700 (768) 7.3, 6.0;
// 2,048 (256) 7.1, 5.6; 500 sequences of one (1,024) 7.3, 8.3; 32 of 32 (512) 8.5, 9.1; 20 of 48 (1,024) 12.0, 10.1.
// Two slices: 6,001 (256) 30.1, 32.3; 700 (1,024) 17.7, 18.7; 2,048 (768) 18.5, 13.6; 20 of 100 (1,024) 39.4,
// 40.5.  The angles of its tokens have to fit into shared memory.
static bool rope_cache_prompt(int n_tokens, int n_seqs, int values, int rot, bool sliced) {
    const long long stored = (long long)n_tokens * values;
    return (sliced ? values >= 512 && stored >= 1 << 20 && n_tokens >= 128LL * n_seqs
                   : stored >= (values >= 512 ? 300 << 10 : 1 << 19) && n_tokens >= 48LL * n_seqs) &&
           RC_TOKENS * rot * sizeof(float) <= 32 * 1024;
}

template <bool SLICED>
static int rope_cache_launch(const void* qkv, int S, size_t slice, void* q_out, void* k_pages, void* v_pages,
                             const float* freqs, const int* tok_seq, const int* tok_pos, const int* table,
                             int table_stride, int n_tokens, int H, int Hkv, int hd, int rot, hipStream_t stream) {
    const int qk_blocks = ((H + Hkv) * (hd / 8) + 255) / 256, columns = (n_tokens + RC_TOKENS - 1) / RC_TOKENS;
    // rows of the grid for the values: every column takes RC_VALUE_TOKENS tokens in each of them
    const int v_blocks = v_pages ? ((n_tokens + RC_VALUE_TOKENS - 1) / RC_VALUE_TOKENS + columns - 1) / columns : 0;
    rope_cache_rows_kernel<SLICED><<<dim3(columns, qk_blocks + v_blocks), 256,
                                     RC_TOKENS * (rot > 0 ? rot : 2) * sizeof(float), stream>>>(
        qkv, S, slice, (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, freqs, tok_seq, tok_pos, table,
        table_stride, n_tokens, H, Hkv, hd, rot, qk_blocks);
    return GFA_LAUNCH_RESULT();
}

// part [S, n_tokens, (H + 2 Hkv) * hd] float; interleaved pairs, hd and rot multiples of 8.
extern "C" int gfa_rope_cache_write_sliced(const float* part, int S, void* q_out, void* k_pages,
                                           void* v_pages, const float* freqs, const int* tok_seq,
                                           const int* tok_pos, const int* table, int table_stride,
                                           int n_seqs, int n_tokens, int H, int Hkv, int hd, int rot,
                                           hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (S <= 0 || hd % 8 != 0 || rot % 8 != 0 || rot > hd || (rot > 0 && !freqs))
        return (int)hipErrorInvalidValue;
    const size_t slice = (size_t)n_tokens * (H + 2 * Hkv) * hd;
    if (rope_cache_prompt(n_tokens, n_seqs, v_pages ? Hkv * hd : 0, rot, true))
        return rope_cache_launch<true>(part, S, slice, q_out, k_pages, v_pages, freqs, tok_seq, tok_pos, table,
                                       table_stride, n_tokens, H, Hkv, hd, rot, stream);
    const dim3 grid(n_tokens, ((H + 2 * Hkv) * (hd / 8) + 255) / 256);
    rope_cache_sliced_bf16x8_kernel<<<grid, 256, (size_t)(rot > 0 ? rot : 2) * sizeof(float), stream>>>(
        part, S, slice, (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, freqs, tok_seq, tok_pos,
        table, table_stride, H, Hkv, hd, rot);
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_rope_cache_write(const void* qkv, void* q_out, void* k_pages, void* v_pages,
                                    const float* freqs, const int* tok_seq, const int* tok_pos,
                                    const int* table, int table_stride, int n_seqs, int n_tokens, int H,
                                    int Hkv, int hd, int rot, int layout, int is_bf16,
                                    hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (is_bf16 && layout == 0 && hd % 8 == 0 && rot % 8 == 0) {
        if (rope_cache_prompt(n_tokens, n_seqs, v_pages ? Hkv * hd : 0, rot, false))
            return rope_cache_launch<false>(qkv, 1, 0, q_out, k_pages, v_pages, freqs, tok_seq, tok_pos, table,
                                            table_stride, n_tokens, H, Hkv, hd, rot, stream);
        const dim3 grid8(n_tokens, ((H + 2 * Hkv) * (hd / 8) + 255) / 256);
        rope_cache_bf16x8_kernel<<<grid8, 256, (size_t)(rot > 0 ? rot : 2) * sizeof(float), stream>>>(
            (const bf16_t*)qkv, (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, freqs, tok_seq,
            tok_pos, table, table_stride, H, Hkv, hd, rot);
        return GFA_LAUNCH_RESULT();
    }
    const dim3 grid(n_tokens, ((H + 2 * Hkv) * (hd / 2) + 255) / 256);
    if (is_bf16)
        rope_cache_kernel<bf16_t><<<grid, 256, (size_t)rot * sizeof(float), stream>>>(
            (const bf16_t*)qkv, (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, freqs,
            tok_seq, tok_pos, table, table_stride, H, Hkv, hd, rot, layout);
    else
        rope_cache_kernel<float><<<grid, 256, (size_t)rot * sizeof(float), stream>>>(
            (const float*)qkv, (float*)q_out, (float*)k_pages, (float*)v_pages, freqs, tok_seq,
            tok_pos, table, table_stride, H, Hkv, hd, rot, layout);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// Attention of each new token over its sequence's cache (model.py:209-211 with the mask of
// model.py:134,138): query head h reads kv head h / (H/Hkv); keys j with
// max(0, pos-window+1) <= j <= pos (window 0: from 0); scores scaled, softmax with running
// maximum, all in float.  One workgroup of 128 threads per (head, token); keys in chunks of
// 128, one key per thread for the scores, one output element per thread for the values.
#define AG_THREADS 128
#define AG_MAX_PER_THREAD 4            // head_dim <= 512
template <typename T>
__global__ __launch_bounds__(AG_THREADS) void attention_generic_kernel(
        const T* __restrict__ q, const T* __restrict__ k_pages, const T* __restrict__ v_pages,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
        const int* __restrict__ table, int table_stride, T* __restrict__ out, int H, int Hkv,
        int hd, float scale, int window) {
    extern __shared__ float shared[];
    float* qs = shared;                 // [hd]
    float* sc = shared + hd;            // [AG_THREADS]
    float* scratch = sc + AG_THREADS;   // [16]
    const int n = blockIdx.x, h = blockIdx.y;     // tokens in x: a step may bring millions
    const int g = h / (H / Hkv);
    const int pos = tok_pos[n];
    const int* pages = table + (size_t)tok_seq[n] * table_stride;
    const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const T* qrow = q + ((size_t)n * H + h) * hd;
    for (int d = threadIdx.x; d < hd; d += AG_THREADS) qs[d] = load_as_float(qrow + d);
    __syncthreads();

    float m = -INFINITY, l = 0.f;
    float acc[AG_MAX_PER_THREAD];
#pragma unroll
    for (int i = 0; i < AG_MAX_PER_THREAD; ++i) acc[i] = 0.f;

    for (int base = lo; base <= pos; base += AG_THREADS) {
        const int j = base + threadIdx.x;
        float s = -INFINITY;
        if (j <= pos) {
            const T* kr = k_pages + cache_region(pages[j / GFA_PAGE], g, Hkv, hd);
            float dot = 0.f;
            for (int d = 0; d < hd; ++d)
                dot = fmaf(qs[d], load_as_float(kr + key_offset(j % GFA_PAGE, d, hd)), dot);
            s = dot * scale;
        }
        const float m_new = fmaxf(m, block_max(s, scratch));
        const float alpha = expf(m - m_new);          // 0 on the first chunk (m = -inf)
        const float p = (j <= pos) ? expf(s - m_new) : 0.f;
        sc[threadIdx.x] = p;
        l = l * alpha + block_sum(p, scratch);        // contains the barrier that publishes sc
        const int count = (pos - base + 1 < AG_THREADS) ? pos - base + 1 : AG_THREADS;
#pragma unroll
        for (int i = 0; i < AG_MAX_PER_THREAD; ++i) {
            const int d = threadIdx.x + i * AG_THREADS;
            if (d < hd) {
                float a = acc[i] * alpha;
                for (int jj = 0; jj < count; ++jj) {
                    const int key = base + jj;
                    const T* vr = v_pages + value_elem(pages[key / GFA_PAGE], g, d,
                                                       key % GFA_PAGE, Hkv, hd);
                    a = fmaf(sc[jj], load_as_float(vr), a);
                }
                acc[i] = a;
            }
        }
        m = m_new;
        __syncthreads();
    }
    T* orow = out + ((size_t)n * H + h) * hd;
#pragma unroll
    for (int i = 0; i < AG_MAX_PER_THREAD; ++i) {
        const int d = threadIdx.x + i * AG_THREADS;
        if (d < hd) store_from_float(orow + d, acc[i] / l);
    }
}

// The same for float32 heads of a multiple of 16 (the float32 engine's attention): one workgroup per (token,
// head), whose four waves take every fourth page each with a running maximum of their own, a key per lane
// for the scores and an element (or HD / 64) per lane for the values, both in 16-byte loads that do not
// depend on each other; the waves' results are merged in their order.  What bounds a single-token step is
// the chain of loads, scores, maximum and values of a page: one page per wave at up to 256 keys, where the
// kernel above walks all keys' values one after the other: four requests of the 110M shape, 20 to 200 tokens
// and then 12 steps, 21.4 -> 12.7 ms with it.
// A row's result depends on its position and window alone.  HD: head size rounded up to 64.
// EARLY (head sizes up to 64): a wave's next page is asked for, keys and values at once, before anything waits - the
// first one beside the query, not behind it: 11.01 -> 10.61 ms for the same requests (with the products of
// normed_gemm_f32_kernel); larger heads do not hold a page in registers.  It pays where reads come from memory and few
// waves hide them, and costs the reads of waves that have no page: attention_f32_early.
template <int HD, bool EARLY>
__global__ __launch_bounds__(256) void attention_f32_kernel(
        const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, const int* __restrict__ table,
        int table_stride, float* __restrict__ out, int H, int Hkv, int hd, float scale, int window) {
    constexpr int PER = HD / 64;
    static_assert(!EARLY || HD == 64, "a page of larger heads does not fit the registers");
    __shared__ __attribute__((aligned(16))) float qs[HD];
    __shared__ __attribute__((aligned(16))) float ps[4][GFA_PAGE];
    __shared__ float merged[4][HD + 2];
    const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = h / (H / Hkv);
    const int pos = tok_pos[n];
    const int* pages = table + (size_t)tok_seq[n] * table_stride;
    const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    // by the page's own index, so that a window's first page does not move a key to another wave
    const int first = lo / GFA_PAGE;
    int page = first + ((wave - first) & 3);
    float4 ke[EARLY ? 16 : 1], ve[EARLY ? 16 : 1];
    auto ask = [&](int p) {                                // lanes beyond the head and pages beyond the last: others again
        const int there = p * GFA_PAGE <= pos ? p : pos / GFA_PAGE;
        const size_t region = cache_region(pages[there], g, Hkv, hd);
        const float* kr = k_pages + region + (lane >> 5) * 32 * hd + key_slot(lane & 31) * 8;
        const int d = lane < hd ? lane : 0;
        const float* vr = v_pages + region + (d >> 4) * 1024 + (d & 15) * 8;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float* at = kr + (c * 8 < hd ? c : 0) * 256;
            ke[EARLY ? 2 * c : 0] = *(const float4*)at;
            ke[EARLY ? 2 * c + 1 : 0] = *(const float4*)(at + 4);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            ve[EARLY ? 2 * c : 0] = *(const float4*)(vr + c * 128);
            ve[EARLY ? 2 * c + 1 : 0] = *(const float4*)(vr + c * 128 + 4);
        }
    };
    if (EARLY) ask(page);
    for (int d = threadIdx.x; d < hd; d += 256) qs[d] = q[((size_t)n * H + h) * hd + d];
    __syncthreads();
    float m = -INFINITY, l = 0.f, acc[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) acc[i] = 0.f;
    for (; page * GFA_PAGE <= pos; page += 4) {
        const size_t region = cache_region(pages[page], g, Hkv, hd);
        const int key = page * GFA_PAGE + lane;
        const float* kr = k_pages + region + (lane >> 5) * 32 * hd + key_slot(lane & 31) * 8;
        float dot0 = 0.f, dot1 = 0.f;
        auto chunk = [&](int c, const float4& a, const float4& b) {
            const float4 x = *(const float4*)(qs + c * 8), y = *(const float4*)(qs + c * 8 + 4);
            dot0 = fmaf(a.w, x.w, fmaf(a.z, x.z, fmaf(a.y, x.y, fmaf(a.x, x.x, dot0))));
            dot1 = fmaf(b.w, y.w, fmaf(b.z, y.z, fmaf(b.y, y.y, fmaf(b.x, y.x, dot1))));
        };
        if (EARLY) {
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (c * 8 < hd) chunk(c, ke[EARLY ? 2 * c : 0], ke[EARLY ? 2 * c + 1 : 0]);
        } else {
#pragma unroll 8
            for (int c = 0; c < hd / 8; ++c) chunk(c, *(const float4*)(kr + c * 256), *(const float4*)(kr + c * 256 + 4));
        }
        const bool seen = key >= lo && key <= pos;
        const float s = seen ? (dot0 + dot1) * scale : -INFINITY;
        const float m_new = fmaxf(m, wave_max(s));
        // scores that are no number do not count in a maximum: where there is nothing else the reference is 0, and
        // their weights, and with them the row, are no number either
        const float ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = m_new == -INFINITY ? 1.f : expf(m - m_new);
        const float p = seen ? expf(s - ref) : 0.f;
        l = l * alpha + wave_sum(p);
        m = m_new;
        ps[wave][lane] = p;                                // read by this wave alone
        __builtin_amdgcn_wave_barrier();
        const bool whole = page * GFA_PAGE >= lo && page * GFA_PAGE + GFA_PAGE - 1 <= pos;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int d = lane + 64 * i;
            if (d >= hd) continue;
            const float* vr = v_pages + region + (d >> 4) * 1024 + (d & 15) * 8;
            float sum = acc[i] * alpha;
#pragma unroll
            for (int c = 0; c < 8; ++c) {                  // keys 8 c .. + 7
                float4 a = EARLY ? ve[EARLY ? 2 * c : 0] : *(const float4*)(vr + c * 128);
                float4 b = EARLY ? ve[EARLY ? 2 * c + 1 : 0] : *(const float4*)(vr + c * 128 + 4);
                if (!whole) {                              // slots that hold no seen key are not numbers to use
                    const int k0 = page * GFA_PAGE + 8 * c;
                    if (k0 + 0 < lo || k0 + 0 > pos) a.x = 0.f;
                    if (k0 + 1 < lo || k0 + 1 > pos) a.y = 0.f;
                    if (k0 + 2 < lo || k0 + 2 > pos) a.z = 0.f;
                    if (k0 + 3 < lo || k0 + 3 > pos) a.w = 0.f;
                    if (k0 + 4 < lo || k0 + 4 > pos) b.x = 0.f;
                    if (k0 + 5 < lo || k0 + 5 > pos) b.y = 0.f;
                    if (k0 + 6 < lo || k0 + 6 > pos) b.z = 0.f;
                    if (k0 + 7 < lo || k0 + 7 > pos) b.w = 0.f;
                }
                const float4 x = *(const float4*)(ps[wave] + 8 * c), y = *(const float4*)(ps[wave] + 8 * c + 4);
                sum = fmaf(a.w, x.w, fmaf(a.z, x.z, fmaf(a.y, x.y, fmaf(a.x, x.x, sum))));
                sum = fmaf(b.w, y.w, fmaf(b.z, y.z, fmaf(b.y, y.y, fmaf(b.x, y.x, sum))));
            }
            acc[i] = sum;
        }
        __builtin_amdgcn_wave_barrier();
        if (EARLY && (page + 4) * GFA_PAGE <= pos) ask(page + 4);
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) merged[wave][lane + 64 * i] = acc[i];
    if (lane == 0) {
        merged[wave][HD] = m;
        merged[wave][HD + 1] = l;
    }
    __syncthreads();
    float top = merged[0][HD];
    for (int w = 1; w < 4; ++w) top = fmaxf(top, merged[w][HD]);
    float total = 0.f, part[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        part[w] = merged[w][HD] == -INFINITY ? 0.f : expf(merged[w][HD] - top);
        total = fmaf(merged[w][HD + 1], part[w], total);
    }
    for (int d = threadIdx.x; d < hd; d += 256) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) v = fmaf(merged[w][d], part[w], v);
        out[((size_t)n * H + h) * hd + d] = v / total;
    }
}

// The same for prompts' rows of head sizes up to 64: a workgroup takes four tokens, as they follow each other in the step, of a
// head, and a wave that has a page in its registers works off all of them that are of its sequence.  The kernel above
// brings every page in anew for every token, 32 KB through the caches for 8,000 multiply-adds, and a wave's time on a page
// is one chain; here four rows' chains run beside each other.  What bounds it still is the way of a wave through its page, loads,
// scores, maximum, values, some 4 us: 717 tokens of four prompts, 12 heads of 64: 59 -> 27 us; one prompt of 200 21 -> 12, of 2,048
// 459 -> 229; 32 heads on 4 128 -> 59, 40 -> 23, 1,196 -> 564.  Eight rows hold too many registers (717: 44 to 56).
// The same arithmetic for a row, so the same bits: its pages are shared out to the waves by their own index; a page that it
// does not see leaves its maximum, sum and elements as they are, and chunks of keys behind its last one are left out.
// A group of four may hold rows of several sequences: its workgroup takes the first run of one sequence, further ones begin
// "inside" and are shared out to workgroups behind the groups', 8 to AF_SLICES for every 64 tokens by the number of sequences: one for
// each but the first were enough where a sequence's tokens follow each other, but 2 x 200 in turn then take 164 us and not 43.
// SINGLES: a run of one token, a decode step's beside prompts, has a code of its own, since that for four takes as long for one: 172
// tokens and one behind 1,800 keys 43 -> 24 us (one at a time 26), 640 and fifteen behind 1,900 126 -> 65 (98).  A single sequence does
// without it, whose code for four then is 1 to 2 % faster.
#define AF_ROWS 4
#define AF_SLICES 16
template <bool SINGLES>
__global__ __launch_bounds__(256, 3) void attention_f32_rows_kernel(
        const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, const int* __restrict__ table,
        int table_stride, float* __restrict__ out, int n_tokens, int slices, int H, int Hkv, int hd, float scale, int window) {
    static_assert(AF_ROWS == 4, "a thread for every element of the queries");
    __shared__ __attribute__((aligned(16))) float qs[AF_ROWS][64];
    __shared__ __attribute__((aligned(16))) float ps[4][AF_ROWS][GFA_PAGE];
    __shared__ float merged[4][AF_ROWS][66];
    const int h = blockIdx.y, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = h / (H / Hkv), groups = (n_tokens + AF_ROWS - 1) / AF_ROWS;
    int base = blockIdx.x * AF_ROWS;
    unsigned long long starts = 1;                         // tokens base + bit: where this workgroup's runs begin
    if ((int)blockIdx.x >= groups) {                       // every slices-th of those that begin inside a group
        const int slice = ((int)blockIdx.x - groups) % slices;
        base = ((int)blockIdx.x - groups) / slices * 64;
        const int n = base + lane;
        const int there = n < n_tokens ? n : 0;
        unsigned long long all = __ballot(there % AF_ROWS != 0 && tok_seq[there] != tok_seq[there > 0 ? there - 1 : 0]);
        starts = 0;
        for (int i = 0; all; ++i, all &= all - 1)
            if (i % slices == slice) starts |= all & -all;
    }
    // the run of `count` tokens from n0 on, worked off by a code for ROWS
    auto walk = [&](auto rows, int n0, int count, int seq) {
        constexpr int ROWS = decltype(rows)::value;
        int lane = threadIdx.x & 63;
        if (SINGLES) asm("" : "+v"(lane));                 // what follows from it is not kept through both codes
        const unsigned vd = lane < hd ? lane : 0;
        const unsigned k_at = (lane >> 5) * 32 * hd + key_slot(lane & 31) * 8, v_at = (vd >> 4) * 1024 + (vd & 15) * 8;
        {                                                  // rows beyond the last: the last one again, not seen
            const int row = wave < count ? wave : count - 1;
            if (lane < hd) qs[wave][lane] = q[((size_t)(n0 + row) * H + h) * hd + lane];
        }
        __syncthreads();
        float m[ROWS], l[ROWS], acc[ROWS];
#pragma unroll
        for (int t = 0; t < ROWS; ++t) {
            m[t] = -INFINITY;
            l[t] = acc[t] = 0.f;
        }
        int pos[ROWS], lo[ROWS];                           // the keys that a row sees; none: another sequence's
        int last = -1, least = 1 << 30, all_from = 0, all_to = 1 << 30;
#pragma unroll
        for (int t = 0; t < ROWS; ++t) {
            const bool in = t < count;
            pos[t] = in ? tok_pos[n0 + (in ? t : 0)] : -1;
            lo[t] = window > 0 && pos[t] - window + 1 > 0 ? pos[t] - window + 1 : 0;
            if (in && lo[t] < least) least = lo[t];
            if (pos[t] > last) last = pos[t];
            if (lo[t] > all_from) all_from = lo[t];
            if (in && pos[t] < all_to) all_to = pos[t];    // what the others add up is not stored
        }
        const int* pages = table + (size_t)seq * table_stride;
        const int first = least / GFA_PAGE;
        for (int page = first + ((wave - first) & 3); page * GFA_PAGE <= last; page += 4) {
            const size_t region = cache_region(pages[page], g, Hkv, hd);
            const float *kr = k_pages + region, *vr = v_pages + region;
            float4 ke[16], ve[16];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const float* at = kr + (c * 8 < hd ? c : 0) * 256;
                ke[2 * c] = *(const float4*)(at + k_at);
                ke[2 * c + 1] = *(const float4*)(at + k_at + 4);
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                ve[2 * c] = *(const float4*)(vr + c * 128 + v_at);
                ve[2 * c + 1] = *(const float4*)(vr + c * 128 + v_at + 4);
            }
            float dot0[ROWS], dot1[ROWS];
#pragma unroll
            for (int t = 0; t < ROWS; ++t) dot0[t] = dot1[t] = 0.f;
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (c * 8 < hd) {
                    const float4 a = ke[2 * c], b = ke[2 * c + 1];
#pragma unroll
                    for (int t = 0; t < ROWS; ++t) {
                        const float4 x = *(const float4*)(qs[t] + c * 8), y = *(const float4*)(qs[t] + c * 8 + 4);
                        dot0[t] = fmaf(a.w, x.w, fmaf(a.z, x.z, fmaf(a.y, x.y, fmaf(a.x, x.x, dot0[t]))));
                        dot1[t] = fmaf(b.w, y.w, fmaf(b.z, y.z, fmaf(b.y, y.y, fmaf(b.x, y.x, dot1[t]))));
                    }
                }
            const int key = page * GFA_PAGE + lane;
#pragma unroll
            for (int t = 0; t < ROWS; ++t) {
                const bool seen = key >= lo[t] && key <= pos[t];
                const float s = seen ? (dot0[t] + dot1[t]) * scale : -INFINITY;
                const float m_new = fmaxf(m[t], wave_max(s));
                const float ref = m_new == -INFINITY ? 0.f : m_new;
                const float alpha = m_new == -INFINITY ? 1.f : expf(m[t] - m_new);
                const float p = seen ? expf(s - ref) : 0.f;
                l[t] = l[t] * alpha + wave_sum(p);
                m[t] = m_new;
                acc[t] *= alpha;
                ps[wave][t][lane] = p;                     // read by this wave alone
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int c = 0; c < 8; ++c) {                  // keys 8 c .. + 7
                const int k0 = page * GFA_PAGE + 8 * c;
                if (k0 > last) break;
                const float4 a = ve[2 * c], b = ve[2 * c + 1];
                auto add = [&](int t, const float4& a, const float4& b) {
                    const float4 x = *(const float4*)(ps[wave][t] + 8 * c), y = *(const float4*)(ps[wave][t] + 8 * c + 4);
                    float sum = acc[t];
                    sum = fmaf(a.w, x.w, fmaf(a.z, x.z, fmaf(a.y, x.y, fmaf(a.x, x.x, sum))));
                    sum = fmaf(b.w, y.w, fmaf(b.z, y.z, fmaf(b.y, y.y, fmaf(b.x, y.x, sum))));
                    acc[t] = sum;
                };
                if (k0 >= all_from && k0 + 7 <= all_to) {  // seen by all rows
#pragma unroll
                    for (int t = 0; t < ROWS; ++t) add(t, a, b);
                    continue;
                }
#pragma unroll
                for (int t = 0; t < ROWS; ++t) {
                    if (k0 > pos[t] || k0 + 7 < lo[t]) continue;
                    float4 u = a, v = b;                   // slots that hold no seen key are not numbers to use
                    if (k0 + 0 < lo[t]) u.x = 0.f;
                    if (k0 + 1 < lo[t] || k0 + 1 > pos[t]) u.y = 0.f;
                    if (k0 + 2 < lo[t] || k0 + 2 > pos[t]) u.z = 0.f;
                    if (k0 + 3 < lo[t] || k0 + 3 > pos[t]) u.w = 0.f;
                    if (k0 + 4 < lo[t] || k0 + 4 > pos[t]) v.x = 0.f;
                    if (k0 + 5 < lo[t] || k0 + 5 > pos[t]) v.y = 0.f;
                    if (k0 + 6 < lo[t] || k0 + 6 > pos[t]) v.z = 0.f;
                    if (k0 + 7 > pos[t]) v.w = 0.f;
                    add(t, u, v);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int t = 0; t < ROWS; ++t) {
            merged[wave][t][lane] = acc[t];
            if (lane == 0) {
                merged[wave][t][64] = m[t];
                merged[wave][t][65] = l[t];
            }
        }
        __syncthreads();
        for (int t = wave; t < count; t += 4) {
            float top = merged[0][t][64];
            for (int w = 1; w < 4; ++w) top = fmaxf(top, merged[w][t][64]);
            float total = 0.f, part[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                part[w] = merged[w][t][64] == -INFINITY ? 0.f : expf(merged[w][t][64] - top);
                total = fmaf(merged[w][t][65], part[w], total);
            }
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) v = fmaf(merged[w][t][lane], part[w], v);
            if (lane < hd) out[((size_t)(n0 + t) * H + h) * hd + lane] = v / total;
        }
        __syncthreads();
    };
    for (; starts; starts &= starts - 1) {
        const int n0 = base + __builtin_ctzll(starts);
        const int seq = tok_seq[n0];
        int count = 1;
        while (n0 + count < n_tokens && (n0 + count) % AF_ROWS != 0 && tok_seq[n0 + count] == seq) ++count;
        if (SINGLES && count == 1) walk(std::integral_constant<int, 1>(), n0, count, seq);
        else walk(std::integral_constant<int, AF_ROWS>(), n0, count, seq);
    }
}

// Whether a step's rows go four at a time; pages: the most that its table has for a sequence.  Not where the groups would
// be too few to hide a wave's way; of several sequences, whose shares of the tokens and keys the host does not know, where it was the faster way
// for all that were measured.  us, one at a time and four, 12 heads of 64: one prompt of 60 8.4, 8.6; 100 12.4, 9.6; 60 behind 2,000 keys
// 39, 47; 100 behind 900 31, 28; several: 4 x 50 behind 900 56, 39; 600 and eight single tokens behind 900 74, 43; 640 and fifteen
// behind 1,900 94, 65.  On the other side 64 single tokens behind 100 12.8, 18.6; 16 behind 900 19.7, 20.6 (32 heads on 4 16.3, 42.3); 4 x 30
// behind 300 20.3, 20.4 (6 heads of 48 10.3, 13.4); but also 20 x 7 17.0, 9.4, behind 200 35, 19, and 30 x 9 behind 100 32, 21.
static bool attention_f32_four(int n_tokens, int n_seqs, int H, int hd, int pages) {
    if (hd > 64) return false;
    if (n_seqs <= 1) return (long long)n_tokens * H >= 1024;
    return n_tokens >= 40ll * n_seqs && (long long)n_tokens * H >= 2048 && pages <= 32;
}

// Whether a step whose rows go one at a time asks early; pages: as above.  Not where there are many workgroups (one
// a token and head) and they walk many pages, or share the keys of a group, which then are in the caches.  us, early and
// not, heads of 64, keys out of memory: 12 heads, a token behind 30 keys 5.6, 6.7; 16 behind 1,000 25.7, 26.2; 32 heads on 4, a token
// behind 1,000 15.6, 17.2; out of the caches: 12 heads, 64 tokens behind 900 65, 68; 64 sequences of 4 behind 100 33, 38; 40 of 30
// 90, 103, behind 500 with a window of 128 101, 123; 3 of 100 behind 3,000 213, 210; 32 heads on 4, 64 of 4 behind 100 55, 54; 32 of 4 behind
// 900 145, 128; 40 of 30 222, 202 (but behind 500 504, 550), with the window 249, 310.  Heads of 48, whose loads are not whole lines: 6 heads, 64 of 4
// behind 100 17, 20; 40 of 30 47, 68.
static bool attention_f32_early(int n_tokens, int H, int Hkv, int hd, int pages, int window) {
    if (window > 0 && window / GFA_PAGE + 2 < pages) pages = window / GFA_PAGE + 2;
    if ((long long)n_tokens * H < 2048 || hd == 48) return hd <= 64;
    return hd <= 64 && pages < 10 && (window > 0 || H < 4 * Hkv);
}

extern "C" int gfa_attention_generic(const void* q, const void* k_pages, const void* v_pages,
                                     const int* tok_seq, const int* tok_pos, const int* table,
                                     int table_stride, int n_seqs, void* out, int n_tokens, int H, int Hkv,
                                     int hd, float scale, int window, int is_bf16,
                                     hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (hd > AG_THREADS * AG_MAX_PER_THREAD || H > 65535) return (int)hipErrorInvalidValue;
    dim3 grid(n_tokens, H);
    // 16-byte loads of the cache's operand order need it to begin at such an address
    if (!is_bf16 && hd % 16 == 0 && hd <= 256 && (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0) {
#define AF_GO(HD, EARLY) attention_f32_kernel<HD, EARLY><<<grid, 256, 0, stream>>>((const float*)q, (const float*)k_pages, \
        (const float*)v_pages, tok_seq, tok_pos, table, table_stride, (float*)out, H, Hkv, hd, scale, window)
        if (attention_f32_four(n_tokens, n_seqs, H, hd, table_stride)) {
            const int groups = (n_tokens + AF_ROWS - 1) / AF_ROWS;
            const int slices = n_seqs <= 1 ? 0 : n_seqs <= 8 ? 8 : n_seqs < AF_SLICES ? n_seqs : AF_SLICES;
#define AF_ROWS_GO(SINGLES) attention_f32_rows_kernel<SINGLES><<<dim3(groups + (n_tokens + 63) / 64 * slices, H), 256, 0, stream>>>( \
        (const float*)q, (const float*)k_pages, (const float*)v_pages, tok_seq, tok_pos, table, table_stride, (float*)out, n_tokens, slices, \
        H, Hkv, hd, scale, window)
            if (n_seqs > 1) AF_ROWS_GO(true);
            else AF_ROWS_GO(false);
#undef AF_ROWS_GO
        } else if (attention_f32_early(n_tokens, H, Hkv, hd, table_stride, window)) AF_GO(64, true);
        else if (hd <= 64) AF_GO(64, false);
        else if (hd <= 128) AF_GO(128, false);
        else AF_GO(256, false);
#undef AF_GO
        return GFA_LAUNCH_RESULT();
    }
    const size_t shmem = (size_t)(hd + AG_THREADS + 16) * sizeof(float);
    if (is_bf16)
        attention_generic_kernel<bf16_t><<<grid, AG_THREADS, shmem, stream>>>(
            (const bf16_t*)q, (const bf16_t*)k_pages, (const bf16_t*)v_pages, tok_seq, tok_pos,
            table, table_stride, (bf16_t*)out, H, Hkv, hd, scale, window);
    else
        attention_generic_kernel<float><<<grid, AG_THREADS, shmem, stream>>>(
            (const float*)q, (const float*)k_pages, (const float*)v_pages, tok_seq, tok_pos,
            table, table_stride, (float*)out, H, Hkv, hd, scale, window);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// gate: out[n, i] = pair(gu[n, i], gu[n, I + i]) with pair(a, b) = act(a) * b; act 0 = silu
// (model.py:227), 1 = the tanh form of gelu, 0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))).  act 2
// clamps both first, a <- min(a, limit), b <- min(max(b, -limit), limit), and gives
// a sigmoid(1.702 a) (b + 1).
template <int ACT>
__device__ __forceinline__ float gate_pair(float a, float b, float limit) {
    if (ACT == 0) return a / (1.f + expf(-a)) * b;
    if (ACT == 2) {
        a = fminf(a, limit);
        b = fminf(fmaxf(b, -limit), limit);
        return a / (1.f + expf(-1.702f * a)) * (b + 1.f);
    }
    return 0.5f * a * (1.f + tanhf(0.7978845608028654f * (a + 0.044715f * a * a * a))) * b;
}

template <typename T, int ACT>
__global__ void gate_mul_kernel(const T* __restrict__ gu, T* __restrict__ out, int I,
                                size_t total, float limit) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const size_t n = e / I;
        const int i = (int)(e % I);
        const float a = load_as_float(gu + n * 2 * I + i);
        const float b = load_as_float(gu + n * 2 * I + I + i);
        store_from_float(out + e, gate_pair<ACT>(a, b, limit));
    }
}

// bfloat16 rows whose width is a multiple of 8: eight elements per thread, 16-byte accesses
template <int ACT>
__global__ __launch_bounds__(256) void gate_mul_bf16x8_kernel(const bf16_t* __restrict__ gu,
                                                              bf16_t* __restrict__ out, int I8,
                                                              size_t total8, float limit) {
    const size_t e = blockIdx.x * (size_t)256 + threadIdx.x;
    if (e >= total8) return;
    const size_t n = e / I8;
    const int i = (int)(e - n * I8);
    const uint4 a = ((const uint4*)gu)[n * 2 * I8 + i], b = ((const uint4*)gu)[n * 2 * I8 + I8 + i];
    const bf16_t* ae = (const bf16_t*)&a;
    const bf16_t* be = (const bf16_t*)&b;
    uint4 o;
    bf16_t* oe = (bf16_t*)&o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
        oe[j] = float_to_bf16(gate_pair<ACT>(bf16_to_float(ae[j]), bf16_to_float(be[j]), limit));
    ((uint4*)out)[e] = o;
}

template <int ACT>
static int launch_gate_mul(const void* gu, void* out, int n_rows, int I, int is_bf16, float limit,
                           hipStream_t stream) {
    const size_t total = (size_t)n_rows * I;
    if (total == 0) return 0;
    if (is_bf16 && I % 8 == 0) {
        const size_t total8 = total / 8;
        gate_mul_bf16x8_kernel<ACT><<<(unsigned)((total8 + 255) / 256), 256, 0, stream>>>(
            (const bf16_t*)gu, (bf16_t*)out, I / 8, total8, limit);
        return GFA_LAUNCH_RESULT();
    }
    const int blocks = (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535);
    if (is_bf16)
        gate_mul_kernel<bf16_t, ACT><<<blocks, 256, 0, stream>>>((const bf16_t*)gu, (bf16_t*)out, I, total, limit);
    else
        gate_mul_kernel<float, ACT><<<blocks, 256, 0, stream>>>((const float*)gu, (float*)out, I, total, limit);
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_gate_mul(const void* gu, void* out, int n_rows, int I, int act, float limit, int is_bf16,
                            hipStream_t stream) {
    if (act == 0) return launch_gate_mul<0>(gu, out, n_rows, I, is_bf16, limit, stream);
    if (act == 1) return launch_gate_mul<1>(gu, out, n_rows, I, is_bf16, limit, stream);
    if (act == 2) return launch_gate_mul<2>(gu, out, n_rows, I, is_bf16, limit, stream);
    return (int)hipErrorInvalidValue;
}

extern "C" int gfa_silu_mul(const void* gu, void* out, int n_rows, int I, int is_bf16,
                            hipStream_t stream) {
    return launch_gate_mul<0>(gu, out, n_rows, I, is_bf16, 0.f, stream);
}

// --------------------------------------------------------------------------------------
// Few rows in float32: a norm, the product behind it and what follows that in one kernel, for the two products
// of a layer that read a norm.  out = act(n Wg^T) * (n Wu^T) with the gate's act (EPI 0 silu, 1 gelu's tanh form,
// w = rows of Wg, then of Wu), or q, k, v = n W^T rotated and stored (EPI 2, interleaved pairs, as
// rope_cache_kernel); n = x * rsqrt(mean(x^2) + eps) * g.
//
// What bounds a layer of few rows is its chain of kernels, 4 to 8 us each whatever they do: a norm, the rotation
// and the gate take 4 to 5 beside products of 5 to 8 (four rows, 768 columns).  Every workgroup reads all of x
// anyway, so each works the rows' factors out for itself, while its first weights are on the way: five kernels a
// layer and not nine, four rows of 768 columns 40 -> 33 us (few_row_f32_fused: up to where).
//
// The same bits as rmsnorm_vec_kernel, gemm_f32_kernel and the kernels behind them: the squares are added by as
// many lanes and in the order of that norm kernel's (256 or 1,024 threads by the width), the products as four chains of
// every fourth 32 k.  K a multiple of 4 up to 4,096, M <= 16, 16-byte aligned rows.
struct NormedEpilogue {
    float* out;                           // EPI 0, 1: [M, N]
    float *q, *k_pages, *v_pages;         // EPI 2
    const float* freqs;
    const int *tok_seq, *tok_pos, *table;
    int table_stride, H, Hkv, hd, rot;
};

template <int EPI>
__global__ __launch_bounds__(256, 2) void normed_gemm_f32_kernel(
        const float* __restrict__ x, const float* __restrict__ g, const float* __restrict__ w, int M, int N, int K,
        float eps, NormedEpilogue e) {
    constexpr int COLS = EPI == 2 ? 16 : 8;
    __shared__ __attribute__((aligned(16))) char lds[4 * 32 * GS_PITCH];
    __shared__ gf_floatx4_t sums[4][64];
    __shared__ float squares[16][16], factor[16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int n0 = blockIdx.x * COLS;
    // what follows the product, asked for in front of it: the lane's row and four columns, their rotation and their place
    const int m = li, n = n0 + 4 * lg;
    const bool mine = wave == 0 && m < M && n < N && 4 * lg < COLS;
    int pos = 0, seq = 0, page = 0, head = 0, d = 0;
    float freq[2] = {0.f, 0.f};
    if (EPI == 2 && mine) {
        head = n / e.hd;                           // hd is a multiple of 16: the columns of one head
        d = n - head * e.hd;
        pos = e.tok_pos[m];
        seq = e.tok_seq[m];
        if (head < e.H + e.Hkv) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
                if (d + 2 * p < e.rot) freq[p] = e.freqs[(d + 2 * p) >> 1];
        }
    }
    // a gate's tile: eight rows of Wg and the same eight of Wu, which keeps as many workgroups at work as sixteen
    // columns of a plain product (four rows, 768 -> 2 x 2,048: 9 us; two tiles each in half as many, 11)
    unsigned from[4];                              // rows beyond the last read it again, never stored
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * (i & 1) + (lane >> 3), wr = EPI == 2 ? r : lane >> 3;
        const int row = i < 2 ? (r < M ? r : M - 1) : (wr < N - n0 ? wr : N - n0 - 1);
        from[i] = (unsigned)row * (unsigned)(4 * K) + 16 * (lane & 7);
    }
    const char* wt = (const char*)(w + (size_t)n0 * K);
    float rs[2] = {0.f, 0.f};
    gf_floatx4_t acc[1][1] = {{gf_floatx4_t{0.f, 0.f, 0.f, 0.f}}};
    // 64 lanes at a time of the norm kernel's threads
    const int groups = K <= 1024 ? 4 : 16, n4 = K >> 2;
    gf_piped<1, 1, 4, true>((const char*)x, wt, EPI == 2 ? wt : (const char*)(w + ((size_t)N + n0) * K), from, g, rs, K,
                            lds + wave * 32 * GS_PITCH, acc, [&] {
        if (EPI == 2 && mine && head >= e.H) page = e.table[(size_t)seq * e.table_stride + pos / GFA_PAGE];
        for (int group = wave; group < groups; group += 4) {
            const int at = group * 64 + lane;
#pragma unroll 4
            for (int r = 0; r < M; ++r) {
                const float4 v = at < n4 ? ((const float4*)(x + (size_t)r * K))[at] : make_float4(0.f, 0.f, 0.f, 0.f);
                float ss = 0.f;
                ss = fmaf(v.x, v.x, ss);
                ss = fmaf(v.y, v.y, ss);
                ss = fmaf(v.z, v.z, ss);
                ss = fmaf(v.w, v.w, ss);
                ss = wave_sum(ss);
                if (lane == 0) squares[r][group] = ss;
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < M) {
            float ss = 0.f;
            for (int i = 0; i < groups; ++i) ss += squares[threadIdx.x][i];
            factor[threadIdx.x] = rsqrtf(ss / (float)K + eps);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = 8 * i + (lane >> 3);
            rs[i] = factor[r < M ? r : M - 1];
        }
    });
    sums[wave][lane] = acc[0][0];
    __syncthreads();
    if (wave != 0) return;
    const gf_floatx4_t v = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
    float up[4];
    if (EPI != 2) {                                // lanes 32 .. 63 hold the sums of Wu
#pragma unroll
        for (int q = 0; q < 4; ++q) up[q] = __shfl_xor(v[q], 32, GFA_WAVE);
    }
    if (!mine) return;                             // four columns of a row
    if (EPI != 2) {
        float* o = e.out + (size_t)m * N + n;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (n + q < N) o[q] = gate_pair<EPI == 1 ? 1 : 0>(v[q], up[q], 0.f);
        return;
    }
    const int hd = e.hd, off = pos % GFA_PAGE;
    float r[4] = {v[0], v[1], v[2], v[3]};
    if (head < e.H + e.Hkv) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
            if (d + 2 * p < e.rot) {
                float s, c;
                sincosf((float)pos * freq[p], &s, &c);
                const float a = r[2 * p], b = r[2 * p + 1];
                r[2 * p] = a * c - b * s;
                r[2 * p + 1] = b * c + a * s;
            }
    }
    if (head < e.H) {
        *(float4*)(e.q + ((size_t)m * e.H + head) * hd + d) = make_float4(r[0], r[1], r[2], r[3]);
        return;
    }
    if (head < e.H + e.Hkv) {
        float* k = e.k_pages + cache_region(page, head - e.H, e.Hkv, hd);
#pragma unroll
        for (int q = 0; q < 4; ++q) k[key_offset(off, d + q, hd)] = r[q];
    } else {
        float* vp = e.v_pages + cache_region(page, head - e.H - e.Hkv, e.Hkv, hd);
#pragma unroll
        for (int q = 0; q < 4; ++q) vp[value_offset(d + q, off, hd)] = r[q];
    }
}

// Whether the products work the norms out themselves.  Every workgroup then goes through all rows again, 256 float4 at
// a time up to 1,024 columns and 1,024 beyond; with more rows or wider ones the separate kernels are the faster way.
// us a layer, fused and separate (30 keys): 288 columns, 16 rows 28.6, 31.0; 512, 16 31.6, 33.9; 768, 4 33.3, 40.0; 12 40.3, 41.7; 14
// 42.4, 42.2; 1,024, 12 47.6, 49.0; 16 51.5, 50.4; 1,536, 5 58.3, 58.5; 6 60.3, 58.9; 2,048, 5 69.1, 69.8; 6 71.1, 70.1; 16 94,
// 77; 3,072, 4 116.9, 117.5; 5 120.2, 117.9; 4,096, 1 185, 197; 3 189, 195; 5 197, 194; 16 256, 207.
static bool few_row_f32_fused(int M, int D) {
    return D <= 1024 ? M <= 12 || D <= 512 : D <= 4096 && M <= 5 && M * D <= 12288;
}

struct FewRowWorkF32 {
    size_t q, y, h, xn, qkv, gu, bytes;
    bool fused;
    FewRowWorkF32(int M, int D, int I, int H, int Hkv, int hd) {
        fused = few_row_f32_fused(M, D);
        size_t at = 0;
        auto take = [&](size_t n) { const size_t o = at; at += (n * 4 + 255) / 256 * 256; return o; };
        q = take((size_t)M * H * hd);
        y = take((size_t)M * H * hd);
        h = take((size_t)M * I);
        xn = take(fused ? 0 : (size_t)M * D);
        qkv = take(fused ? 0 : (size_t)M * (H + 2 * Hkv) * hd);
        gu = take(fused ? 0 : (size_t)M * 2 * I);
        bytes = at;
    }
};

extern "C" long gfa_few_row_work_bytes_f32(int M, int D, int I, int H, int Hkv, int hd) {
    return (long)FewRowWorkF32(M, D, I, H, Hkv, hd).bytes;
}

// The layers' launches: five a layer, nine where norms, rotation and gate are kernels of their own.
extern "C" int gfa_few_row_layers_f32(const FewRowLayer* layers, int n_layers, const FewRowStep* step, hipStream_t stream) {
    const FewRowStep& s = *step;
    const int inner = s.H * s.hd;
    if (n_layers <= 0 || s.M <= 0 || s.M > 16 || s.D <= 0 || s.D % 4 || s.D > 4096 || s.I <= 0 || s.I % 4 ||
        s.hd <= 0 || s.hd % 16 || s.hd > 256 || s.rot % 2 || s.rot > s.hd || (s.gate_mode != 0 && s.gate_mode != 1) ||
        (uintptr_t)s.residual % 16 || (uintptr_t)s.work % 16)
        return (int)hipErrorInvalidValue;
    const FewRowWorkF32 at(s.M, s.D, s.I, s.H, s.Hkv, s.hd);
    float* q = (float*)((char*)s.work + at.q);
    float* y = (float*)((char*)s.work + at.y);
    float* h = (float*)((char*)s.work + at.h);
    float* xn = (float*)((char*)s.work + at.xn);
    float* qkv = (float*)((char*)s.work + at.qkv);
    float* gu = (float*)((char*)s.work + at.gu);
    const int n_qkv = (s.H + 2 * s.Hkv) * s.hd;
    int rc = 0;
    for (int l = 0; l < n_layers && rc == 0; ++l) {
        const FewRowLayer& L = layers[l];
        if ((uintptr_t)L.wqkv % 16 || (uintptr_t)L.w13 % 16 || (uintptr_t)L.norm_mixer % 16 || (uintptr_t)L.norm_ffn % 16)
            return (int)hipErrorInvalidValue;
        NormedEpilogue e = {};
        if (at.fused) {
            e.q = q;
            e.k_pages = (float*)L.k_pages;
            e.v_pages = (float*)L.v_pages;
            e.freqs = s.freqs;
            e.tok_seq = s.tok_seq;
            e.tok_pos = s.tok_pos;
            e.table = L.table;
            e.table_stride = s.table_stride;
            e.H = s.H; e.Hkv = s.Hkv; e.hd = s.hd; e.rot = s.rot;
            normed_gemm_f32_kernel<2><<<n_qkv / 16, 256, 0, stream>>>(s.residual, L.norm_mixer, (const float*)L.wqkv, s.M,
                                                                      n_qkv, s.D, s.eps_mixer, e);
        } else {
            rc = gfa_rmsnorm(s.residual, L.norm_mixer, nullptr, xn, 0, s.M, s.D, s.eps_mixer, stream);
            if (rc) break;
            rc = gfa_gemm_f32(xn, (const float*)L.wqkv, qkv, s.M, n_qkv, s.D, s.D, n_qkv, 0, stream);
            if (rc) break;
            rc = gfa_rope_cache_write(qkv, q, L.k_pages, L.v_pages, s.freqs, s.tok_seq, s.tok_pos, L.table, s.table_stride,
                                      s.n_seqs, s.M, s.H, s.Hkv, s.hd, s.rot, 0, 0, stream);
            if (rc) break;
        }
        rc = gfa_attention_generic(q, L.k_pages, L.v_pages, s.tok_seq, s.tok_pos, L.table, s.table_stride, s.n_seqs, y, s.M,
                                   s.H, s.Hkv, s.hd, s.scale, s.window, 0, stream);
        if (rc) break;
        rc = gfa_gemm_f32(y, (const float*)L.wo, s.residual, s.M, s.D, inner, inner, s.D, 1, stream);
        if (rc) break;
        if (at.fused) {
            e.out = h;
            if (s.gate_mode == 0)
                normed_gemm_f32_kernel<0><<<(s.I + 7) / 8, 256, 0, stream>>>(s.residual, L.norm_ffn, (const float*)L.w13,
                                                                              s.M, s.I, s.D, s.eps_ffn, e);
            else
                normed_gemm_f32_kernel<1><<<(s.I + 7) / 8, 256, 0, stream>>>(s.residual, L.norm_ffn, (const float*)L.w13,
                                                                              s.M, s.I, s.D, s.eps_ffn, e);
        } else {
            rc = gfa_rmsnorm(s.residual, L.norm_ffn, nullptr, xn, 0, s.M, s.D, s.eps_ffn, stream);
            if (rc) break;
            rc = gfa_gemm_f32(xn, (const float*)L.w13, gu, s.M, 2 * s.I, s.D, s.D, 2 * s.I, 0, stream);
            if (rc) break;
            rc = gfa_gate_mul(gu, h, s.M, s.I, s.gate_mode, 0.f, 0, stream);
            if (rc) break;
        }
        rc = gfa_gemm_f32(h, (const float*)L.w2, s.residual, s.M, s.D, s.I, s.I, s.D, 1, stream);
    }
    return rc;
}

// --------------------------------------------------------------------------------------
// residual sum in float: res[e] += float(y[e])          (model.py:162-163)
template <typename T>
__global__ void add_into_kernel(float* __restrict__ res, const T* __restrict__ y, size_t total) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x)
        res[e] += load_as_float(y + e);
}

// bfloat16 addend, four elements per thread
__global__ __launch_bounds__(256) void add_into_bf16x4_kernel(float4* __restrict__ res,
                                                              const uint2* __restrict__ y,
                                                              size_t total4) {
    const size_t e = blockIdx.x * (size_t)256 + threadIdx.x;
    if (e >= total4) return;
    float4 r = res[e];
    const uint2 v = y[e];
    r.x += __uint_as_float(v.x << 16);
    r.y += __uint_as_float(v.x & 0xffff0000u);
    r.z += __uint_as_float(v.y << 16);
    r.w += __uint_as_float(v.y & 0xffff0000u);
    res[e] = r;
}

extern "C" int gfa_add_into(float* res, const void* y, size_t total, int y_bf16,
                            hipStream_t stream) {
    if (total == 0) return 0;
    if (y_bf16 && total % 4 == 0 && ((uintptr_t)res % 16 == 0) && ((uintptr_t)y % 8 == 0)) {
        const size_t total4 = total / 4;
        add_into_bf16x4_kernel<<<(unsigned)((total4 + 255) / 256), 256, 0, stream>>>(
            (float4*)res, (const uint2*)y, total4);
        return GFA_LAUNCH_RESULT();
    }
    const int blocks = (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535);
    if (y_bf16)
        add_into_kernel<bf16_t><<<blocks, 256, 0, stream>>>(res, (const bf16_t*)y, total);
    else
        add_into_kernel<float><<<blocks, 256, 0, stream>>>(res, (const float*)y, total);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// x[e] = scale * x[e], then, if cap > 0, cap * tanh(x[e] / cap): a factor on the embedded
// rows or on the logits, and a soft cap of the logits, for plans that state one.
__global__ void scale_cap_kernel(float* __restrict__ x, size_t total, float scale, float cap) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        float v = x[e] * scale;
        if (cap > 0.f) v = cap * tanhf(v / cap);
        x[e] = v;
    }
}

extern "C" int gfa_scale_cap(float* x, size_t total, float scale, float cap, hipStream_t stream) {
    if (total == 0) return 0;
    const int blocks = (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535);
    scale_cap_kernel<<<blocks, 256, 0, stream>>>(x, total, scale, cap);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// naive matrix product with bfloat16 operands and float accumulation, one thread per
// output: the plain counterpart of the fast bfloat16 kernels (tests only).
__global__ void gemm_bf16_naive_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
                                       float* __restrict__ out, int M, int N, int K) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x, m = blockIdx.y;
    if (n >= N || m >= M) return;
    float acc = 0.f;
    for (int k = 0; k < K; ++k)
        acc = fmaf(bf16_to_float(a[(size_t)m * K + k]), bf16_to_float(w[(size_t)n * K + k]), acc);
    out[(size_t)m * N + n] = acc;
}

extern "C" int gfa_gemm_bf16_naive(const void* a, const void* w, float* out, int M, int N, int K,
                                   hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 65535) return (int)hipErrorInvalidValue;     // rows ride in the grid's second dimension
    dim3 grid((N + 255) / 256, M);
    gemm_bf16_naive_kernel<<<grid, 256, 0, stream>>>((const bf16_t*)a, (const bf16_t*)w, out, M, N, K);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// A sublayer's result joins the stream through a norm of its own ("sandwich" blocks):
//     res[r, :] += y[r, :] * rsqrt(mean(y[r, :]^2) + eps_y) * wy[:]
// and, if next_w is given, the norm that reads the stream next in the same pass:
//     out[r, :] = res[r, :] * rsqrt(mean(res[r, :]^2) + eps_n) * next_w[:]     (type T)
// y is float (a product's float sums).  One workgroup per row; statistics in float.
template <typename T>
__global__ __launch_bounds__(256) void normed_add_kernel(
        float* __restrict__ res, const float* __restrict__ y, const float* __restrict__ wy,
        float eps_y, const float* __restrict__ next_w, float eps_n, T* __restrict__ out, int dim) {
    __shared__ float scratch[16];
    const size_t row = (size_t)blockIdx.x * dim;
    const float* yr = y + row;
    float* rr = res + row;
    float ss = 0.f;
    for (int d = threadIdx.x; d < dim; d += 256) ss = fmaf(yr[d], yr[d], ss);
    ss = block_sum(ss, scratch);
    const float ry = rsqrtf(ss / (float)dim + eps_y);
    float sn = 0.f;
    for (int d = threadIdx.x; d < dim; d += 256) {
        const float v = rr[d] + yr[d] * ry * wy[d];
        rr[d] = v;
        sn = fmaf(v, v, sn);
    }
    if (next_w == nullptr) return;
    sn = block_sum(sn, scratch);
    const float rn = rsqrtf(sn / (float)dim + eps_n);
    T* o = out + row;
    // every thread reads back only what it wrote itself
    for (int d = threadIdx.x; d < dim; d += 256) store_from_float(o + d, rr[d] * rn * next_w[d]);
}

// The same for rows of up to 1024 * VPT * 4 elements (a multiple of 4): y and the stream are
// read once with 16-byte loads and kept in registers between the sums and the stores.
template <typename T, int VPT, int THREADS>
__global__ __launch_bounds__(THREADS) void normed_add_vec_kernel(
        float* __restrict__ res, const float* __restrict__ y, const float* __restrict__ wy,
        float eps_y, const float* __restrict__ next_w, float eps_n, T* __restrict__ out, int dim) {
    __shared__ float scratch[16];
    const size_t row = (size_t)blockIdx.x * dim;
    const float4* y4 = (const float4*)(y + row);
    float4* r4 = (float4*)(res + row);
    const float4* wy4 = (const float4*)wy;
    const int n4 = dim >> 2;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 yv[VPT], rv[VPT];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        yv[j] = idx < n4 ? y4[idx] : zero;
        rv[j] = idx < n4 ? r4[idx] : zero;
        ss = fmaf(yv[j].x, yv[j].x, ss);
        ss = fmaf(yv[j].y, yv[j].y, ss);
        ss = fmaf(yv[j].z, yv[j].z, ss);
        ss = fmaf(yv[j].w, yv[j].w, ss);
    }
    ss = block_sum(ss, scratch);
    const float ry = rsqrtf(ss / (float)dim + eps_y);
    float sn = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            const float4 g = wy4[idx];
            rv[j].x += yv[j].x * ry * g.x;
            rv[j].y += yv[j].y * ry * g.y;
            rv[j].z += yv[j].z * ry * g.z;
            rv[j].w += yv[j].w * ry * g.w;
            r4[idx] = rv[j];
            sn = fmaf(rv[j].x, rv[j].x, sn);
            sn = fmaf(rv[j].y, rv[j].y, sn);
            sn = fmaf(rv[j].z, rv[j].z, sn);
            sn = fmaf(rv[j].w, rv[j].w, sn);
        }
    }
    if (next_w == nullptr) return;
    sn = block_sum(sn, scratch);
    const float rn = rsqrtf(sn / (float)dim + eps_n);
    const float4* nw4 = (const float4*)next_w;
    T* o = out + row;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            const float4 g = nw4[idx];
            store_from_float(o + 4 * idx + 0, rv[j].x * rn * g.x);
            store_from_float(o + 4 * idx + 1, rv[j].y * rn * g.y);
            store_from_float(o + 4 * idx + 2, rv[j].z * rn * g.z);
            store_from_float(o + 4 * idx + 3, rv[j].w * rn * g.w);
        }
    }
}

template <typename T>
static int launch_normed_add(float* res, const float* y, const float* wy, float eps_y,
                             const float* next_w, float eps_n, T* out, int n_rows, int dim,
                             hipStream_t stream) {
    if (dim % 4 == 0 && dim <= 8192) {
        if (dim <= 1024)
            normed_add_vec_kernel<T, 1, 256><<<n_rows, 256, 0, stream>>>(res, y, wy, eps_y, next_w, eps_n, out, dim);
        else if (dim <= 4096)
            normed_add_vec_kernel<T, 1, 1024><<<n_rows, 1024, 0, stream>>>(res, y, wy, eps_y, next_w, eps_n, out, dim);
        else
            normed_add_vec_kernel<T, 2, 1024><<<n_rows, 1024, 0, stream>>>(res, y, wy, eps_y, next_w, eps_n, out, dim);
    } else {
        normed_add_kernel<T><<<n_rows, 256, 0, stream>>>(res, y, wy, eps_y, next_w, eps_n, out, dim);
    }
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_normed_add(float* res, const float* y, const float* wy, float eps_y,
                              const float* next_w, float eps_n, void* out, int out_bf16,
                              int n_rows, int dim, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (out_bf16)
        return launch_normed_add<bf16_t>(res, y, wy, eps_y, next_w, eps_n, (bf16_t*)out, n_rows, dim, stream);
    return launch_normed_add<float>(res, y, wy, eps_y, next_w, eps_n, (float*)out, n_rows, dim, stream);
}

// --------------------------------------------------------------------------------------
// Activations of a feed-forward without a gate, element by element, in float:
//   0 silu, 1 gelu (tanh form), 3 gelu (exact, with erf), 2 xIELU with two numbers a = softplus(p), b = 1/2 + softplus(q):
//     z > 0: a z^2 + z/2        z <= 0: b (exp(z) - 1 - z) + z/2
template <int ACT>
__device__ __forceinline__ float activation(float z, float a, float b) {
    if (ACT == 0) return z / (1.f + expf(-z));
    if (ACT == 1) return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    if (ACT == 3) return 0.5f * z * (1.f + erff(z * 0.7071067811865476f));
    return z > 0.f ? fmaf(a * z, z, 0.5f * z) : fmaf(b, expm1f(z) - z, 0.5f * z);
}

template <typename T, int ACT>
__global__ void activate_kernel(const T* __restrict__ x, T* __restrict__ out, size_t total,
                                float a, float b) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x)
        store_from_float(out + e, activation<ACT>(load_as_float(x + e), a, b));
}

// eight bfloat16 per thread
template <int ACT>
__global__ __launch_bounds__(256) void activate_bf16x8_kernel(const uint4* __restrict__ x,
                                                              uint4* __restrict__ out, size_t total8,
                                                              float a, float b) {
    for (size_t e = blockIdx.x * (size_t)256 + threadIdx.x; e < total8; e += (size_t)gridDim.x * 256) {
        uint4 v = x[e];
        uint32_t* w = (uint32_t*)&v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float lo = activation<ACT>(__uint_as_float(w[i] << 16), a, b);
            const float hi = activation<ACT>(__uint_as_float(w[i] & 0xffff0000u), a, b);
            w[i] = (uint32_t)float_to_bf16(lo) | ((uint32_t)float_to_bf16(hi) << 16);
        }
        out[e] = v;
    }
}

template <int ACT>
static int launch_activate(const void* x, void* out, size_t total, float a, float b, int is_bf16,
                           hipStream_t stream) {
    if (is_bf16 && total % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)out % 16) == 0) {
        const size_t n8 = total / 8;
        const int blocks = (int)((n8 + 255) / 256 < 262144 ? (n8 + 255) / 256 : 262144);
        activate_bf16x8_kernel<ACT><<<blocks, 256, 0, stream>>>((const uint4*)x, (uint4*)out, n8, a, b);
        return GFA_LAUNCH_RESULT();
    }
    const int blocks = (int)((total + 255) / 256 < 262144 ? (total + 255) / 256 : 262144);
    if (is_bf16)
        activate_kernel<bf16_t, ACT><<<blocks, 256, 0, stream>>>((const bf16_t*)x, (bf16_t*)out, total, a, b);
    else
        activate_kernel<float, ACT><<<blocks, 256, 0, stream>>>((const float*)x, (float*)out, total, a, b);
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_activate(const void* x, void* out, size_t total, int act, float a, float b,
                            int is_bf16, hipStream_t stream) {
    if (total == 0) return 0;
    if (act == 0) return launch_activate<0>(x, out, total, a, b, is_bf16, stream);
    if (act == 1) return launch_activate<1>(x, out, total, a, b, is_bf16, stream);
    if (act == 2) return launch_activate<2>(x, out, total, a, b, is_bf16, stream);
    if (act == 3) return launch_activate<3>(x, out, total, a, b, is_bf16, stream);
    return (int)hipErrorInvalidValue;
}

// --------------------------------------------------------------------------------------
// out[r, :] = [a[r, :], b[r, :]] in type T from two float matrices of dim columns each: the
// operand of a product over the stream and the embedded rows side by side.
template <typename T>
__global__ void concat_rows_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                   T* __restrict__ out, int dim) {
    const size_t r = blockIdx.x;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) {
        store_from_float(out + r * 2 * dim + d, a[r * dim + d]);
        store_from_float(out + r * 2 * dim + dim + d, b[r * dim + d]);
    }
}

extern "C" int gfa_concat_rows(const float* a, const float* b, void* out, int out_bf16, int n_rows,
                               int dim, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (out_bf16) concat_rows_kernel<bf16_t><<<n_rows, 256, 0, stream>>>(a, b, (bf16_t*)out, dim);
    else concat_rows_kernel<float><<<n_rows, 256, 0, stream>>>(a, b, (float*)out, dim);
    return GFA_LAUNCH_RESULT();
}

// res[r, :] += bias[:]
__global__ void add_bias_kernel(float* __restrict__ res, const float* __restrict__ bias, int dim) {
    const size_t r = blockIdx.x;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) res[r * dim + d] += bias[d];
}

extern "C" int gfa_add_bias(float* res, const float* bias, int n_rows, int dim, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    add_bias_kernel<<<n_rows, 256, 0, stream>>>(res, bias, dim);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// out[n, :] += float(table[idx[n], :]): rows of a table picked by an index per token, added to
// the embedded rows (a learned position vector: idx = the tokens' positions).
template <typename T>
__global__ void add_table_rows_kernel(const T* __restrict__ table, const int* __restrict__ idx,
                                      float* __restrict__ out, int dim) {
    const int n = blockIdx.x;
    const T* row = table + (size_t)idx[n] * dim;
    float* o = out + (size_t)n * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) o[d] += load_as_float(row + d);
}

extern "C" int gfa_add_table_rows(const void* table, int table_bf16, const int* idx, float* out,
                                  int n_tokens, int dim, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (table_bf16)
        add_table_rows_kernel<bf16_t><<<n_tokens, 256, 0, stream>>>((const bf16_t*)table, idx, out, dim);
    else
        add_table_rows_kernel<float><<<n_tokens, 256, 0, stream>>>((const float*)table, idx, out, dim);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// The embedding of the pair (previous token, token): out[n, :] += table[row(n), :] with
//   row = (previous * mul_prev + token * mul_cur) mod buckets       (64-bit integers)
//   row = buckets (the table's last row) for a sequence's first token.
// The previous token of the first token a step brings to a sequence is last[slot], where the
// step before left it; the workgroup of that first token reads it and then puts the
// sequence's last token of this step there (no other workgroup touches the entry).
template <typename T>
__global__ void pair_embed_add_kernel(const T* __restrict__ table, const int* __restrict__ tokens,
                                      const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
                                      const int* __restrict__ q_start, const int* __restrict__ slots,
                                      int* __restrict__ last, float* __restrict__ out, int dim,
                                      long long buckets, long long mul_prev, long long mul_cur) {
    const int n = blockIdx.x;
    const int b = tok_seq[n];
    const bool first_of_step = n == q_start[b];
    const int slot = slots[b];
    long long row = buckets;
    if (tok_pos[n] > 0) {
        const long long prev = first_of_step ? last[slot] : tokens[n - 1];
        row = (prev * mul_prev + (long long)tokens[n] * mul_cur) % buckets;
    }
    __syncthreads();                                   // every thread has read last[slot]
    if (first_of_step && threadIdx.x == 0) last[slot] = tokens[q_start[b + 1] - 1];
    const T* src = table + (size_t)row * dim;
    float* o = out + (size_t)n * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) o[d] += load_as_float(src + d);
}

extern "C" int gfa_pair_embed_add(const void* table, int table_bf16, const int* tokens,
                                  const int* tok_seq, const int* tok_pos, const int* q_start,
                                  const int* slots, int* last, float* out, int n_tokens, int dim,
                                  long long buckets, long long mul_prev, long long mul_cur,
                                  hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (buckets <= 0) return (int)hipErrorInvalidValue;
    if (table_bf16)
        pair_embed_add_kernel<bf16_t><<<n_tokens, 256, 0, stream>>>(
            (const bf16_t*)table, tokens, tok_seq, tok_pos, q_start, slots, last, out, dim, buckets,
            mul_prev, mul_cur);
    else
        pair_embed_add_kernel<float><<<n_tokens, 256, 0, stream>>>(
            (const float*)table, tokens, tok_seq, tok_pos, q_start, slots, last, out, dim, buckets,
            mul_prev, mul_cur);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// out[i, :] = T(x[r, :]), r = rows ? rows[i] : i: the float rows of the stream in the compute
// type, for a sublayer that reads the stream itself.
template <typename T>
__global__ void cast_rows_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                 T* __restrict__ out, int dim) {
    const size_t r = rows ? (size_t)rows[blockIdx.x] : (size_t)blockIdx.x;
    const float* src = x + r * dim;
    T* o = out + (size_t)blockIdx.x * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) store_from_float(o + d, src[d]);
}

extern "C" int gfa_cast_rows(const float* x, const int* rows, void* out, int out_bf16, int n_rows,
                             int dim, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (out_bf16)
        cast_rows_kernel<bf16_t><<<n_rows, 256, 0, stream>>>(x, rows, (bf16_t*)out, dim);
    else
        cast_rows_kernel<float><<<n_rows, 256, 0, stream>>>(x, rows, (float*)out, dim);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// A sublayer's result joins the stream through a gate and a norm of its own:
//   y'  = y * sigmoid(gate + gate_bias)          (gate: float sums of a projection, row stride
//                                                 gate_stride; gate null: y' = y)
//   res += y' * rsqrt(mean(y'^2) + eps_y) * wy
// and, from the same pass, what reads the stream next: next_mode 1: the RMS norm of the new
// rows with next_w and eps_n; 2: the new rows as they are; both in type T.  One workgroup per
// row of up to 256 * GN_MAX elements kept in registers; longer rows take the plain loops.
#define GN_MAX 32
template <typename T>
__global__ __launch_bounds__(256) void gated_normed_add_kernel(
        float* __restrict__ res, const float* __restrict__ y, const float* __restrict__ gate,
        long long gate_stride, const float* __restrict__ gate_bias, const float* __restrict__ wy,
        float eps_y, int next_mode, const float* __restrict__ next_w, float eps_n,
        T* __restrict__ out, int dim) {
    __shared__ float scratch[16];
    const size_t row = (size_t)blockIdx.x * dim;
    const float* yr = y + row;
    const float* gr = gate ? gate + (size_t)blockIdx.x * gate_stride : nullptr;
    float* rr = res + row;
    const bool fits = dim <= 256 * GN_MAX;
    float held[GN_MAX];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < GN_MAX; ++j) {
        const int d = threadIdx.x + 256 * j;
        float v = 0.f;
        if (fits && d < dim) {
            v = yr[d];
            if (gr) v *= 1.f / (1.f + expf(-(gr[d] + (gate_bias ? gate_bias[d] : 0.f))));
        }
        held[j] = v;
        ss = fmaf(v, v, ss);
    }
    if (!fits) {
        for (int d = threadIdx.x; d < dim; d += 256) {
            float v = yr[d];
            if (gr) v *= 1.f / (1.f + expf(-(gr[d] + (gate_bias ? gate_bias[d] : 0.f))));
            ss = fmaf(v, v, ss);
        }
    }
    ss = block_sum(ss, scratch);
    const float ry = rsqrtf(ss / (float)dim + eps_y);
    float sn = 0.f;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            if (d < dim) {
                const float v = rr[d] + held[j] * ry * wy[d];
                rr[d] = v;
                held[j] = v;
                sn = fmaf(v, v, sn);
            }
        }
    } else {
        for (int d = threadIdx.x; d < dim; d += 256) {
            float v = yr[d];
            if (gr) v *= 1.f / (1.f + expf(-(gr[d] + (gate_bias ? gate_bias[d] : 0.f))));
            v = rr[d] + v * ry * wy[d];
            rr[d] = v;
            sn = fmaf(v, v, sn);
        }
    }
    if (next_mode == 0) return;
    float rn = 1.f;
    if (next_mode == 1) {
        sn = block_sum(sn, scratch);
        rn = rsqrtf(sn / (float)dim + eps_n);
    }
    T* o = out + row;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            if (d < dim) store_from_float(o + d, next_mode == 1 ? held[j] * rn * next_w[d] : held[j]);
        }
    } else {
        // every thread reads back only what it wrote itself
        for (int d = threadIdx.x; d < dim; d += 256)
            store_from_float(o + d, next_mode == 1 ? rr[d] * rn * next_w[d] : rr[d]);
    }
}

// The same for rows of up to 1024 * VPT * 4 elements (a multiple of 4, gate rows at addresses
// that are multiples of 16): everything is read once with 16-byte loads and kept in registers
// between the sums and the stores.
template <typename T, int VPT, int THREADS>
__global__ __launch_bounds__(THREADS) void gated_normed_add_vec_kernel(
        float* __restrict__ res, const float* __restrict__ y, const float* __restrict__ gate,
        long long gate_stride, const float* __restrict__ gate_bias, const float* __restrict__ wy,
        float eps_y, int next_mode, const float* __restrict__ next_w, float eps_n,
        T* __restrict__ out, int dim) {
    __shared__ float scratch[16];
    const size_t row = (size_t)blockIdx.x * dim;
    const float4* y4 = (const float4*)(y + row);
    const float4* g4 = gate ? (const float4*)(gate + (size_t)blockIdx.x * gate_stride) : nullptr;
    const float4* b4 = (const float4*)gate_bias;
    float4* r4 = (float4*)(res + row);
    const float4* wy4 = (const float4*)wy;
    const int n4 = dim >> 2;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 yv[VPT], rv[VPT];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        const bool in = idx < n4;
        yv[j] = in ? y4[idx] : zero;
        rv[j] = in ? r4[idx] : zero;
        if (g4 && in) {
            float4 g = g4[idx];
            if (b4) {
                const float4 b = b4[idx];
                g.x += b.x; g.y += b.y; g.z += b.z; g.w += b.w;
            }
            yv[j].x *= 1.f / (1.f + expf(-g.x));
            yv[j].y *= 1.f / (1.f + expf(-g.y));
            yv[j].z *= 1.f / (1.f + expf(-g.z));
            yv[j].w *= 1.f / (1.f + expf(-g.w));
        }
        ss = fmaf(yv[j].x, yv[j].x, ss);
        ss = fmaf(yv[j].y, yv[j].y, ss);
        ss = fmaf(yv[j].z, yv[j].z, ss);
        ss = fmaf(yv[j].w, yv[j].w, ss);
    }
    ss = block_sum(ss, scratch);
    const float ry = rsqrtf(ss / (float)dim + eps_y);
    float sn = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            const float4 g = wy4[idx];
            rv[j].x += yv[j].x * ry * g.x;
            rv[j].y += yv[j].y * ry * g.y;
            rv[j].z += yv[j].z * ry * g.z;
            rv[j].w += yv[j].w * ry * g.w;
            r4[idx] = rv[j];
            sn = fmaf(rv[j].x, rv[j].x, sn);
            sn = fmaf(rv[j].y, rv[j].y, sn);
            sn = fmaf(rv[j].z, rv[j].z, sn);
            sn = fmaf(rv[j].w, rv[j].w, sn);
        }
    }
    if (next_mode == 0) return;
    float rn = 1.f;
    if (next_mode == 1) {
        sn = block_sum(sn, scratch);
        rn = rsqrtf(sn / (float)dim + eps_n);
    }
    const float4* nw4 = (const float4*)next_w;
    T* o = out + row;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            float4 v = rv[j];
            if (next_mode == 1) {
                const float4 g = nw4[idx];
                v.x *= rn * g.x; v.y *= rn * g.y; v.z *= rn * g.z; v.w *= rn * g.w;
            }
            store_from_float(o + 4 * idx + 0, v.x);
            store_from_float(o + 4 * idx + 1, v.y);
            store_from_float(o + 4 * idx + 2, v.z);
            store_from_float(o + 4 * idx + 3, v.w);
        }
    }
}

template <typename T>
static int launch_gated_normed_add(float* res, const float* y, const float* gate, long long gate_stride,
                                   const float* gate_bias, const float* wy, float eps_y, int next_mode,
                                   const float* next_w, float eps_n, T* out, int n_rows, int dim,
                                   hipStream_t stream) {
    const bool vec = dim % 4 == 0 && dim <= 8192 && (!gate || (gate_stride % 4 == 0 && (size_t)gate % 16 == 0))
        && (size_t)res % 16 == 0 && (size_t)y % 16 == 0 && (size_t)wy % 16 == 0
        && (size_t)gate_bias % 16 == 0 && (size_t)next_w % 16 == 0;
#define GFA_GN_ARGS res, y, gate, gate_stride, gate_bias, wy, eps_y, next_mode, next_w, eps_n, out, dim
    if (!vec)
        gated_normed_add_kernel<T><<<n_rows, 256, 0, stream>>>(GFA_GN_ARGS);
    else if (dim <= 1024)
        gated_normed_add_vec_kernel<T, 1, 256><<<n_rows, 256, 0, stream>>>(GFA_GN_ARGS);
    else if (dim <= 4096)
        gated_normed_add_vec_kernel<T, 1, 1024><<<n_rows, 1024, 0, stream>>>(GFA_GN_ARGS);
    else
        gated_normed_add_vec_kernel<T, 2, 1024><<<n_rows, 1024, 0, stream>>>(GFA_GN_ARGS);
#undef GFA_GN_ARGS
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_gated_normed_add(float* res, const float* y, const float* gate,
                                    long long gate_stride, const float* gate_bias, const float* wy,
                                    float eps_y, int next_mode, const float* next_w, float eps_n,
                                    void* out, int out_bf16, int n_rows, int dim,
                                    hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (next_mode < 0 || next_mode > 2 || (next_mode == 1 && !next_w) || (next_mode && !out))
        return (int)hipErrorInvalidValue;
    if (out_bf16)
        return launch_gated_normed_add<bf16_t>(res, y, gate, gate_stride, gate_bias, wy, eps_y, next_mode,
                                               next_w, eps_n, (bf16_t*)out, n_rows, dim, stream);
    return launch_gated_normed_add<float>(res, y, gate, gate_stride, gate_bias, wy, eps_y, next_mode,
                                          next_w, eps_n, (float*)out, n_rows, dim, stream);
}

// --------------------------------------------------------------------------------------
// Layer norm with a weight and, if `bias` is given, a bias:
//   out[i, :] = (x[r, :] - mean) * rsqrt(mean((x[r, :] - mean)^2) + eps) * w[:] + bias[:],  r = rows ? rows[i] : i
// The variance is the mean of the squared deviations (a second pass over the row, which a
// thread keeps in registers up to 256 * GN_MAX elements).  Float arithmetic, one rounding at
// the store.
template <typename T>
__global__ __launch_bounds__(256) void layer_norm_kernel(
        const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
        const int* __restrict__ rows, T* __restrict__ out, int dim, float eps) {
    __shared__ float scratch[16];
    const size_t r = rows ? (size_t)rows[blockIdx.x] : (size_t)blockIdx.x;
    const float* xr = x + r * dim;
    const bool fits = dim <= 256 * GN_MAX;
    float held[GN_MAX];
    float sum = 0.f;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            held[j] = d < dim ? xr[d] : 0.f;
            sum += held[j];
        }
    } else {
        for (int d = threadIdx.x; d < dim; d += 256) sum += xr[d];
    }
    const float mean = block_sum(sum, scratch) / (float)dim;
    float sq = 0.f;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            const float c = d < dim ? held[j] - mean : 0.f;
            sq = fmaf(c, c, sq);
        }
    } else {
        for (int d = threadIdx.x; d < dim; d += 256) {
            const float c = xr[d] - mean;
            sq = fmaf(c, c, sq);
        }
    }
    const float rs = rsqrtf(block_sum(sq, scratch) / (float)dim + eps);
    T* o = out + (size_t)blockIdx.x * dim;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            if (d < dim) store_from_float(o + d, (held[j] - mean) * rs * w[d] + (bias ? bias[d] : 0.f));
        }
    } else {
        for (int d = threadIdx.x; d < dim; d += 256)
            store_from_float(o + d, (xr[d] - mean) * rs * w[d] + (bias ? bias[d] : 0.f));
    }
}

extern "C" int gfa_layer_norm(const float* x, const float* w, const float* bias, const int* rows, void* out,
                              int out_bf16, int n_rows, int dim, float eps, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (out_bf16)
        layer_norm_kernel<bf16_t><<<n_rows, 256, 0, stream>>>(x, w, bias, rows, (bf16_t*)out, dim, eps);
    else
        layer_norm_kernel<float><<<n_rows, 256, 0, stream>>>(x, w, bias, rows, (float*)out, dim, eps);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// A sublayer's result joins a stream that is normed AFTER the sum:
//   y    = ya                                                   (yb null), or
//   y    = (ya rsqrt(mean(ya^2) + eps_b) wa + yb rsqrt(mean(yb^2) + eps_b) wb) / 2
//          (two branches that read the same input, each RMS-normed with a weight of its own)
//   v    = alpha * res + ls * y                                 (ls: a weight per column, or null)
//   res  = (v - mean(v)) * rsqrt(mean((v - mean(v))^2) + eps) * w
// and, from the same pass, the new rows in type T for whoever reads the stream next (out null:
// not).  One workgroup per row; a thread keeps its elements in registers up to 256 * GN_MAX
// per row, longer rows go through res (every thread reads back only what it wrote).
template <typename T>
__global__ __launch_bounds__(256) void post_norm_join_kernel(
        float* __restrict__ res, const float* __restrict__ ya, const float* __restrict__ yb,
        const float* __restrict__ wa, const float* __restrict__ wb, float eps_b,
        const float* __restrict__ ls, float alpha, const float* __restrict__ w, float eps,
        T* __restrict__ out, int dim) {
    __shared__ float scratch[16];
    const size_t row = (size_t)blockIdx.x * dim;
    float* rr = res + row;
    const float* ar = ya + row;
    const float* br = yb ? yb + row : nullptr;
    const bool fits = dim <= 256 * GN_MAX;
    float fa = 1.f, fb = 0.f;
    if (br) {
        float sa = 0.f, sb = 0.f;
        for (int d = threadIdx.x; d < dim; d += 256) {
            sa = fmaf(ar[d], ar[d], sa);
            sb = fmaf(br[d], br[d], sb);
        }
        fa = 0.5f * rsqrtf(block_sum(sa, scratch) / (float)dim + eps_b);
        fb = 0.5f * rsqrtf(block_sum(sb, scratch) / (float)dim + eps_b);
    }
    float held[GN_MAX];
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < GN_MAX; ++j) {
        const int d = threadIdx.x + 256 * j;
        float v = 0.f;
        if (fits && d < dim) {
            const float y = br ? ar[d] * fa * wa[d] + br[d] * fb * wb[d] : ar[d];
            v = fmaf(alpha, rr[d], ls ? ls[d] * y : y);
        }
        held[j] = v;
        sum += v;
    }
    if (!fits) {
        for (int d = threadIdx.x; d < dim; d += 256) {
            const float y = br ? ar[d] * fa * wa[d] + br[d] * fb * wb[d] : ar[d];
            const float v = fmaf(alpha, rr[d], ls ? ls[d] * y : y);
            rr[d] = v;
            sum += v;
        }
    }
    const float mean = block_sum(sum, scratch) / (float)dim;
    float sq = 0.f;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            const float c = d < dim ? held[j] - mean : 0.f;
            sq = fmaf(c, c, sq);
        }
    } else {
        for (int d = threadIdx.x; d < dim; d += 256) {
            const float c = rr[d] - mean;
            sq = fmaf(c, c, sq);
        }
    }
    const float rs = rsqrtf(block_sum(sq, scratch) / (float)dim + eps);
    T* o = out ? out + row : nullptr;
    if (fits) {
#pragma unroll
        for (int j = 0; j < GN_MAX; ++j) {
            const int d = threadIdx.x + 256 * j;
            if (d < dim) {
                const float v = (held[j] - mean) * rs * w[d];
                rr[d] = v;
                if (o) store_from_float(o + d, v);
            }
        }
    } else {
        for (int d = threadIdx.x; d < dim; d += 256) {
            const float v = (rr[d] - mean) * rs * w[d];
            rr[d] = v;
            if (o) store_from_float(o + d, v);
        }
    }
}

// The same for rows of up to THREADS * VPT * 4 elements (a multiple of 4, every pointer at a
// multiple of 16 bytes): everything is read once with 16-byte loads and kept in registers
// between the sums and the stores.
template <typename T, int VPT, int THREADS>
__global__ __launch_bounds__(THREADS) void post_norm_join_vec_kernel(
        float* __restrict__ res, const float* __restrict__ ya, const float* __restrict__ yb,
        const float* __restrict__ wa, const float* __restrict__ wb, float eps_b,
        const float* __restrict__ ls, float alpha, const float* __restrict__ w, float eps,
        T* __restrict__ out, int dim) {
    __shared__ float scratch[16];
    const size_t row = (size_t)blockIdx.x * dim;
    float4* r4 = (float4*)(res + row);
    const float4* a4 = (const float4*)(ya + row);
    const float4* b4 = yb ? (const float4*)(yb + row) : nullptr;
    const int n4 = dim >> 2;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[VPT], yv[VPT], zv[VPT];
    float sa = 0.f, sb = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        const bool in = idx < n4;
        v[j] = in ? r4[idx] : zero;
        yv[j] = in ? a4[idx] : zero;
        zv[j] = (in && b4) ? b4[idx] : zero;
        sa += yv[j].x * yv[j].x + yv[j].y * yv[j].y + yv[j].z * yv[j].z + yv[j].w * yv[j].w;
        sb += zv[j].x * zv[j].x + zv[j].y * zv[j].y + zv[j].z * zv[j].z + zv[j].w * zv[j].w;
    }
    float fa = 1.f, fb = 0.f;
    if (b4) {
        fa = 0.5f * rsqrtf(block_sum(sa, scratch) / (float)dim + eps_b);
        fb = 0.5f * rsqrtf(block_sum(sb, scratch) / (float)dim + eps_b);
    }
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            float4 y = yv[j];
            if (b4) {
                const float4 ga = ((const float4*)wa)[idx], gb = ((const float4*)wb)[idx];
                y.x = y.x * fa * ga.x + zv[j].x * fb * gb.x;
                y.y = y.y * fa * ga.y + zv[j].y * fb * gb.y;
                y.z = y.z * fa * ga.z + zv[j].z * fb * gb.z;
                y.w = y.w * fa * ga.w + zv[j].w * fb * gb.w;
            }
            if (ls) {
                const float4 l = ((const float4*)ls)[idx];
                y.x *= l.x; y.y *= l.y; y.z *= l.z; y.w *= l.w;
            }
            v[j].x = fmaf(alpha, v[j].x, y.x);
            v[j].y = fmaf(alpha, v[j].y, y.y);
            v[j].z = fmaf(alpha, v[j].z, y.z);
            v[j].w = fmaf(alpha, v[j].w, y.w);
            sum += v[j].x + v[j].y + v[j].z + v[j].w;
        }
    }
    const float mean = block_sum(sum, scratch) / (float)dim;
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            v[j].x -= mean; v[j].y -= mean; v[j].z -= mean; v[j].w -= mean;
            sq += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
        }
    }
    const float rs = rsqrtf(block_sum(sq, scratch) / (float)dim + eps);
    T* o = out ? out + row : nullptr;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int idx = threadIdx.x + j * THREADS;
        if (idx < n4) {
            const float4 g = ((const float4*)w)[idx];
            float4 x = v[j];
            x.x *= rs * g.x; x.y *= rs * g.y; x.z *= rs * g.z; x.w *= rs * g.w;
            r4[idx] = x;
            if (o) {
                store_from_float(o + 4 * idx + 0, x.x);
                store_from_float(o + 4 * idx + 1, x.y);
                store_from_float(o + 4 * idx + 2, x.z);
                store_from_float(o + 4 * idx + 3, x.w);
            }
        }
    }
}

template <typename T>
static int launch_post_norm_join(float* res, const float* ya, const float* yb, const float* wa,
                                 const float* wb, float eps_b, const float* ls, float alpha,
                                 const float* w, float eps, T* out, int n_rows, int dim,
                                 hipStream_t stream) {
    const bool vec = dim % 4 == 0 && dim <= 8192 && (size_t)res % 16 == 0 && (size_t)ya % 16 == 0
        && (size_t)yb % 16 == 0 && (size_t)wa % 16 == 0 && (size_t)wb % 16 == 0 && (size_t)ls % 16 == 0
        && (size_t)w % 16 == 0;
#define GFA_PJ_ARGS res, ya, yb, wa, wb, eps_b, ls, alpha, w, eps, out, dim
    if (!vec)
        post_norm_join_kernel<T><<<n_rows, 256, 0, stream>>>(GFA_PJ_ARGS);
    else if (dim <= 1024)
        post_norm_join_vec_kernel<T, 1, 256><<<n_rows, 256, 0, stream>>>(GFA_PJ_ARGS);
    else if (dim <= 4096)
        post_norm_join_vec_kernel<T, 1, 1024><<<n_rows, 1024, 0, stream>>>(GFA_PJ_ARGS);
    else
        post_norm_join_vec_kernel<T, 2, 1024><<<n_rows, 1024, 0, stream>>>(GFA_PJ_ARGS);
#undef GFA_PJ_ARGS
    return GFA_LAUNCH_RESULT();
}

extern "C" int gfa_post_norm_join(float* res, const float* ya, const float* yb, const float* wa,
                                  const float* wb, float eps_b, const float* ls, float alpha,
                                  const float* w, float eps, void* out, int out_bf16, int n_rows,
                                  int dim, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (!res || !ya || !w || (yb && (!wa || !wb))) return (int)hipErrorInvalidValue;
    if (out_bf16)
        return launch_post_norm_join<bf16_t>(res, ya, yb, wa, wb, eps_b, ls, alpha, w, eps, (bf16_t*)out,
                                             n_rows, dim, stream);
    return launch_post_norm_join<float>(res, ya, yb, wa, wb, eps_b, ls, alpha, w, eps, (float*)out,
                                        n_rows, dim, stream);
}

// --------------------------------------------------------------------------------------
// Rotation of heads that lie in float rows, in place: rows [N, row_width], H heads of hd
// elements from column `off`; the first `rot` elements of every head are turned by
// pos * freqs[i], pairs (2i, 2i + 1) (layout 0) or (i, i + rot / 2) (layout 1):
//   (u, v) -> (u c - v s, v c + u s),  c = trig * cos(a), s = trig * sin(a)
// and then EVERY element of the head is multiplied by `factor` - heads from number `late` on
// by `late_factor` instead (q and k that lie one behind the other, k with a factor of its
// own).  One thread per pair, or per element behind the rotated part; grid (tokens, heads).
__global__ void rotate_rows_kernel(float* __restrict__ x, int row_width, int off, int hd, int rot,
                                   int layout, const float* __restrict__ freqs, float trig,
                                   float factor, int late, float late_factor,
                                   const int* __restrict__ tok_pos) {
    const int n = blockIdx.x, h = blockIdx.y;
    float* head = x + (size_t)n * row_width + off + h * hd;
    const float pos = (float)tok_pos[n];
    const float f = h >= late ? late_factor : factor;
    const int half = rot >> 1;
    for (int e = threadIdx.x; e < half + (hd - rot); e += blockDim.x) {
        if (e < half) {
            const int iu = layout == 0 ? 2 * e : e, iv = layout == 0 ? 2 * e + 1 : e + half;
            float sn, cs;
            sincosf(pos * freqs[e], &sn, &cs);
            sn *= trig;
            cs *= trig;
            const float u = head[iu], v = head[iv];
            head[iu] = (u * cs - v * sn) * f;
            head[iv] = (v * cs + u * sn) * f;
        } else {
            head[rot + e - half] *= f;
        }
    }
}

extern "C" int gfa_rotate_rows(float* x, int row_width, int off, int n_heads, int hd, int rot,
                               int layout, const float* freqs, float trig, float factor, int late,
                               float late_factor, const int* tok_pos, int n_tokens, hipStream_t stream) {
    if (n_tokens <= 0 || n_heads <= 0) return 0;
    if (rot < 0 || rot > hd || rot % 2 || (rot && !freqs) || n_heads > 65535 ||
            off + n_heads * hd > row_width)
        return (int)hipErrorInvalidValue;
    rotate_rows_kernel<<<dim3(n_tokens, n_heads), 64, 0, stream>>>(x, row_width, off, hd, rot, layout,
                                                                  freqs, trig, factor, late, late_factor,
                                                                  tok_pos);
    return GFA_LAUNCH_RESULT();
}

// --------------------------------------------------------------------------------------
// The gate over float sums, rounded once: out[n, i] = pair(gu[n, i], gu[n, I + i]) as
// bfloat16, gu float [N, 2 I] (the sums of a product whose rows are the gate rows and then
// the up rows).  act as above.
template <int ACT>
__global__ void gate_mul_sums_kernel(const float* __restrict__ gu, bf16_t* __restrict__ out, int I,
                                     size_t total, float limit) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const size_t n = e / I;
        const int i = (int)(e % I);
        out[e] = float_to_bf16(gate_pair<ACT>(gu[n * 2 * I + i], gu[n * 2 * I + I + i], limit));
    }
}

extern "C" int gfa_gate_mul_sums(const float* gu, void* out, int n_rows, int I, int act, float limit,
                                 hipStream_t stream) {
    const size_t total = (size_t)n_rows * I;
    if (total == 0) return 0;
    const int blocks = (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535);
    if (act == 0) gate_mul_sums_kernel<0><<<blocks, 256, 0, stream>>>(gu, (bf16_t*)out, I, total, limit);
    else if (act == 1) gate_mul_sums_kernel<1><<<blocks, 256, 0, stream>>>(gu, (bf16_t*)out, I, total, limit);
    else if (act == 2) gate_mul_sums_kernel<2><<<blocks, 256, 0, stream>>>(gu, (bf16_t*)out, I, total, limit);
    else return (int)hipErrorInvalidValue;
    return GFA_LAUNCH_RESULT();
}

// out[n, i] = x[n * x_stride + i] for i < width, rounded to T: columns of float rows as rows of
// their own (the operand of a further product).
template <typename T>
__global__ void cast_columns_kernel(const float* __restrict__ x, long long x_stride, T* __restrict__ out,
                                    int width, size_t total) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const size_t n = e / width;
        store_from_float(out + e, x[n * x_stride + (e - n * width)]);
    }
}

extern "C" int gfa_cast_columns(const float* x, long long x_stride, void* out, int n_rows, int width,
                                int out_bf16, hipStream_t stream) {
    const size_t total = (size_t)n_rows * width;
    if (total == 0) return 0;
    const int blocks = (int)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535);
    if (out_bf16) cast_columns_kernel<bf16_t><<<blocks, 256, 0, stream>>>(x, x_stride, (bf16_t*)out, width, total);
    else cast_columns_kernel<float><<<blocks, 256, 0, stream>>>(x, x_stride, (float*)out, width, total);
    return GFA_LAUNCH_RESULT();
}

// y[n, :] *= sigmoid(g[n * g_stride]): a gate of one number per row on float rows.
__global__ void scale_rows_sigmoid_kernel(float* __restrict__ y, const float* __restrict__ g,
                                          long long g_stride, int dim) {
    const float f = 1.f / (1.f + expf(-g[(size_t)blockIdx.x * g_stride]));
    float* row = y + (size_t)blockIdx.x * dim;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) row[d] *= f;
}

extern "C" int gfa_scale_rows_sigmoid(float* y, const float* g, long long g_stride, int n_rows, int dim,
                                      hipStream_t stream) {
    if (n_rows <= 0) return 0;
    scale_rows_sigmoid_kernel<<<n_rows, 256, 0, stream>>>(y, g, g_stride, dim);
    return GFA_LAUNCH_RESULT();
}
