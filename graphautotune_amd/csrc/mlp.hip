// Cost model for the autotuner: a 3-layer MLP (in -> H -> H -> 1, ReLU),
// trained and evaluated on the GPU with hand-written kernels.
//
// Every matrix product runs on gfx950 BF16 matrix cores
// (v_mfma_f32_16x16x32_bf16): operands are rounded to bfloat16
// (round-to-nearest-even) as they are loaded, products accumulate in FP32.
// Master weights and Adam state stay FP32. One wavefront owns one 16x16
// output tile. Operand layout of the 16x16x32 instruction:
//   A[i][k]: lane i + 16*(k/8), element k%8
//   B[k][j]: lane j + 16*(k/8), element k%8
//   C[i][j]: lane j + 16*(i/4), element i%4
// The model only ranks kernel configs for the tuner (it replaces the
// reference's XGBoost regressor, tuning/tuning/role/modeling.py:16-162).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "handles.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace gatm {

// Rounds to nearest even (the conversion instruction of gfx950).
__device__ __forceinline__ __bf16 to_bf16(float f) { return (__bf16)f; }

// One 16 x 16 tile of A B by a wave, K in steps of 32 from 0 up. A_K: A is
// stored with k running fastest (element (i,k) at A[i lda + k]), else with i
// fastest (A[k lda + i]); B likewise (B_K: (k,j) at B[j ldb + k], else B[k ldb +
// j]). Rows, columns and k outside M, N, K count as zero. The operands of kSteps
// steps are loaded while the previous ones are multiplied: with one step at a
// time every step waited for memory, and the eight to eleven steps of a tile
// were most of a launch. (The order of the products is part of the results.)
// A step of Adam on 325 rows of 96 features: 190 us with 16 launches of simple
// tiles, 53 us with six launches of these; ms for 400 steps with kSteps 1, 2, 3,
// 4: 22.0, 21.4, 26.8, 26.7 (at most 63 loads can be outstanding).
constexpr int kSteps = 2;
template <bool A_K, bool B_K>
__device__ __forceinline__ floatx4 tile(const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb,
                                        int M, int N, int K, int tm, int tn, int lane) {
    const int i = tm * 16 + lane % 16, j = tn * 16 + lane % 16, kq = (lane / 16) * 8;
    // 16-byte loads where a row starts on 16 bytes (the same in every lane)
    const bool va = A_K && lda % 4 == 0 && ((unsigned long long)A & 15) == 0;
    const bool vb = B_K && ldb % 4 == 0 && ((unsigned long long)B & 15) == 0;
    auto load = [&](float (&v)[8], const float *X, int ld, bool k_fast, bool vec, int r, bool in, int k) {
        if (k_fast && vec && in && k + 8 <= K) {
            const float4 *q = reinterpret_cast<const float4 *>(X + (long long)r * ld + k);
            const float4 lo = q[0], hi = q[1];
            v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w;
            v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
            return;
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            v[e] = 0.f;
            if (in && k + e < K) v[e] = k_fast ? X[(long long)r * ld + k + e] : X[(long long)(k + e) * ld + r];
        }
    };
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    float av[2][kSteps][8], bv[2][kSteps][8];
    auto fetch = [&](auto buf, int k0) {
        constexpr int p = decltype(buf)::value;
#pragma unroll
        for (int u = 0; u < kSteps; u++) {
            if (k0 + 32 * u >= K) break;
            load(av[p][u], A, lda, A_K, va, i, i < M, k0 + 32 * u + kq);
            load(bv[p][u], B, ldb, B_K, vb, j, j < N, k0 + 32 * u + kq);
        }
    };
    auto multiply = [&](auto buf, int k0) {
        constexpr int p = decltype(buf)::value;
#pragma unroll
        for (int u = 0; u < kSteps; u++) {
            if (k0 + 32 * u >= K) break;
            bf16x8 a, b;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                a[e] = to_bf16(av[p][u][e]);
                b[e] = to_bf16(bv[p][u][e]);
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    constexpr int group = 32 * kSteps;
    fetch(even, 0);
    for (int k0 = 0; k0 < K; k0 += 2 * group) {
        fetch(odd, k0 + group);
        multiply(even, k0);
        fetch(even, k0 + 2 * group);
        multiply(odd, k0 + group);
    }
    return acc;
}

// Calls put(row, column, value) for the elements of a tile this lane holds.
template <class F>
__device__ __forceinline__ void each(floatx4 acc, int M, int N, int tm, int tn, int lane, F put) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int r = tm * 16 + (lane / 16) * 4 + e, c = tn * 16 + lane % 16;
        if (r < M && c < N) put(r, c, acc[e]);
    }
}
__host__ __device__ constexpr int tiles(int n) { return (n + 15) / 16; }

// C = A B + bias, with optional ReLU: a forward layer (A: rows x K, B: K x N).
// Given targets t, also the gradient of the loss by the outputs, 2 (C - t) / M.
__global__ void __launch_bounds__(256) layer(const float *A, const float *B, float *C, int M, int N, int K,
                                             const float *bias, int relu, const float *t, float *dy) {
    const int lane = threadIdx.x % 64, wave = (blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int tm = wave / tiles(N), tn = wave % tiles(N);
    if (tm * 16 >= M) return;  // whole wave exits together
    const floatx4 acc = tile<true, false>(A, K, B, N, M, N, K, tm, tn, lane);
    each(acc, M, N, tm, tn, lane, [&](int r, int c, float v) {
        v += bias[c];
        if (relu) v = v > 0.f ? v : 0.f;
        C[(long long)r * N + c] = v;
        if (t) {
            const float e = v - t[(long long)r * N + c];
            dy[(long long)r * N + c] = 2.f * e / M;
        }
    });
}

// Mean squared error of y against t, by 256 threads.
__device__ __forceinline__ void mse(const float *y, const float *t, int B, float *loss) {
    __shared__ float part[256];
    float s = 0.f;
    for (int r = threadIdx.x; r < B; r += blockDim.x) {
        const float e = y[r] - t[r];
        s += e * e;
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = part[0] / B;
}

// put(c, sum over r of d[r][c]), rows in order, for columns [c0, c0 + 16), by a
// workgroup of 256 threads: it stages 256 rows at a time in LDS, and one
// thread per column adds them up.
template <class F>
__device__ __forceinline__ void col_sum(const float *d, int rows, int cols, int c0, F put) {
    __shared__ float buf[256][17];
    const int c = threadIdx.x % 16, r1 = threadIdx.x / 16;
    float s = 0.f;
    for (int r0 = 0; r0 < rows; r0 += 256) {
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const int r = r0 + u * 16 + r1;
            if (r < rows && c0 + c < cols) buf[u * 16 + r1][c] = d[(long long)r * cols + c0 + c];
        }
        __syncthreads();
        const int n = rows - r0 < 256 ? rows - r0 : 256;
        if (threadIdx.x < 16 && c0 + c < cols) {
            // 32 reads in flight, then their additions one after the other
            int r = 0;
            for (; r + 32 <= n; r += 32) {
                float v[32];
#pragma unroll
                for (int u = 0; u < 32; u++) v[u] = buf[r + u][c];
#pragma unroll
                for (int u = 0; u < 32; u++) s += v[u];
            }
            for (; r < n; r++) s += buf[r][c];
        }
        __syncthreads();
    }
    if (threadIdx.x < 16 && c0 + c < cols) put(c0 + c, s);
}

struct Adam {
    float *p, *m, *v;  // parameters and state; p null: gradients only
    float lr, b1, b2, eps, c1, c2;
};
// Parameter t, whose gradient is gt.
__device__ __forceinline__ void adam(const Adam &o, long long t, float gt) {
    o.m[t] = o.b1 * o.m[t] + (1.f - o.b1) * gt;
    o.v[t] = o.b2 * o.v[t] + (1.f - o.b2) * gt * gt;
    o.p[t] -= o.lr * (o.m[t] / o.c1) / (sqrtf(o.v[t] / o.c2) + o.eps);
}

// Backward of one layer with rows x n_out pre-activation gradients d and inputs
// a (rows x n_in): the workgroups of one launch share out
//   gW = a^T d (n_in x n_out), gb = column sums of d, and, given W, d_in = (d
//   W^T) where act > 0 (the ReLU of the layer below),
// which do not depend on each other; put_w(i, c, v) and put_b(c, v) take the
// gradients. Returns the workgroup's number past these.
__host__ __device__ constexpr int backward_blocks(int rows, int n_in, int n_out, bool has_w) {
    return (tiles(n_in) * tiles(n_out) + 3) / 4 + (has_w ? (tiles(rows) * tiles(n_in) + 3) / 4 : 0) + tiles(n_out);
}
template <class FW, class FB>
__device__ __forceinline__ void backward_layer(const float *a, const float *d, const float *W, const float *act, float *d_in,
                                               int rows, int n_in, int n_out, FW put_w, FB put_b) {
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int t_w = tiles(n_in) * tiles(n_out), b_w = (t_w + 3) / 4;
    const int t_d = W ? tiles(rows) * tiles(n_in) : 0, b_d = (t_d + 3) / 4;
    int b = blockIdx.x;
    if (b < b_d) {
        const int k = b * 4 + w, tm = k / tiles(n_in), tn = k % tiles(n_in);
        if (k >= t_d) return;
        const floatx4 acc = tile<true, true>(d, n_out, W, n_out, rows, n_in, n_out, tm, tn, lane);
        each(acc, rows, n_in, tm, tn, lane, [&](int r, int c, float v) {
            const long long x = (long long)r * n_in + c;
            d_in[x] = act[x] > 0.f ? v : 0.f;
        });
    } else if ((b -= b_d) < b_w) {
        const int k = b * 4 + w, tm = k / tiles(n_out), tn = k % tiles(n_out);
        if (k >= t_w) return;
        const floatx4 acc = tile<false, false>(a, n_in, d, n_out, n_in, n_out, rows, tm, tn, lane);
        each(acc, n_in, n_out, tm, tn, lane, put_w);
    } else if ((b -= b_w) < tiles(n_out)) {
        col_sum(d, rows, n_out, b * 16, put_b);
    }
}

// The backward launches. One of them replaces four (product, sums, product,
// mask) of 12 us each; the output layer's also adds up the loss (its last
// workgroup), the first layer's applies Adam to
// its own gradients as they arise and, in further workgroups, to the others.
__global__ void __launch_bounds__(256) backward_output(const float *a2, const float *y, const float *t, const float *dy,
                                                       const float *W3, float *gW3, float *gb3, float *d2, float *loss, int B, int H) {
    if (blockIdx.x == gridDim.x - 1) {
        mse(y, t, B, loss);
        return;
    }
    backward_layer(a2, dy, W3, a2, d2, B, H, 1, [&](int r, int, float v) { gW3[r] = v; },
                   [&](int, float v) { gb3[0] = v; });
}
__global__ void __launch_bounds__(256) backward_hidden(const float *a1, const float *d2, const float *W2, float *gW2,
                                                       float *gb2, float *d1, int B, int H) {
    backward_layer(a1, d2, W2, a1, d1, B, H, H, [&](int r, int c, float v) { gW2[(long long)r * H + c] = v; },
                   [&](int c, float v) { gb2[c] = v; });
}
// g: all gradients; those of the first layer (W1, then b1) come first.
__global__ void __launch_bounds__(256) backward_input(const float *x, const float *d1, float *g, long long P, int B,
                                                      int F, int H, Adam o) {
    const int own = backward_blocks(B, F, H, false);
    if ((int)blockIdx.x >= own) {
        const long long step = (long long)(gridDim.x - own) * blockDim.x;
        for (long long t = (long long)F * H + H + (blockIdx.x - own) * (long long)blockDim.x + threadIdx.x; t < P; t += step)
            adam(o, t, g[t]);
        return;
    }
    auto put = [&](long long t, float v) {
        g[t] = v;
        if (o.p) adam(o, t, v);
    };
    backward_layer(x, d1, nullptr, nullptr, nullptr, B, F, H, [&](int r, int c, float v) { put((long long)r * H + c, v); },
                   [&](int c, float v) { put((long long)F * H + c, v); });
}

}  // namespace gatm

struct gat_mlp {
    int F = 0, H = 0;
    long long P = 0;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    int cap = 0;  // batch capacity of the activation buffers
    float *x = nullptr, *t = nullptr, *a1 = nullptr, *a2 = nullptr, *y = nullptr;
    float *dy = nullptr, *d2 = nullptr, *d1 = nullptr, *loss = nullptr;
    long long step = 0;
    hipStream_t s = nullptr;
    // parameter views
    float *W1() { return p; }
    float *b1() { return p + (long long)F * H; }
    float *W2() { return b1() + H; }
    float *b2() { return W2() + (long long)H * H; }
    float *W3() { return b2() + H; }
    float *b3() { return W3() + H; }
    float *gW1() { return g; }
    float *gb1() { return g + (long long)F * H; }
    float *gW2() { return gb1() + H; }
    float *gb2() { return gW2() + (long long)H * H; }
    float *gW3() { return gb2() + H; }
    float *gb3() { return gW3() + H; }
};

using namespace gat;

#define MCHECK(x)                                                                                   \
    do {                                                                                            \
        hipError_t e_ = (x);                                                                        \
        if (e_ != hipSuccess) GAT_FAIL(GAT_ENODEV, "%s failed: %s", #x, hipGetErrorString(e_));     \
    } while (0)

// Device memory, if need be what counts can do without.
template <class T>
static hipError_t mlp_malloc(T **p, size_t bytes) {
    for (bool again = false;; again = true) {
        const hipError_t e = hipMalloc((void **)p, bytes);
        if (e == hipSuccess) return e;
        *p = nullptr;
        (void)hipGetLastError();  // the runtime keeps an error until it is asked for
        if (again || e != hipErrorOutOfMemory || !give_back_memory()) return e;
    }
}

static int ensure_batch(gat_mlp *n, int B) {
    if (B <= n->cap) return GAT_OK;
    for (float **q : {&n->x, &n->t, &n->a1, &n->a2, &n->y, &n->dy, &n->d2, &n->d1})
        if (*q) (void)hipFree(*q), *q = nullptr;
    n->cap = 0;
    const int c = ((B + 63) / 64) * 64;
    MCHECK(mlp_malloc(&n->x, sizeof(float) * (size_t)c * n->F));
    MCHECK(mlp_malloc(&n->t, sizeof(float) * c));
    for (float **q : {&n->a1, &n->a2, &n->d2, &n->d1})
        MCHECK(mlp_malloc(q, sizeof(float) * (size_t)c * n->H));
    MCHECK(mlp_malloc(&n->y, sizeof(float) * c));
    MCHECK(mlp_malloc(&n->dy, sizeof(float) * c));
    n->cap = c;
    return GAT_OK;
}

static void run_layer(gat_mlp *n, const float *A, const float *W, const float *bias, float *C, int M, int N, int K,
                      int relu, const float *t = nullptr, float *dy = nullptr) {
    const long long waves = (long long)gatm::tiles(M) * gatm::tiles(N);
    hipLaunchKernelGGL(gatm::layer, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, n->s, A, W, C, M, N, K, bias,
                       relu, t, dy);
}

// With train also the gradient of the loss by the outputs (n->dy).
static int forward(gat_mlp *n, int B, bool train) {
    const int F = n->F, H = n->H;
    run_layer(n, n->x, n->W1(), n->b1(), n->a1, B, H, F, 1);
    run_layer(n, n->a1, n->W2(), n->b2(), n->a2, B, H, H, 1);
    run_layer(n, n->a2, n->W3(), n->b3(), n->y, B, 1, H, 0, train ? n->t : nullptr, n->dy);
    MCHECK(hipGetLastError());
    return GAT_OK;
}

static int backward(gat_mlp *n, int B, const gatm::Adam &o) {
    const int F = n->F, H = n->H;
    hipStream_t s = n->s;
    hipLaunchKernelGGL(gatm::backward_output, dim3(gatm::backward_blocks(B, H, 1, true) + 1), dim3(256), 0, s, n->a2,
                       n->y, n->t, n->dy, n->W3(), n->gW3(), n->gb3(), n->d2, n->loss, B, H);
    hipLaunchKernelGGL(gatm::backward_hidden, dim3(gatm::backward_blocks(B, H, H, true)), dim3(256), 0, s, n->a1,
                       n->d2, n->W2(), n->gW2(), n->gb2(), n->d1, B, H);
    const long long others = n->P - ((long long)F * H + H);
    const int update = o.p ? (int)std::min<long long>((others + 255) / 256, 1024) : 0;
    hipLaunchKernelGGL(gatm::backward_input, dim3(gatm::backward_blocks(B, F, H, false) + update), dim3(256), 0, s,
                       n->x, n->d1, n->g, n->P, B, F, H, o);
    MCHECK(hipGetLastError());
    return GAT_OK;
}

static int upload(gat_mlp *n, const float *x, const float *t, int B) {
    int rc = ensure_batch(n, B);
    if (rc) return rc;
    MCHECK(hipMemcpyAsync(n->x, x, sizeof(float) * (size_t)B * n->F, hipMemcpyHostToDevice, n->s));
    if (t) MCHECK(hipMemcpyAsync(n->t, t, sizeof(float) * B, hipMemcpyHostToDevice, n->s));
    return GAT_OK;
}

extern "C" {

int gat_mlp_create(int32_t in_dim, int32_t hidden, uint64_t seed, gat_mlp **out) {
    if (!out || in_dim < 1 || hidden < 1 || in_dim > 4096 || hidden > 4096) GAT_FAIL(GAT_EINVAL, "bad MLP shape");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) GAT_FAIL(GAT_ENODEV, "no HIP device visible");
    auto *n = new gat_mlp();
    n->F = in_dim;
    n->H = hidden;
    n->P = (long long)in_dim * hidden + hidden + (long long)hidden * hidden + hidden + hidden + 1;
    // He-uniform init from a seeded stream
    std::vector<float> h(n->P, 0.f);
    Rng r(seed);
    auto fill = [&](long long off, long long cnt, int fan_in) {
        const double lim = std::sqrt(6.0 / fan_in);
        for (long long k = 0; k < cnt; k++) h[off + k] = (float)((r.uniform() * 2 - 1) * lim);
    };
    fill(0, (long long)in_dim * hidden, in_dim);
    fill((long long)in_dim * hidden + hidden, (long long)hidden * hidden, hidden);
    fill((long long)in_dim * hidden + hidden + (long long)hidden * hidden + hidden, hidden, hidden);
    hipError_t e = hipStreamCreateWithFlags(&n->s, hipStreamNonBlocking);
    for (float **q : {&n->p, &n->g, &n->m, &n->v})
        if (e == hipSuccess) e = mlp_malloc(q, sizeof(float) * n->P);
    if (e == hipSuccess) e = mlp_malloc(&n->loss, sizeof(float));
    if (e == hipSuccess) e = hipMemcpy(n->p, h.data(), sizeof(float) * n->P, hipMemcpyHostToDevice);
    std::vector<float> z(n->P, 0.f);
    if (e == hipSuccess) e = hipMemcpy(n->m, z.data(), sizeof(float) * n->P, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(n->v, z.data(), sizeof(float) * n->P, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        set_error("MLP allocation failed: %s", hipGetErrorString(e));
        delete n;
        return GAT_ENODEV;
    }
    *out = n;
    return GAT_OK;
}

int gat_mlp_param_count(const gat_mlp *n, int64_t *out) {
    if (!n || !out) GAT_FAIL(GAT_EINVAL, "null argument");
    *out = n->P;
    return GAT_OK;
}

int gat_mlp_get_params(gat_mlp *n, float *out, int64_t count) {
    if (!n || !out || count != n->P) GAT_FAIL(GAT_EINVAL, "parameter buffer must hold %lld floats", n ? n->P : 0);
    MCHECK(hipMemcpy(out, n->p, sizeof(float) * n->P, hipMemcpyDeviceToHost));
    return GAT_OK;
}

int gat_mlp_set_params(gat_mlp *n, const float *in, int64_t count) {
    if (!n || !in || count != n->P) GAT_FAIL(GAT_EINVAL, "parameter buffer must hold %lld floats", n ? n->P : 0);
    MCHECK(hipMemcpy(n->p, in, sizeof(float) * n->P, hipMemcpyHostToDevice));
    return GAT_OK;
}

int gat_mlp_forward(gat_mlp *n, const float *x, int32_t batch, float *y_out) {
    if (!n || !x || !y_out || batch < 1) GAT_FAIL(GAT_EINVAL, "bad forward arguments");
    int rc = upload(n, x, nullptr, batch);
    if (!rc) rc = forward(n, batch, false);
    if (rc) return rc;
    MCHECK(hipMemcpyAsync(y_out, n->y, sizeof(float) * batch, hipMemcpyDeviceToHost, n->s));
    MCHECK(hipStreamSynchronize(n->s));
    return GAT_OK;
}

int gat_mlp_gradients(gat_mlp *n, const float *x, const float *t, int32_t batch, float *grads_out, float *loss_out) {
    if (!n || !x || !t || batch < 1) GAT_FAIL(GAT_EINVAL, "bad gradient arguments");
    int rc = upload(n, x, t, batch);
    if (!rc) rc = forward(n, batch, true);
    if (!rc) rc = backward(n, batch, gatm::Adam{});
    if (rc) return rc;
    if (grads_out) MCHECK(hipMemcpyAsync(grads_out, n->g, sizeof(float) * n->P, hipMemcpyDeviceToHost, n->s));
    if (loss_out) MCHECK(hipMemcpyAsync(loss_out, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->s));
    MCHECK(hipStreamSynchronize(n->s));
    return GAT_OK;
}

int gat_mlp_train(gat_mlp *n, const float *x, const float *t, int32_t batch, int32_t steps, float lr,
                  float *loss_out) {
    if (!n || !x || !t || batch < 1 || steps < 1 || !(lr > 0)) GAT_FAIL(GAT_EINVAL, "bad training arguments");
    int rc = upload(n, x, t, batch);
    if (rc) return rc;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int k = 0; k < steps; k++) {
        n->step++;
        const float c1 = 1.f - std::pow(b1, (float)n->step), c2 = 1.f - std::pow(b2, (float)n->step);
        rc = forward(n, batch, true);
        if (!rc) rc = backward(n, batch, gatm::Adam{n->p, n->m, n->v, lr, b1, b2, eps, c1, c2});
        if (rc) return rc;
    }
    if (loss_out) MCHECK(hipMemcpyAsync(loss_out, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->s));
    MCHECK(hipStreamSynchronize(n->s));
    return GAT_OK;
}

void gat_mlp_free(gat_mlp *n) {
    if (!n) return;
    for (float *q : {n->p, n->g, n->m, n->v, n->loss, n->x, n->t, n->a1, n->a2, n->y, n->dy, n->d2, n->d1})
        if (q) (void)hipFree(q);
    if (n->s) (void)hipStreamDestroy(n->s);
    delete n;
}

}  // extern "C"
