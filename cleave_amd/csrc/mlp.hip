// mlp.hip -- one SGD step of a 2-layer sigmoid MLP with MSE loss, in the style
// of examples/xor_tensor.cleave:38-92 (config: batch mean, no biases).
//
// Forward ops are the stdlib bodies (matmul stdlib/linalg/matrix.cleave:27-61,
// sigmoid stdlib/nn/nn.cleave:87-93, mean stdlib/nn/nn.cleave:135-138); the
// backward applies the reference's derivative rules in reverse mode:
//   MatMul product rule (stdlib/linalg/matrix.cleave:24) -> dA = dC B^T, dB = A^T dC
//   d(e*e) = de*e + e*de (stdlib/num/num.cleave:125)      -> dL/dyhat = (e+e)/B
//   sigmoid via quotient + exp rules (num.cleave:132-134, :222) -> s(1-s)
//
// Kernel sequence on the library stream (device-resident, no host sync):
//   1. X W1                             gemm_f32 NN   (M=B, N=Hd, K=D)
//   2. per row: H = sigmoid(X W1), z2 = H W2, yhat, e, e*e,
//      d2 = (e+e)/B * yhat(1-yhat), d1 = (d2 W2) h(1-h) over X W1, and
//      partial sums of h*d2 and e*e     mlp_rows_kernel (Hd > 4096: mlp_wide_rows_kernel,
//                                       mlp_cols_kernel)
//   3. dW1 = X^T d1                     gemm_f32 TN
//   4. dW2 = sum of partials; W1 -= lr dW1, W2 -= lr dW2;
//      loss = sum(e*e) / B              mlp_finish_kernel
#include <algorithm>

#include "common.hpp"
#include "gemm_f32_pingpong.hpp"

namespace ch {
int32_t gemm_f32_device(const float* a, const float* b, float* c, int M, int N, int K, int ta, int tb);
}

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float sigmoidf_ref(float x) { return 1.0f / (1.0f + expf(-x)); }

// Fused path, after the MODE-1 GEMM: z2[row] = sum of the P partials of
// H[row] . W2 (in order; loads eight at a time), then the same per-row loss
// pieces as mlp_rows_kernel.  Each block also reduces its rows' squared
// errors into sqpart[block] (wave shuffles, then the 4 wave sums in order),
// which loss_kernel adds up.
constexpr int kPartUnroll = 8;

// The P partials of row `row` of H W2, added in order (eight loads in flight).
__device__ __forceinline__ float sum_row_partials(const float* __restrict__ zpart, int P, int B, int row) {
    float z = zpart[row];
    int p = 1;
    for (; p + kPartUnroll <= P; p += kPartUnroll) {
        float v[kPartUnroll];
#pragma unroll
        for (int u = 0; u < kPartUnroll; ++u) v[u] = zpart[(int64_t)(p + u) * B + row];
#pragma unroll
        for (int u = 0; u < kPartUnroll; ++u) z += v[u];
    }
    for (; p < P; ++p) z += zpart[(int64_t)p * B + row];
    return z;
}

__global__ __launch_bounds__(kThreads) void row_finish_kernel(const float* __restrict__ zpart, int P,
                                                              const float* __restrict__ y, int B,
                                                              float* __restrict__ sqpart,
                                                              float* __restrict__ d2) {
    __shared__ float wsum[kThreads / 64];
    const int row = blockIdx.x * kThreads + threadIdx.x;
    float sq = 0.0f;
    if (row < B) {
        const float z = sum_row_partials(zpart, P, B, row);
        const float yh = sigmoidf_ref(z);
        const float e = yh - y[row];
        sq = e * e;
        const float gy = (e + e) / (float)B;
        d2[row] = gy * yh * (1.0f - yh);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = wsum[0];
        for (int w = 1; w < kThreads / 64; ++w) r += wsum[w];
        sqpart[blockIdx.x] = r;
    }
}

// The hidden layer's z = H W2 alone, from the fused GEMM's partials.
__global__ __launch_bounds__(kThreads) void z_finish_kernel(const float* __restrict__ zpart, int P, int B,
                                                            float* __restrict__ z) {
    const int row = blockIdx.x * kThreads + threadIdx.x;
    if (row < B) z[row] = sum_row_partials(zpart, P, B, row);
}

// Step 2 of the unfused path, and the hidden layer's two halves alone.  TPR threads
// own a row, E elements of it each, in registers from the load to the store, so X W1
// is read once and only d1 (or H) is written; dW2 partials stay in registers over the
// rows a thread meets, and each workgroup writes one row of them.
//   kStep  H holds X W1; v is y; writes d1 over H, dW2 and squared-error partials
//   kFwd   H holds X W1; writes H over it and z = H W2 to z
//   kBwd   H holds sigmoid(X W1), v is g = dL/dz; writes d1 to D1, dW2 partials
// 1000 x 300 took 217 us in a column pass on 4 workgroups, after 14 us in three
// launches for the sigmoid, the row products and the loss; it takes 8 us here.
enum class Rows { kStep, kFwd, kBwd };
template <int TPR, int E, bool VEC, Rows MODE>
__global__ __launch_bounds__(kThreads) void mlp_rows_kernel(float* H, float* D1, const float* __restrict__ W2,
                                                            const float* __restrict__ v, int B, int Hd,
                                                            float* __restrict__ part, float* __restrict__ sqpart,
                                                            float* __restrict__ z) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    constexpr int RL = kThreads / TPR;  // rows in flight a workgroup
    static_assert(E % 4 == 0 && (TPR == 64 || TPR == kThreads), "row shape");
    __shared__ float cross[4];
    __shared__ float red[RL > 1 ? RL * TPR * E : 1];
    const int t = threadIdx.x % TPR, rl = threadIdx.x / TPR;
    auto col = [&](int i) { return VEC ? ((i / 4) * TPR + t) * 4 + i % 4 : i * TPR + t; };
    auto load = [&](const float* __restrict__ p, float (&x)[E]) {
        if constexpr (VEC) {
#pragma unroll
            for (int i = 0; i < E; i += 4) {
                const v4 q = col(i) < Hd ? *reinterpret_cast<const v4*>(p + col(i)) : v4(0.0f);
#pragma unroll
                for (int j = 0; j < 4; ++j) x[i + j] = q[j];
            }
        } else {
#pragma unroll
            for (int i = 0; i < E; ++i) x[i] = col(i) < Hd ? p[col(i)] : 0.0f;
        }
    };
    auto store = [&](float* p, const float (&x)[E]) {
        if constexpr (VEC) {
#pragma unroll
            for (int i = 0; i < E; i += 4)
                if (col(i) < Hd) *reinterpret_cast<v4*>(p + col(i)) = v4{x[i], x[i + 1], x[i + 2], x[i + 3]};
        } else {
#pragma unroll
            for (int i = 0; i < E; ++i)
                if (col(i) < Hd) p[col(i)] = x[i];
        }
    };
    float w[E], s[E], h[E], next[E];
    load(W2, w);
#pragma unroll
    for (int i = 0; i < E; ++i) s[i] = 0.0f;
    float sq = 0.0f;
    const int step = (int)gridDim.x * RL;
    int64_t r = (int64_t)blockIdx.x * RL + rl;
    if (r < B) load(H + r * Hd, next);
    for (; r < B; r += step) {
#pragma unroll
        for (int i = 0; i < E; ++i) h[i] = next[i];
        if (r + step < B) load(H + (r + step) * Hd, next);
        float d2;
        if constexpr (MODE == Rows::kBwd) {
            d2 = v[r];
        } else {
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                h[i] = sigmoidf_ref(h[i]);
                acc += h[i] * w[i];
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
            if constexpr (TPR > 64) {
                __syncthreads();
                if ((t & 63) == 0) cross[t >> 6] = acc;
                __syncthreads();
                acc = (cross[0] + cross[1]) + (cross[2] + cross[3]);
            }
            if constexpr (MODE == Rows::kFwd) {
                if (t == 0) z[r] = acc;
                store(H + r * Hd, h);
                continue;
            }
            const float yh = sigmoidf_ref(acc);
            const float e = yh - v[r];
            sq += e * e;
            const float gy = (e + e) / (float)B;
            d2 = gy * yh * (1.0f - yh);
        }
        float d1[E];
#pragma unroll
        for (int i = 0; i < E; ++i) {
            s[i] += h[i] * d2;
            const float g = d2 * w[i];
            d1[i] = g * h[i] * (1.0f - h[i]);
        }
        store((MODE == Rows::kBwd ? D1 : H) + r * Hd, d1);
    }
    if constexpr (MODE == Rows::kFwd) return;
    // the workgroup's row of dW2 partials: its RL rows' sums in order
    if constexpr (RL > 1) {
#pragma unroll
        for (int i = 0; i < E; ++i) red[(rl * E + i) * TPR + t] = s[i];
        if (t == 0) cross[rl] = sq;
        __syncthreads();
        if (rl != 0) return;
#pragma unroll
        for (int i = 0; i < E; ++i)
#pragma unroll
            for (int q = 1; q < RL; ++q) s[i] += red[(q * E + i) * TPR + t];
        sq = ((cross[0] + cross[1]) + cross[2]) + cross[3];
    }
    store(part + (int64_t)blockIdx.x * Hd, s);
    if (MODE == Rows::kStep && t == 0) sqpart[blockIdx.x] = sq;
}

// Rows past 16 elements a thread (Hd > 4096) take two passes.  This one forms H over
// X W1 and z = H W2 a row at a time (8 workgroups a CU), and with STEP d2 and the
// workgroup's squared errors; mlp_cols_kernel reads H again.  (One pass that walked its
// row twice and added to a row of dW2 partials in memory moved those as often as H:
// the step of 65536 x 16 x 4500 took 3334 us, 1623 here, the forward layer alone 1681, 745.)
constexpr int kWideUnroll = 4;
template <bool VEC, bool STEP>
__global__ __launch_bounds__(kThreads) void mlp_wide_rows_kernel(float* H, const float* __restrict__ W2,
                                                                 const float* __restrict__ y, int B, int Hd,
                                                                 float* __restrict__ out, float* __restrict__ sqpart) {
    constexpr int V = VEC ? 4 : 1;
    typedef float vec __attribute__((ext_vector_type(V)));
    __shared__ float cross[4];
    float sq = 0.0f;
    const int n = Hd / V;  // whole vectors: VEC needs Hd % 4 == 0
    for (int64_t r = blockIdx.x; r < B; r += gridDim.x) {
        vec* h = reinterpret_cast<vec*>(H + r * Hd);
        const vec* w = reinterpret_cast<const vec*>(W2);
        float acc = 0.0f;
        for (int c0 = threadIdx.x; c0 < n; c0 += kWideUnroll * kThreads) {
            vec x[kWideUnroll];
#pragma unroll
            for (int u = 0; u < kWideUnroll; ++u)
                if (c0 + u * kThreads < n) x[u] = h[c0 + u * kThreads];
#pragma unroll
            for (int u = 0; u < kWideUnroll; ++u)
                if (c0 + u * kThreads < n) {
                    const vec q = w[c0 + u * kThreads];
#pragma unroll
                    for (int e = 0; e < V; ++e) {
                        x[u][e] = sigmoidf_ref(x[u][e]);
                        acc += x[u][e] * q[e];
                    }
                    h[c0 + u * kThreads] = x[u];
                }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
        __syncthreads();  // the last row's reads of cross
        if ((threadIdx.x & 63) == 0) cross[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            acc = (cross[0] + cross[1]) + (cross[2] + cross[3]);
            if constexpr (STEP) {
                const float yh = sigmoidf_ref(acc);
                const float e = yh - y[r];
                sq += e * e;
                const float gy = (e + e) / (float)B;
                out[r] = gy * yh * (1.0f - yh);
            } else {
                out[r] = acc;
            }
        }
    }
    if (STEP && threadIdx.x == 0) sqpart[blockIdx.x] = sq;
}

// d1 (over H, when D1 is H) and a row of dW2 partials per band of rows_per_band rows;
// a workgroup owns kWideCols columns, four a thread, and keeps their sums in registers.
constexpr int kWideCols = 4 * kThreads;
template <bool VEC>
__global__ __launch_bounds__(kThreads) void mlp_cols_kernel(const float* H, float* D1, const float* __restrict__ W2,
                                                            const float* __restrict__ d2, int B, int Hd,
                                                            int rows_per_band, float* __restrict__ part) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    const int first = blockIdx.x * kWideCols + (VEC ? 4 : 1) * threadIdx.x;
    auto col = [&](int j) { return first + (VEC ? j : j * kThreads); };
    auto load = [&](const float* p, float (&x)[4]) {
        if constexpr (VEC) {
            const v4 q = first < Hd ? *reinterpret_cast<const v4*>(p + first) : v4(0.0f);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = q[j];
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = col(j) < Hd ? p[col(j)] : 0.0f;
        }
    };
    auto store = [&](float* p, const float (&x)[4]) {
        if constexpr (VEC) {
            if (first < Hd) *reinterpret_cast<v4*>(p + first) = v4{x[0], x[1], x[2], x[3]};
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (col(j) < Hd) p[col(j)] = x[j];
        }
    };
    const int64_t r0 = (int64_t)blockIdx.y * rows_per_band;
    const int64_t r1 = r0 + rows_per_band < B ? r0 + rows_per_band : B;
    float w[4], s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    load(W2, w);
    for (int64_t r = r0; r < r1; r += kWideUnroll) {
        float h[kWideUnroll][4];
#pragma unroll
        for (int u = 0; u < kWideUnroll; ++u)
            if (r + u < r1) load(H + (r + u) * Hd, h[u]);
#pragma unroll
        for (int u = 0; u < kWideUnroll; ++u)
            if (r + u < r1) {
                const float d = d2[r + u];
                float d1[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[j] += h[u][j] * d;
                    const float g = d * w[j];
                    d1[j] = g * h[u][j] * (1.0f - h[u][j]);
                }
                store(D1 + (r + u) * Hd, d1);
            }
    }
    store(part + (int64_t)blockIdx.y * Hd, s);
}

constexpr int kRowsMaxHd = 4096;  // the widest row of mlp_rows_kernel

// Workgroups of the row passes: one row a thread group.  Up to two a CU where each
// writes a row of dW2 partials, up to eight where none does (29289 x 16 X W1 in the
// forward layer: 26.6 us, with two a CU 30.9).
int row_groups(int B, int Hd, bool partials) {
    const int lanes = Hd <= 1024 ? kThreads / 64 : 1;
    const int64_t want = ((int64_t)B + lanes - 1) / lanes, cap = (partials ? 2 : 8) * (int64_t)ch::num_cus();
    return (int)(want < cap ? want : cap);
}

// Rows of a band of mlp_cols_kernel: about four workgroups a CU over all bands.
int wide_rows_per_band(int B, int Hd) {
    const int64_t across = (Hd + kWideCols - 1) / kWideCols;
    const int64_t bands = std::max<int64_t>(1, 4 * (int64_t)ch::num_cus() / across);
    return (int)(((int64_t)B + bands - 1) / bands);
}

// Rows of dW2 partials that the passes of a B x Hd layer write.
int partial_rows(int B, int Hd) {
    if (Hd <= kRowsMaxHd) return row_groups(B, Hd, true);
    const int rows = wide_rows_per_band(B, Hd);
    return (B + rows - 1) / rows;
}

// The hidden layer's passes over H (mlp_rows_kernel, or the two above).  d2: B floats of
// workspace of the wide step; part has partial_rows(B, Hd) rows, sqpart row_groups(...).
template <Rows MODE>
int32_t run_rows(float* H, float* D1, const float* W2, const float* v, int B, int Hd, float* d2, float* part,
                 float* sqpart, float* z, hipStream_t st) {
    const bool vec = Hd % 4 == 0 && (((uintptr_t)H | (uintptr_t)D1 | (uintptr_t)W2 | (uintptr_t)part) & 15) == 0;
    if (Hd > kRowsMaxHd) {
        constexpr bool kIsStep = MODE == Rows::kStep;
        if constexpr (MODE != Rows::kBwd) {
            auto rows = [&](auto kernel) {
                kernel<<<(unsigned)row_groups(B, Hd, false), kThreads, 0, st>>>(H, W2, v, B, Hd, kIsStep ? d2 : z,
                                                                               sqpart);
            };
            vec ? rows(mlp_wide_rows_kernel<true, kIsStep>) : rows(mlp_wide_rows_kernel<false, kIsStep>);
            CH_LAUNCHED("mlp_wide_rows_kernel");
        }
        if constexpr (MODE != Rows::kFwd) {
            const dim3 grid((unsigned)((Hd + kWideCols - 1) / kWideCols), (unsigned)partial_rows(B, Hd));
            auto cols = [&](auto kernel) {
                kernel<<<grid, kThreads, 0, st>>>(H, kIsStep ? H : D1, W2, kIsStep ? d2 : v, B, Hd,
                                                 wide_rows_per_band(B, Hd), part);
            };
            vec ? cols(mlp_cols_kernel<true>) : cols(mlp_cols_kernel<false>);
            CH_LAUNCHED("mlp_cols_kernel");
        }
        return CLEAVE_HIP_OK;
    }
    const unsigned grid = (unsigned)row_groups(B, Hd, MODE != Rows::kFwd);
    auto go = [&](auto kernel) { kernel<<<grid, kThreads, 0, st>>>(H, D1, W2, v, B, Hd, part, sqpart, z); };
    if (Hd <= 256) vec ? go(mlp_rows_kernel<64, 4, true, MODE>) : go(mlp_rows_kernel<64, 4, false, MODE>);
    else if (Hd <= 512) vec ? go(mlp_rows_kernel<64, 8, true, MODE>) : go(mlp_rows_kernel<64, 8, false, MODE>);
    else if (Hd <= 1024) vec ? go(mlp_rows_kernel<64, 16, true, MODE>) : go(mlp_rows_kernel<64, 16, false, MODE>);
    else if (Hd <= 2048) vec ? go(mlp_rows_kernel<256, 8, true, MODE>) : go(mlp_rows_kernel<256, 8, false, MODE>);
    else vec ? go(mlp_rows_kernel<256, 16, true, MODE>) : go(mlp_rows_kernel<256, 16, false, MODE>);
    CH_LAUNCHED("mlp_rows_kernel");
    return CLEAVE_HIP_OK;
}

// Step 4: workgroups [0, blocks1) update W1; the next
// ceil(Hd / kFoldCols) sum the dW2 partials (kFoldLanes threads a column, each its
// run of them in order, then the runs in order) and update W2; the last one, if
// there is a loss to write, sums the squared errors.  A null dw or w is left out.
constexpr int kFoldCols = 16, kFoldLanes = kThreads / kFoldCols;
struct Finish {
    const float* g1;  // dW1
    int blocks1;
    int64_t n1;
    float* w1;
    const float* part2;  // groups x Hd
    int groups, Hd;
    float *dw2, *w2;
    const float* sqpart;  // errs
    int errs;
    float* loss;
    float count, lr;
};
unsigned finish_grid(const Finish& f) {
    return (unsigned)(f.blocks1 + (f.Hd + kFoldCols - 1) / kFoldCols + (f.loss ? 1 : 0));
}
__global__ __launch_bounds__(kThreads) void mlp_finish_kernel(Finish f) {
    auto update = [&](float g, float* dw, float* w, int64_t i) {
        if (dw) dw[i] = g;
        if (f.lr != 0.0f && w) w[i] = w[i] - f.lr * g;
    };
    if ((int)blockIdx.x < f.blocks1) {
        for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < f.n1; i += (int64_t)f.blocks1 * kThreads) {
            f.w1[i] = f.w1[i] - f.lr * f.g1[i];
        }
        return;
    }
    __shared__ float red[kThreads];
    const int fold = (f.Hd + kFoldCols - 1) / kFoldCols;
    const bool errors = (int)blockIdx.x == f.blocks1 + fold;
    // a run of partials: a column's, or the squared errors (a thread each)
    const int cols = errors ? 1 : kFoldCols, lanes = errors ? kThreads : kFoldLanes;
    const int lane = threadIdx.x / cols;
    const int c = errors ? 0 : ((int)blockIdx.x - f.blocks1) * kFoldCols + (int)threadIdx.x % cols;
    const float* p = errors ? f.sqpart : f.part2 + c;
    const int64_t pitch = errors ? 1 : f.Hd;
    const int64_t runs = errors ? f.errs : f.groups;
    const int q0 = (int)(runs * lane / lanes), q1 = (int)(runs * (lane + 1) / lanes);
    float acc = 0.0f;
    if (errors || c < f.Hd) {
        int q = q0;
        for (; q + kPartUnroll <= q1; q += kPartUnroll) {
            float x[kPartUnroll];
#pragma unroll
            for (int u = 0; u < kPartUnroll; ++u) x[u] = p[(q + u) * pitch];
#pragma unroll
            for (int u = 0; u < kPartUnroll; ++u) acc += x[u];
        }
        for (; q < q1; ++q) acc += p[q * pitch];
    }
    red[threadIdx.x] = acc;
    for (int half = lanes / 2; half > 0; half /= 2) {
        __syncthreads();
        if (lane < half) red[threadIdx.x] += red[threadIdx.x + half * cols];
    }
    if (lane != 0) return;
    if (errors) *f.loss = red[threadIdx.x] / f.count;
    else if (c < f.Hd) update(red[threadIdx.x], f.dw2, f.w2, c);
}

// out[i] = sum_s part[s*n + i] (fixed order); optional copy to dW; W -= lr * out.
__global__ __launch_bounds__(kThreads) void sum_slices_sgd_kernel(const float* __restrict__ part,
                                                                  int slices, int64_t n,
                                                                  float* __restrict__ dw,
                                                                  float* __restrict__ w, float lr) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        float g = part[i];
        int s = 1;
        for (; s + kPartUnroll <= slices; s += kPartUnroll) {  // kPartUnroll loads in flight, same order
            float v[kPartUnroll];
#pragma unroll
            for (int u = 0; u < kPartUnroll; ++u) v[u] = part[(int64_t)(s + u) * n + i];
#pragma unroll
            for (int u = 0; u < kPartUnroll; ++u) g += v[u];
        }
        for (; s < slices; ++s) g += part[(int64_t)s * n + i];
        if (dw) dw[i] = g;
        if (lr != 0.0f) w[i] = w[i] - lr * g;
    }
}

// Fused path: dW1[m][n] = w2[n] * sum_s part[s][m][n] (fixed order) -- the
// column factor of d1 = (d2 w2) h(1-h), left out of the GEMM's operand
// transform -- with an optional copy to dW, then W -= lr * dW1.  Blocks cover
// 256 columns and stride over rows.
__global__ __launch_bounds__(kThreads) void dw1_finish_kernel(const float* __restrict__ part, int slices,
                                                              int rows, int cols, const float* __restrict__ w2,
                                                              float* __restrict__ dw, float* __restrict__ w,
                                                              float lr) {
    const int c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= cols) return;
    const float f = w2[c];
    const int64_t n = (int64_t)rows * cols;
    for (int r = blockIdx.y; r < rows; r += gridDim.y) {
        const int64_t i = (int64_t)r * cols + c;
        float g = part[i];
        for (int s = 1; s < slices; ++s) g += part[(int64_t)s * n + i];
        g = f * g;
        if (dw) dw[i] = g;
        if (lr != 0.0f) w[i] = w[i] - lr * g;
    }
}

// loss = (sum of the n values v) / count: the row blocks' sums of squared errors.
__global__ __launch_bounds__(kThreads) void loss_kernel(const float* __restrict__ v, int n, float count,
                                                        float* __restrict__ loss) {
    __shared__ float part[kThreads / 64];
    float acc = 0.0f;
    // v[t], v[t + 256], ... in that order, kPartUnroll loads in flight
    int i = threadIdx.x;
    for (; i + (kPartUnroll - 1) * kThreads < n; i += kPartUnroll * kThreads) {
        float w[kPartUnroll];
#pragma unroll
        for (int u = 0; u < kPartUnroll; ++u) w[u] = v[i + u * kThreads];
#pragma unroll
        for (int u = 0; u < kPartUnroll; ++u) acc += w[u];
    }
    for (; i < n; i += kThreads) acc += v[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = 0.0f;
        for (int w = 0; w < kThreads / 64; ++w) r += part[w];
        *loss = r / count;
    }
}

unsigned capped_grid(int64_t n) {
    int64_t want = (n + kThreads - 1) / kThreads;
    int64_t cap = (int64_t)ch::num_cus() * 8;
    if (want > cap) want = cap;
    return (unsigned)(want < 1 ? 1 : want);
}

// ---- fused path (shapes that divide the 256 x 256 x 16 f32 tile) -----------
//   1. H = sigmoid(X W1) and partials of H W2      f32 ping-pong GEMM, MODE 1
//   2. z2, yhat, e, sq, d2 per row; loss           row_finish, loss kernels
//   3. slices of X^T (d1 / W2) with d1 / W2 = d2 H(1-H) formed as the MFMA
//      reads H, and dW2 partials                   f32 ping-pong GEMM, MODE 2
//   4. dW1 = W2 (column factor) * sum of slices, W1 -= lr dW1; dW2 likewise
//      (W2 is updated last: steps 3 and 4 read it)
using FusedTile1 = ch::F32PingPong<true, false, 1>;
using FusedTile2 = ch::F32PingPong<false, false, 2>;

int fused_splits(int B, int D, int Hd) {
    const int tiles = (D / 256) * (Hd / 256);
    int splits = 1;
    while (tiles * splits < ch::num_cus() && splits < 64 && B % (splits * 2 * 16) == 0) splits *= 2;
    return splits;
}

bool fused_fits(const float* x, const float* w1, int B, int D, int Hd) {
    if (B % 256 || D % 256 || Hd % 256) return false;
    if (((uintptr_t)x & 15) || ((uintptr_t)w1 & 15)) return false;  // 16-byte operand loads
    const int splits = fused_splits(B, D, Hd);
    return FusedTile1::fits(B, Hd, D, D, Hd) && FusedTile2::fits(D, Hd, B / splits, D, Hd);
}

int32_t fused_step(const float* x, const float* y, float* w1, float* w2, float* dw1, float* dw2,
                   float* loss_dev, int B, int D, int Hd, float lr, hipStream_t st) {
    const int splits = fused_splits(B, D, Hd);
    const int P = (Hd / 256) * 4;  // H W2 partials per row (tiles_n x waves along N)
    const int row_blocks = (B + kThreads - 1) / kThreads;
    // dW2 partials: one per (split, M-tile, row-half wave), see MlpFuse
    const int dw2_slices = splits * (D / 256) * 2;
    // Scratch slot 4: H | zpart | sq | d2 | dW2 partials | dW1 slices | loss.
    const size_t nH = (size_t)B * Hd, nZ = (size_t)P * B, nPart = (size_t)dw2_slices * Hd,
                 nSl = (size_t)splits * D * Hd;
    auto up = [](size_t n) { return (n + 63) & ~(size_t)63; };
    const size_t total = up(nH) + up(nZ) + up(B) + up(B) + up(nPart) + up(nSl) + 64;
    float* base = (float*)ch::scratch(4, total * sizeof(float));
    if (!base) return CLEAVE_HIP_ERR_OOM;
    float* H = base;
    float* zpart = H + up(nH);
    float* sq = zpart + up(nZ);
    float* d2 = sq + up(B);
    float* part = d2 + up(B);
    float* slices = part + up(nPart);
    float* loss_tmp = slices + up(nSl);

    ch::MlpFuse f1;
    f1.w2 = w2;
    f1.zpart = zpart;
    ch::gemm_f32_pingpong_kernel<true, false, 1>
        <<<dim3((unsigned)((B / 256) * (Hd / 256))), FusedTile1::THREADS, 0, st>>>(
            x, w1, H, B, Hd, D, D, Hd, 0, 0, 0, B / 256, Hd / 256, 1, 1, f1);
    CH_LAUNCHED("gemm_f32_pingpong_kernel(MODE 1)");
    row_finish_kernel<<<row_blocks, kThreads, 0, st>>>(zpart, P, y, B, sq, d2);
    CH_LAUNCHED("row_finish_kernel");
    // mean of the squared errors: the row blocks' sums, added in order, over B
    loss_kernel<<<1, kThreads, 0, st>>>(sq, row_blocks, (float)B, loss_dev ? loss_dev : loss_tmp);
    CH_LAUNCHED("loss_kernel");
    const int kk = B / splits;
    ch::MlpFuse f2;
    f2.d2 = d2;
    f2.dw2part = part;
    ch::gemm_f32_pingpong_kernel<false, false, 2>
        <<<dim3((unsigned)((D / 256) * (Hd / 256) * splits)), FusedTile2::THREADS, 0, st>>>(
            x, H, slices, D, Hd, kk, D, Hd, (int64_t)kk * D, (int64_t)kk * Hd, (int64_t)D * Hd, D / 256,
            Hd / 256, splits, 1, f2);
    CH_LAUNCHED("gemm_f32_pingpong_kernel(MODE 2)");
    dw1_finish_kernel<<<dim3((unsigned)((Hd + kThreads - 1) / kThreads), (unsigned)(D < 1024 ? D : 1024)),
                        kThreads, 0, st>>>(slices, splits, D, Hd, w2, dw1, w1, lr);
    CH_LAUNCHED("dw1_finish_kernel");
    sum_slices_sgd_kernel<<<capped_grid(Hd), kThreads, 0, st>>>(part, dw2_slices, Hd, dw2, w2, lr);
    CH_LAUNCHED("sum_slices_sgd_kernel(dW2)");
    return CLEAVE_HIP_OK;
}

// ---- the hidden layer alone: z = sigmoid(X W1) w2 and its reverse rule ----------
// The same kernels as the step, for a host (the reverse-mode tape) that meets
// this subgraph in a program: forward writes H and z; backward takes H and
// g = dL/dz and writes dW1 = X^T d1, dW2 = H^T g with d1 = (g w2^T) H(1-H).
bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// The product that forms dW1 reads x: a dW1 that shares memory with x is formed aside.
bool dw1_aside(const float* dw1, const float* x, int B, int D, int Hd) {
    return dw1 && ch::overlaps(dw1, sizeof(float) * (size_t)D * Hd, x, sizeof(float) * (size_t)B * D);
}

bool layer_fwd_fits(const float* x, const float* w1, const float* h, int B, int D, int Hd) {
    return B % 256 == 0 && D % 256 == 0 && Hd % 256 == 0 && aligned16(x) && aligned16(w1) && aligned16(h) &&
           FusedTile1::fits(B, Hd, D, D, Hd);
}

bool layer_bwd_fits(const float* x, const float* h, int B, int D, int Hd) {
    return B % 256 == 0 && D % 256 == 0 && Hd % 256 == 0 && aligned16(x) && aligned16(h) &&
           FusedTile2::fits(D, Hd, B / fused_splits(B, D, Hd), D, Hd);
}

int32_t hidden_fwd(const float* x, const float* w1, const float* w2, float* h, float* z, int B, int D, int Hd,
                   hipStream_t st) {
    if (layer_fwd_fits(x, w1, h, B, D, Hd)) {
        const int P = (Hd / 256) * 4;
        float* zpart = (float*)ch::scratch(4, sizeof(float) * (size_t)P * B);
        if (!zpart) return CLEAVE_HIP_ERR_OOM;
        ch::MlpFuse f1;
        f1.w2 = w2;
        f1.zpart = zpart;
        ch::gemm_f32_pingpong_kernel<true, false, 1>
            <<<dim3((unsigned)((B / 256) * (Hd / 256))), FusedTile1::THREADS, 0, st>>>(
                x, w1, h, B, Hd, D, D, Hd, 0, 0, 0, B / 256, Hd / 256, 1, 1, f1);
        CH_LAUNCHED("gemm_f32_pingpong_kernel(MODE 1)");
        z_finish_kernel<<<(B + kThreads - 1) / kThreads, kThreads, 0, st>>>(zpart, P, B, z);
        CH_LAUNCHED("z_finish_kernel");
        return CLEAVE_HIP_OK;
    }
    int32_t rc = ch::gemm_f32_device(x, w1, h, B, Hd, D, 0, 0);
    if (rc != CLEAVE_HIP_OK) return rc;
    return run_rows<Rows::kFwd>(h, nullptr, w2, nullptr, B, Hd, nullptr, nullptr, nullptr, z, st);
}

int32_t hidden_bwd(const float* x, const float* h, const float* w2, const float* g, float* dw1, float* dw2, int B,
                   int D, int Hd, hipStream_t st) {
    auto up = [](size_t n) { return (n + 63) & ~(size_t)63; };
    if (layer_bwd_fits(x, h, B, D, Hd)) {
        const int splits = fused_splits(B, D, Hd);
        const int dw2_slices = splits * (D / 256) * 2;
        const size_t nPart = (size_t)dw2_slices * Hd, nSl = (size_t)splits * D * Hd;
        float* part = (float*)ch::scratch(4, sizeof(float) * (up(nPart) + up(nSl)));
        if (!part) return CLEAVE_HIP_ERR_OOM;
        float* slices = part + up(nPart);
        const int kk = B / splits;
        ch::MlpFuse f2;
        f2.d2 = g;
        f2.dw2part = part;
        ch::gemm_f32_pingpong_kernel<false, false, 2>
            <<<dim3((unsigned)((D / 256) * (Hd / 256) * splits)), FusedTile2::THREADS, 0, st>>>(
                x, h, slices, D, Hd, kk, D, Hd, (int64_t)kk * D, (int64_t)kk * Hd, (int64_t)D * Hd, D / 256,
                Hd / 256, splits, 1, f2);
        CH_LAUNCHED("gemm_f32_pingpong_kernel(MODE 2)");
        if (dw1) {
            dw1_finish_kernel<<<dim3((unsigned)((Hd + kThreads - 1) / kThreads), (unsigned)(D < 1024 ? D : 1024)),
                                kThreads, 0, st>>>(slices, splits, D, Hd, w2, dw1, nullptr, 0.0f);
            CH_LAUNCHED("dw1_finish_kernel");
        }
        if (dw2) {
            sum_slices_sgd_kernel<<<capped_grid(Hd), kThreads, 0, st>>>(part, dw2_slices, Hd, dw2, nullptr, 0.0f);
            CH_LAUNCHED("sum_slices_sgd_kernel(dW2)");
        }
        return CLEAVE_HIP_OK;
    }
    const int groups = partial_rows(B, Hd);
    const bool aside = dw1_aside(dw1, x, B, D, Hd);
    const size_t nH = (size_t)B * Hd, nPart = (size_t)groups * Hd, nG = aside ? (size_t)D * Hd : 0;
    float* d1 = (float*)ch::scratch(4, sizeof(float) * (up(nH) + up(nPart) + up(nG)));
    if (!d1) return CLEAVE_HIP_ERR_OOM;
    float* part = d1 + up(nH);
    float* g1 = aside ? part + up(nPart) : dw1;
    int32_t rc = run_rows<Rows::kBwd>(const_cast<float*>(h), d1, w2, g, B, Hd, nullptr, part, nullptr, nullptr, st);
    if (rc != CLEAVE_HIP_OK) return rc;
    if (dw1) {
        rc = ch::gemm_f32_device(x, d1, g1, D, Hd, B, 1, 0);
        if (rc != CLEAVE_HIP_OK) return rc;
        if (aside) CH_HIP(hipMemcpyAsync(dw1, g1, sizeof(float) * nG, hipMemcpyDeviceToDevice, st));
    }
    Finish f{};
    if (dw2) f.part2 = part, f.groups = groups, f.Hd = Hd, f.dw2 = dw2;
    if (finish_grid(f) == 0) return CLEAVE_HIP_OK;
    mlp_finish_kernel<<<finish_grid(f), kThreads, 0, st>>>(f);
    CH_LAUNCHED("mlp_finish_kernel");
    return CLEAVE_HIP_OK;
}

}  // namespace

extern "C" int32_t cleave_hip_mlp_step_f32(const float* x, int64_t xlen, const float* y,
                                           int64_t ylen, float* w1, int64_t w1len, float* w2,
                                           int64_t w2len, float* dw1, int64_t dw1len, float* dw2,
                                           int64_t dw2len, float* loss_dev, int32_t B, int32_t D,
                                           int32_t Hd, float lr) {
    CH_REQUIRE(B > 0 && D > 0 && Hd > 0, "cleave_hip_mlp_step_f32: dims must be positive (B=%d D=%d Hd=%d)", B, D, Hd);
    CH_REQUIRE(xlen == (int64_t)B * D, "cleave_hip_mlp_step_f32: xlen %lld != B*D", (long long)xlen);
    CH_REQUIRE(ylen == B, "cleave_hip_mlp_step_f32: ylen %lld != B", (long long)ylen);
    CH_REQUIRE(w1len == (int64_t)D * Hd, "cleave_hip_mlp_step_f32: w1len %lld != D*Hd", (long long)w1len);
    CH_REQUIRE(w2len == Hd, "cleave_hip_mlp_step_f32: w2len %lld != Hd", (long long)w2len);
    CH_REQUIRE(!dw1 || dw1len == (int64_t)D * Hd, "cleave_hip_mlp_step_f32: dw1len %lld != D*Hd", (long long)dw1len);
    CH_REQUIRE(!dw2 || dw2len == Hd, "cleave_hip_mlp_step_f32: dw2len %lld != Hd", (long long)dw2len);
    CH_REQUIRE(x && y && w1 && w2, "cleave_hip_mlp_step_f32: null buffer");
    CH_REQUIRE(((uintptr_t)w2 & 15) == 0, "cleave_hip_mlp_step_f32: w2 must be 16-byte aligned");
    CH_INIT_OR_RETURN();
    const char* fn = "cleave_hip_mlp_step_f32";
    CH_DEVICE(fn, x, xlen * 4);
    CH_DEVICE(fn, y, ylen * 4);
    CH_DEVICE(fn, w1, w1len * 4);
    CH_DEVICE(fn, w2, w2len * 4);
    if (dw1) CH_DEVICE(fn, dw1, dw1len * 4);
    if (dw2) CH_DEVICE(fn, dw2, dw2len * 4);
    if (loss_dev) CH_DEVICE(fn, loss_dev, 4);

    hipStream_t st = ch::stream();
    if (fused_fits(x, w1, B, D, Hd)) return fused_step(x, y, w1, w2, dw1, dw2, loss_dev, B, D, Hd, lr, st);

    const bool wide = Hd > kRowsMaxHd;
    const int groups = partial_rows(B, Hd), errs = row_groups(B, Hd, !wide);
    const bool aside = dw1_aside(dw1, x, B, D, Hd);
    // Scratch slot 4: H/d1 | dW2 partials | squared errors | d2 of the wide passes | dW1 if not asked for, or aside.
    const size_t nH = (size_t)B * Hd, nPart = (size_t)groups * Hd, nD2 = wide ? B : 0;
    const size_t nG = dw1 && !aside ? 0 : (size_t)D * Hd;
    auto up = [](size_t n) { return (n + 63) & ~(size_t)63; };
    float* H = (float*)ch::scratch(4, sizeof(float) * (up(nH) + up(nPart) + up(errs) + up(nD2) + up(nG)));
    if (!H) return CLEAVE_HIP_ERR_OOM;
    float* part = H + up(nH);
    float* sq = part + up(nPart);
    float* d2 = sq + up(errs);
    float* g1 = nG == 0 ? dw1 : d2 + up(nD2);

    int32_t rc = ch::gemm_f32_device(x, w1, H, B, Hd, D, 0, 0);
    if (rc != CLEAVE_HIP_OK) return rc;
    rc = run_rows<Rows::kStep>(H, nullptr, w2, y, B, Hd, d2, part, sq, nullptr, st);
    if (rc != CLEAVE_HIP_OK) return rc;
    rc = ch::gemm_f32_device(x, H, g1, D, Hd, B, 1, 0);
    if (rc != CLEAVE_HIP_OK) return rc;
    Finish f{};
    f.g1 = g1, f.n1 = (int64_t)D * Hd, f.blocks1 = lr != 0.0f ? (int)capped_grid(f.n1) : 0;
    f.w1 = w1;
    f.part2 = part, f.groups = groups, f.Hd = Hd, f.dw2 = dw2, f.w2 = w2;
    f.sqpart = sq, f.errs = errs, f.loss = loss_dev, f.count = (float)B, f.lr = lr;
    mlp_finish_kernel<<<finish_grid(f), kThreads, 0, st>>>(f);
    CH_LAUNCHED("mlp_finish_kernel");
    if (aside) CH_HIP(hipMemcpyAsync(dw1, g1, sizeof(float) * nG, hipMemcpyDeviceToDevice, st));
    return CLEAVE_HIP_OK;
}

extern "C" int32_t cleave_hip_sigmoid_hidden_fwd_f32(const float* x, int64_t xlen, const float* w1, int64_t w1len,
                                                     const float* w2, int64_t w2len, float* h, int64_t hlen,
                                                     float* z, int64_t zlen, int32_t B, int32_t D, int32_t Hd) {
    const char* fn = "cleave_hip_sigmoid_hidden_fwd_f32";
    CH_REQUIRE(B > 0 && D > 0 && Hd > 0, "%s: dims must be positive (B=%d D=%d Hd=%d)", fn, B, D, Hd);
    CH_REQUIRE(xlen == (int64_t)B * D && w1len == (int64_t)D * Hd && w2len == Hd && hlen == (int64_t)B * Hd &&
                   zlen == B,
               "%s: lengths (%lld, %lld, %lld, %lld, %lld) do not match B=%d D=%d Hd=%d", fn, (long long)xlen,
               (long long)w1len, (long long)w2len, (long long)hlen, (long long)zlen, B, D, Hd);
    CH_REQUIRE(x && w1 && w2 && h && z, "%s: null buffer", fn);
    CH_REQUIRE(aligned16(w2) && aligned16(h), "%s: w2 and h must be 16-byte aligned", fn);
    CH_INIT_OR_RETURN();
    CH_DEVICE(fn, x, xlen * 4);
    CH_DEVICE(fn, w1, w1len * 4);
    CH_DEVICE(fn, w2, w2len * 4);
    CH_DEVICE(fn, h, hlen * 4);
    CH_DEVICE(fn, z, zlen * 4);
    return hidden_fwd(x, w1, w2, h, z, B, D, Hd, ch::stream());
}

extern "C" int32_t cleave_hip_sigmoid_hidden_bwd_f32(const float* x, int64_t xlen, const float* h, int64_t hlen,
                                                     const float* w2, int64_t w2len, const float* g, int64_t glen,
                                                     float* dw1, int64_t dw1len, float* dw2, int64_t dw2len,
                                                     int32_t B, int32_t D, int32_t Hd) {
    const char* fn = "cleave_hip_sigmoid_hidden_bwd_f32";
    CH_REQUIRE(B > 0 && D > 0 && Hd > 0, "%s: dims must be positive (B=%d D=%d Hd=%d)", fn, B, D, Hd);
    CH_REQUIRE(xlen == (int64_t)B * D && hlen == (int64_t)B * Hd && w2len == Hd && glen == B,
               "%s: lengths (%lld, %lld, %lld, %lld) do not match B=%d D=%d Hd=%d", fn, (long long)xlen,
               (long long)hlen, (long long)w2len, (long long)glen, B, D, Hd);
    CH_REQUIRE(!dw1 || dw1len == (int64_t)D * Hd, "%s: dw1len %lld != D*Hd", fn, (long long)dw1len);
    CH_REQUIRE(!dw2 || dw2len == Hd, "%s: dw2len %lld != Hd", fn, (long long)dw2len);
    CH_REQUIRE(x && h && w2 && g, "%s: null buffer", fn);
    CH_INIT_OR_RETURN();
    CH_DEVICE(fn, x, xlen * 4);
    CH_DEVICE(fn, h, hlen * 4);
    CH_DEVICE(fn, w2, w2len * 4);
    CH_DEVICE(fn, g, glen * 4);
    if (dw1) CH_DEVICE(fn, dw1, dw1len * 4);
    if (dw2) CH_DEVICE(fn, dw2, dw2len * 4);
    if (!dw1 && !dw2) return CLEAVE_HIP_OK;
    return hidden_bwd(x, h, w2, g, dw1, dw2, B, D, Hd, ch::stream());
}
