/*
 * The closure network (include/lbm_amd_closure.h) on gfx950: 87 -> 64 -> 64 -> 3 with SiLU, trained and evaluated by
 * FP16 MFMA kernels with FP32 accumulation.
 *
 * Wave layout of v_mfma_f32_16x16x16_f16 (64 lanes; lane l, row = l % 16, quad = 4 (l / 16)):
 *   A operand (M x K):  lane holds A[row][quad .. quad + 3]
 *   B operand (K x N):  lane holds B[quad .. quad + 3][row]
 *   C / D     (M x N):  lane holds D[quad .. quad + 3][row]
 * The network runs transposed, Z^T = W^T X^T, with the 16 particles of a tile as N: the D tile of a layer's outputs
 * 16t .. 16t + 15 is then, element for element, the B operand of the next layer's K step t, so activations stay in
 * registers from the input to the output; the weights are A operands held in registers by every wave for the whole
 * kernel.  Backward, dH^T = W dZ^T has the same property.  Per tile of 16 particles: 24 + 16 + 4 MFMAs forward,
 * 4 + 16 more backward.
 *
 * Training (lbm_mlp_train): per minibatch, mlpTrainForward (forward, error, backward through the activations; writes the
 * FP16 activations and errors transposed, 256 particles to a chunk) and mlpGradUpdate (dW = P^T Q, one 16 x 16 tile of one
 * matrix per work-group and one chunk per wave; the chunks summed in a fixed order, Adam on the FP32 master parameters, new
 * FP16 operands).  Every sum has a fixed order: training is reproducible run to run.
 */
#include "lbm_mlp.h"
#include <algorithm>
#include <cmath>
#include <mutex>
#include <numeric>
#include <random>
#include <sstream>
#include <stdexcept>

namespace lbm {
void setLastError(const std::string& message);
}

using namespace lbm;

namespace {

constexpr int WAVES = 4;                 // waves per work-group of the network kernels
constexpr int CHUNK = 256;               // particles per partial sum of the weight gradients
constexpr int GRAD_JOBS = 24 + 16 + 4;   // 16 x 16 tiles of dW1, dW2, dW3
constexpr int GRAD_WAVES = 8;            // chunks that a work-group of the weight gradients takes at a time
// Chunks up to which one work-group per tile takes them all and updates the parameters (minibatches of up to 8,192 rows).
constexpr int GRAD_ONE_LAUNCH = 32;

__device__ __forceinline__ float dsiluf(float z) {
    float s = 1.0f/(1.0f + __expf(-z));
    return s*(1.0f + z*(1.0f - s));
}

struct ForwardWeights {
    half4_t w1[4][6], w2[4][4], w3[4];
    float4_t b1[4], b2[4], b3;
};

__device__ __forceinline__ void loadForward(const MlpDevice* __restrict__ m, int row, int quad, ForwardWeights& w) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
        for (int s = 0; s < 6; s++)
            w.w1[t][s] = load4(m->w1t + (16*t + row)*MLP_IN_PAD + 16*s + quad);
#pragma unroll
        for (int s = 0; s < 4; s++)
            w.w2[t][s] = load4(m->w2t + (16*t + row)*MLP_H + 16*s + quad);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            w.b1[t][r] = m->b1[16*t + quad + r];
            w.b2[t][r] = m->b2[16*t + quad + r];
        }
    }
#pragma unroll
    for (int s = 0; s < 4; s++)
        w.w3[s] = load4(m->w3t + row*MLP_H + 16*s + quad);
#pragma unroll
    for (int r = 0; r < 4; r++)
        w.b3[r] = m->b3[quad + r];
}

struct Activations {
    float4_t z1[4], z2[4], y;
    half4_t h1[4], h2[4];
};

/* The forward pass of one tile: x[s] is the B operand of input columns 16s .. 16s + 15. */
__device__ __forceinline__ void forwardTile(const ForwardWeights& w, const half4_t x[6], Activations& a) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
        float4_t acc = w.b1[t];
#pragma unroll
        for (int s = 0; s < 6; s++)
            acc = mfma16(w.w1[t][s], x[s], acc);
        a.z1[t] = acc;
#pragma unroll
        for (int r = 0; r < 4; r++)
            a.h1[t][r] = (_Float16) siluf(acc[r]);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        float4_t acc = w.b2[t];
#pragma unroll
        for (int s = 0; s < 4; s++)
            acc = mfma16(w.w2[t][s], a.h1[s], acc);
        a.z2[t] = acc;
#pragma unroll
        for (int r = 0; r < 4; r++)
            a.h2[t][r] = (_Float16) siluf(acc[r]);
    }
    float4_t acc = w.b3;
#pragma unroll
    for (int s = 0; s < 4; s++)
        acc = mfma16(w.w3[s], a.h2[s], acc);
    a.y = acc;
}

/* Inference: persistent waves, each loading the weights once and looping over tiles of 16 particles. */
__global__ void __launch_bounds__(64*WAVES) mlpInfer(const MlpDevice* __restrict__ m, const _Float16* __restrict__ X,
        int n, float outInv, float* __restrict__ du) {
    int lane = threadIdx.x & 63;
    int wave = blockIdx.x*WAVES + (threadIdx.x >> 6);
    int waves = gridDim.x*WAVES;
    int tiles = (n + 15)/16;
    if (wave >= tiles)
        return;
    int row = lane & 15, quad = (lane >> 4)*4;
    ForwardWeights w;
    loadForward(m, row, quad, w);
    for (int tile = wave; tile < tiles; tile += waves) {
        int b = tile*16 + row;
        bool valid = b < n;
        half4_t x[6];
#pragma unroll
        for (int s = 0; s < 6; s++)
            x[s] = valid ? load4(X + (size_t) b*MLP_IN_PAD + 16*s + quad) : half4_t{0, 0, 0, 0};
        Activations a;
        forwardTile(w, x, a);
        if (lane < 16 && valid)
            for (int r = 0; r < MLP_OUT; r++)
                du[3*(size_t) b + r] = a.y[r]*outInv;
    }
}

/*
 * The layer inputs P and errors Q of a minibatch, as the weight gradients read them: per chunk of CHUNK rows, [unit][row] in
 * FP16, so that the four consecutive rows of an MFMA operand are one 8-byte load.
 */
struct TrainActivations {
    _Float16 *X, *H1, *H2, *dZ1, *dZ2, *dY;
};

/* Elements (unit 16t + quad + r, this row) of a tile -> out[chunk][unit][row]. */
__device__ __forceinline__ void storeTransposed(_Float16* out, int units, int b, int t, int quad, half4_t v) {
    _Float16* p = out + ((size_t) (b/CHUNK)*units + 16*t + quad)*CHUNK + b % CHUNK;
#pragma unroll
    for (int r = 0; r < 4; r++)
        p[r*CHUNK] = v[r];
}

/*
 * Training, forward and backward through the activations, one work-group of four waves per tile of 16 rows of the
 * minibatch (rows[b] is the dataset row of minibatch row b; rows at or beyond count are padding and get zero errors): wave
 * t computes units 16t .. 16t + 15 of every layer, and the waves exchange their tiles, which are the next layer's B
 * operands as they are, through LDS.  Stores X, H1, H2 (post-activation), dZ1, dZ2 (errors at the pre-activations) and
 * dY = (2/3)(y - t); the loss sum goes to lossSum (a diagnostic).  A minibatch of 2,048 rows is 128 tiles: bound by the
 * latency of one tile's chain (64 divisions and exponentials per lane with one wave per tile), 11.5 us with one wave per
 * tile, 7.3 us with four.
 */
__global__ void __launch_bounds__(64*WAVES) mlpTrainForward(const MlpDevice* __restrict__ m,
        const _Float16* __restrict__ X, const float* __restrict__ T, const int* __restrict__ rows, int count,
        TrainActivations act, double* __restrict__ lossSum) {
    static_assert(WAVES == 4 && MLP_H == 64, "one wave per 16 hidden units");
    __shared__ half4_t shared[3][WAVES][64];
    const int lane = threadIdx.x & 63, t = threadIdx.x >> 6;
    const int row = lane & 15, quad = (lane >> 4)*4;
    const int b = blockIdx.x*16 + row;
    const bool valid = b < count;
    const int src = rows[b];
    half4_t x[6], w1[6], w2[4], w3[4], w2n[4];
    float4_t z1, z2, y;
#pragma unroll
    for (int s = 0; s < 6; s++) {
        x[s] = load4(X + (size_t) src*MLP_IN_PAD + 16*s + quad);
        w1[s] = load4(m->w1t + (16*t + row)*MLP_IN_PAD + 16*s + quad);
    }
#pragma unroll
    for (int s = 0; s < 4; s++) {
        w2[s] = load4(m->w2t + (16*t + row)*MLP_H + 16*s + quad);
        w3[s] = load4(m->w3t + row*MLP_H + 16*s + quad);
        w2n[s] = load4(m->w2 + (16*t + row)*MLP_H + 16*s + quad);
    }
    const half4_t w3n = load4(m->w3 + (16*t + row)*MLP_OUT_PAD + quad);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        z1[r] = m->b1[16*t + quad + r];
        z2[r] = m->b2[16*t + quad + r];
        y[r] = m->b3[quad + r];
    }
    // Forward (the sums of forwardTile).
    half4_t h1, h2, dz1, dz2;
#pragma unroll
    for (int s = 0; s < 6; s++)
        z1 = mfma16(w1[s], x[s], z1);
#pragma unroll
    for (int r = 0; r < 4; r++)
        h1[r] = toHalf(siluf(z1[r]));
    shared[0][t][lane] = h1;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; s++)
        z2 = mfma16(w2[s], shared[0][s][lane], z2);
#pragma unroll
    for (int r = 0; r < 4; r++)
        h2[r] = toHalf(siluf(z2[r]));
    shared[1][t][lane] = h2;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; s++)
        y = mfma16(w3[s], shared[1][s][lane], y);
    // Output error (lanes 0-15 hold outputs 0-3 of their row; output 3 and up are padding).
    float4_t dy = {0, 0, 0, 0};
    float e = 0;
    if (quad == 0 && valid)
        for (int r = 0; r < MLP_OUT; r++) {
            float d = y[r] - T[3*(size_t) src + r];
            dy[r] = (2.0f/3.0f)*d;
            e += d*d;
        }
    half4_t dyb;
#pragma unroll
    for (int r = 0; r < 4; r++)
        dyb[r] = toHalf(dy[r]);
    // Backward: dH2^T = W3 dY^T, dZ2 = dH2 silu'(Z2), dH1^T = W2 dZ2^T, dZ1 = dH1 silu'(Z1).
    float4_t acc = mfma16(w3n, dyb, float4_t{0, 0, 0, 0});
#pragma unroll
    for (int r = 0; r < 4; r++)
        dz2[r] = toHalf(acc[r]*dsiluf(z2[r]));
    shared[2][t][lane] = dz2;
    __syncthreads();
    acc = float4_t{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++)
        acc = mfma16(w2n[s], shared[2][s][lane], acc);
#pragma unroll
    for (int r = 0; r < 4; r++)
        dz1[r] = toHalf(acc[r]*dsiluf(z1[r]));
    storeTransposed(act.H1, MLP_H, b, t, quad, h1);
    storeTransposed(act.H2, MLP_H, b, t, quad, h2);
    storeTransposed(act.dZ1, MLP_H, b, t, quad, dz1);
    storeTransposed(act.dZ2, MLP_H, b, t, quad, dz2);
#pragma unroll
    for (int s = 0; s < 6; s++)
        if (s % WAVES == t)
            storeTransposed(act.X, MLP_IN_PAD, b, s, quad, x[s]);
    if (t != WAVES - 1)
        return;
    storeTransposed(act.dY, MLP_OUT_PAD, b, 0, quad, dyb);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
        e += __shfl_xor(e, off);
    if (lane == 0)
        atomicAdd(lossSum, (double) e/3.0);
}

/* The FP16 operands and FP32 biases of parameter p. */
__device__ __forceinline__ void storeOperand(MlpDevice* d, int p, float w) {
    _Float16 h = (_Float16) w;
    if (p < MLP_OFF_B1) {
        int i = p/MLP_H, o = p % MLP_H;
        d->w1t[o*MLP_IN_PAD + i] = h;
    }
    else if (p < MLP_OFF_W2)
        d->b1[p - MLP_OFF_B1] = w;
    else if (p < MLP_OFF_B2) {
        int q = p - MLP_OFF_W2, i = q/MLP_H, o = q % MLP_H;
        d->w2t[o*MLP_H + i] = h;
        d->w2[i*MLP_H + o] = h;
    }
    else if (p < MLP_OFF_W3)
        d->b2[p - MLP_OFF_B2] = w;
    else if (p < MLP_OFF_B3) {
        int q = p - MLP_OFF_W3, i = q/MLP_OUT_PAD, o = q % MLP_OUT_PAD;
        d->w3t[o*MLP_H + i] = h;
        d->w3[i*MLP_OUT_PAD + o] = h;
    }
    else
        d->b3[p - MLP_OFF_B3] = w;
}

__global__ void mlpPack(const float* __restrict__ master, MlpDevice* __restrict__ d) {
    int p = blockIdx.x*blockDim.x + threadIdx.x;
    if (p < MLP_PARAMS)
        storeOperand(d, p, master[p]);
}

/* The gradient g (summed over the chunks) of parameter p / count; with apply, one Adam step (beta 0.9, 0.999, eps 1e-8; c1,
   c2 the bias corrections 1/(1 - beta^t)) and the new FP16 operands. */
struct UpdateArgs {
    float *master, *m1, *m2;
    float invCount, lr, c1, c2;
    MlpDevice* dev;
    float* gradOut;
    int apply;
};

__device__ __forceinline__ void updateParameter(const UpdateArgs& u, int p, float g) {
    g *= u.invCount;
    if (u.gradOut)
        u.gradOut[p] = g;
    if (!u.apply)
        return;
    float mm = 0.9f*u.m1[p] + 0.1f*g;
    float vv = 0.999f*u.m2[p] + 0.001f*g*g;
    u.m1[p] = mm;
    u.m2[p] = vv;
    float w = u.master[p] - u.lr*(mm*u.c1)/(sqrtf(vv*u.c2) + 1e-8f);
    u.master[p] = w;
    storeOperand(u.dev, p, w);
}

/*
 * Weight gradients and update, one work-group per 16 x 16 tile of dW = P^T Q (P the layer input X, H1, H2; Q the layer error
 * dZ1, dZ2, dY): wave w forms the tile over the 256 rows of chunk w, w + GRAD_WAVES, ..., and for the first row tile the bias
 * gradient (column sums of Q); the chunks are summed in their order and the parameters updated (updateParameter), which
 * nothing else in this launch reads.  All loads of a chunk are in flight at once (their latency is what bounds it): with a
 * minibatch of 2,048 rows 10.5 us, where partial sums from 8 two-byte gathers per MFMA took 24.1 us and their sum and update
 * 4.8 us in a launch of its own.  Many chunks (above GRAD_ONE_LAUNCH) take blockIdx.y work-groups per tile, each of which
 * leaves its chunks' tiles in partials[chunk][parameter] for mlpUpdate.
 */
__global__ void __launch_bounds__(64*GRAD_WAVES) mlpGradUpdate(TrainActivations act, int chunks, UpdateArgs u,
        float* __restrict__ partials) {
    __shared__ float part[GRAD_WAVES][256 + 16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, job = blockIdx.x;
    const int row = lane & 15, quad = (lane >> 4)*4;
    const _Float16 *P, *Q;
    int pw, qw, ti, to, offW, offB, width;
    if (job < 24) {
        P = act.X; pw = MLP_IN_PAD; Q = act.dZ1; qw = MLP_H; ti = job/4; to = job % 4;
        offW = MLP_OFF_W1; offB = MLP_OFF_B1; width = MLP_H;
    }
    else if (job < 40) {
        P = act.H1; pw = MLP_H; Q = act.dZ2; qw = MLP_H; ti = (job - 24)/4; to = (job - 24) % 4;
        offW = MLP_OFF_W2; offB = MLP_OFF_B2; width = MLP_H;
    }
    else {
        P = act.H2; pw = MLP_H; Q = act.dY; qw = MLP_OUT_PAD; ti = job - 40; to = 0;
        offW = MLP_OFF_W3; offB = MLP_OFF_B3; width = MLP_OUT_PAD;
    }
    // The sum over the chunks: thread p < 256 of weight (16 ti + p/16, 16 to + p % 16), thread 256 + o of bias 16 to + o.
    const int p = threadIdx.x;
    int index = -1;
    if (p < 256)
        index = offW + (16*ti + p/16)*width + 16*to + p % 16;
    else if (p < 256 + 16 && ti == 0)
        index = offB + 16*to + p - 256;
    float g = 0;
    for (int first = (int) blockIdx.y*GRAD_WAVES; first < chunks; first += (int) gridDim.y*GRAD_WAVES) {
        const int chunk = first + wave;
        if (chunk < chunks) {
            const _Float16* pt = P + ((size_t) chunk*pw + 16*ti + row)*CHUNK + quad;
            const _Float16* qt = Q + ((size_t) chunk*qw + 16*to + row)*CHUNK + quad;
            half4_t pa[CHUNK/16], qb[CHUNK/16];
#pragma unroll
            for (int k = 0; k < CHUNK/16; k++) {
                pa[k] = load4(pt + 16*k);
                qb[k] = load4(qt + 16*k);
            }
            float4_t acc = {0, 0, 0, 0};
            float bsum = 0;
#pragma unroll
            for (int k = 0; k < CHUNK/16; k++) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    bsum += (float) qb[k][e];
                acc = mfma16(pa[k], qb[k], acc);
            }
#pragma unroll
            for (int r = 0; r < 4; r++)
                part[wave][16*(quad + r) + row] = acc[r];
            bsum += __shfl_xor(bsum, 16);
            bsum += __shfl_xor(bsum, 32);
            if (lane < 16)
                part[wave][256 + lane] = bsum;
        }
        __syncthreads();
        if (index >= 0)
            for (int w = 0; w < GRAD_WAVES && first + w < chunks; w++) {
                if (partials != nullptr)
                    partials[(size_t) (first + w)*MLP_PARAMS + index] = part[w][p];
                g += part[w][p];
            }
        __syncthreads();
    }
    if (index >= 0 && partials == nullptr)
        updateParameter(u, index, g);
}

/* The chunks' partial sums in their order, and the update. */
__global__ void mlpUpdate(const float* __restrict__ partials, int chunks, UpdateArgs u) {
    int p = blockIdx.x*blockDim.x + threadIdx.x;
    if (p >= MLP_PARAMS)
        return;
    float g = 0;
    for (int c = 0; c < chunks; c++)
        g += partials[(size_t) c*MLP_PARAMS + p];
    updateParameter(u, p, g);
}

/* Raw pairs -> normalized FP16 inputs [n][96] and normalized FP32 targets [n][3]. */
__global__ void mlpNormalize(const float* __restrict__ raw, const float* __restrict__ rawTargets, int64_t n,
        ClosureNorm norm, _Float16* __restrict__ X, float* __restrict__ T) {
    int64_t idx = (int64_t) blockIdx.x*blockDim.x + threadIdx.x;
    if (idx < n*MLP_IN_PAD) {
        int64_t b = idx/MLP_IN_PAD;
        int c = (int) (idx - b*MLP_IN_PAD);
        float v = 0;
        if (c < 3)
            v = raw[b*MLP_IN + c];
        else if (c < 84)
            v = raw[b*MLP_IN + c]*norm.uScale;
        else if (c < MLP_IN)
            v = raw[b*MLP_IN + c]*norm.vScale;
        X[idx] = (_Float16) v;
    }
    if (rawTargets != nullptr && idx < n*MLP_OUT)
        T[idx] = rawTargets[idx]*norm.outScale;
}

struct MlpError : public std::runtime_error {
    int status;
    MlpError(int s, const std::string& msg) : std::runtime_error(msg), status(s) {}
};

void hipCheck(hipError_t e, const char* what) {
    if (e != hipSuccess)
        throw MlpError(LBM_ERROR_RUNTIME, std::string(what) + ": " + hipGetErrorString(e));
}

template <typename T>
T* deviceAlloc(size_t count) {
    void* p = nullptr;
    hipCheck(hipMalloc(&p, std::max<size_t>(count, 1)*sizeof(T)), "hipMalloc");
    return (T*) p;
}

unsigned blocksFor(int64_t n, int threads) {
    return (unsigned) ((n + threads - 1)/threads);
}

}  // namespace

/*
 * The device working memory of lbm_mlp_forward_noalloc: raw inputs, normalized FP16 inputs and outputs of up to
 * LBM_MLP_NOALLOC_MAX_ROWS rows (9.0 MB), one copy per GPU for the life of the process.  Every call on a GPU shares
 * that GPU's copy; nothing in it has to start at zero (each call writes every element it reads).
 */
namespace {
constexpr size_t NOALLOC_RAW_BYTES = (size_t) LBM_MLP_NOALLOC_MAX_ROWS*MLP_IN*sizeof(float);
constexpr size_t NOALLOC_X_BYTES = (size_t) LBM_MLP_NOALLOC_MAX_ROWS*MLP_IN_PAD*sizeof(_Float16);
constexpr size_t NOALLOC_OUT_BYTES = (size_t) LBM_MLP_NOALLOC_MAX_ROWS*MLP_OUT*sizeof(float);
static_assert(NOALLOC_RAW_BYTES % 256 == 0 && NOALLOC_X_BYTES % 256 == 0, "256-byte aligned parts");
}  // namespace

static __device__ __align__(256) unsigned char scratch[NOALLOC_RAW_BYTES + NOALLOC_X_BYTES + NOALLOC_OUT_BYTES];

namespace {
std::mutex scratchMutex;
std::vector<void*> scratchByDevice;

/* The device address of `scratch` on the current device (the host-side name is only a stand-in), looked up once per
   device with that device current. */
void* scratchOnCurrentDevice() {
    int device = 0;
    hipCheck(hipGetDevice(&device), "hipGetDevice");
    std::lock_guard<std::mutex> lock(scratchMutex);
    if ((int) scratchByDevice.size() <= device)
        scratchByDevice.resize(device + 1, nullptr);
    if (scratchByDevice[device] == nullptr) {
        void* ptr = nullptr;
        hipCheck(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        scratchByDevice[device] = ptr;
    }
    return scratchByDevice[device];
}
}  // namespace

struct lbm_mlp {
    hipStream_t stream = nullptr;
    void* scratch = nullptr;          // this GPU's no-allocation working memory (scratchOnCurrentDevice)
    MlpDevice* dev = nullptr;
    float* master = nullptr;
    float* mom1 = nullptr;
    float* mom2 = nullptr;
    lbm_mlp_normalization norm{1.0, 1.0, 1.0, 1e30, 1e30};
    int64_t adamStep = 0;
};

namespace lbm {

const MlpDevice* mlpDeviceWeights(const lbm_mlp* mlp) {
    return mlp->dev;
}

ClosureNorm mlpClosureNorm(const lbm_mlp* mlp) {
    ClosureNorm n;
    n.uScale = (float) mlp->norm.u_scale;
    n.vScale = (float) mlp->norm.v_scale;
    n.outScale = (float) mlp->norm.out_scale;
    n.uBound = (float) std::min(mlp->norm.u_bound, 1e30);
    n.vBound = (float) std::min(mlp->norm.v_bound, 1e30);
    return n;
}

void launchMlpInfer(const MlpDevice* weights, const _Float16* X, int n, float outScale, float* du, hipStream_t stream) {
    if (n <= 0)
        return;
    int tiles = (n + 15)/16;
    // Persistent waves, one per SIMD of the 256 compute units: each loads the weights once.
    int waves = std::min(tiles, 1024);
    mlpInfer<<<blocksFor(waves, WAVES), 64*WAVES, 0, stream>>>(weights, X, n, 1.0f/outScale, du);
}

}  // namespace lbm

namespace {

/* Minibatch buffers of the training kernels, for up to `rows` rows (a multiple of CHUNK). */
struct TrainBuffers {
    _Float16* halves = nullptr;
    TrainActivations act{};
    float* partials = nullptr;        // above GRAD_ONE_LAUNCH chunks
    double* loss = nullptr;
    void allocate(int rows) {
        const size_t n = (size_t) rows;
        halves = deviceAlloc<_Float16>(n*(MLP_IN_PAD + 4*MLP_H + MLP_OUT_PAD));
        act.X = halves;
        act.H1 = act.X + n*MLP_IN_PAD;
        act.H2 = act.H1 + n*MLP_H;
        act.dZ1 = act.H2 + n*MLP_H;
        act.dZ2 = act.dZ1 + n*MLP_H;
        act.dY = act.dZ2 + n*MLP_H;
        if (rows/CHUNK > GRAD_ONE_LAUNCH)
            partials = deviceAlloc<float>((size_t) (rows/CHUNK)*MLP_PARAMS);
        loss = deviceAlloc<double>(1);
    }
    ~TrainBuffers() {
        if (halves)
            (void) hipFree(halves);
        if (partials)
            (void) hipFree(partials);
        if (loss)
            (void) hipFree(loss);
    }
};

/*
 * Sums of squares and largest magnitudes of raw pairs, FP64, per work-group: partials[block] = {fluid velocities (columns 3 to
 * 83), bead velocity (84 to 86), targets; largest of the first, of the second}.  A fixed grid and order, so a run is
 * reproducible.  Read at the rate of the memory; the host, which summed one value after the other, took 10 of the 17 ms of
 * training 200,000 pairs for two epochs.
 */
constexpr int STAT_BLOCKS = 512, STAT_THREADS = 256, STATS = 5;
__global__ void __launch_bounds__(STAT_THREADS) pairStatistics(const float* __restrict__ features,
        const float* __restrict__ targets, int64_t n, double* __restrict__ partials) {
    constexpr int STRIDE = STAT_BLOCKS*STAT_THREADS;
    double v[STATS] = {0, 0, 0, 0, 0};
    const int64_t first = (int64_t) blockIdx.x*STAT_THREADS + threadIdx.x;
    int column = (int) (first % MLP_IN);
    for (int64_t i = first; i < n*MLP_IN; i += STRIDE) {
        const double f = (double) features[i];
        if (column >= 84) {
            v[1] += f*f;
            v[4] = fmax(v[4], fabs(f));
        }
        else if (column >= 3) {
            v[0] += f*f;
            v[3] = fmax(v[3], fabs(f));
        }
        column += STRIDE % MLP_IN;
        column -= column >= MLP_IN ? MLP_IN : 0;
    }
    for (int64_t i = first; i < n*MLP_OUT; i += STRIDE) {
        const double t = (double) targets[i];
        v[2] += t*t;
    }
    __shared__ double waves[STAT_THREADS/64][STATS];
    for (int k = 0; k < STATS; k++) {
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_xor(v[k], off, 64);
            v[k] = k < 3 ? v[k] + o : fmax(v[k], o);
        }
        if ((threadIdx.x & 63) == 0)
            waves[threadIdx.x/64][k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < STATS) {
        const int k = (int) threadIdx.x;
        double r = waves[0][k];
        for (int w = 1; w < STAT_THREADS/64; w++)
            r = k < 3 ? r + waves[w][k] : fmax(r, waves[w][k]);
        partials[STATS*blockIdx.x + k] = r;
    }
}

/* Scales and bounds from raw pairs on the device: inverse RMS of the fluid velocities, of the bead velocity and of the
   targets; bounds = largest normalized magnitude of each group. */
lbm_mlp_normalization normalizationOf(const float* features, const float* targets, int64_t n, hipStream_t stream) {
    double* partials = deviceAlloc<double>(STATS*STAT_BLOCKS);
    std::vector<double> host(STATS*STAT_BLOCKS);
    pairStatistics<<<STAT_BLOCKS, STAT_THREADS, 0, stream>>>(features, targets, n, partials);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(host.data(), partials, host.size()*sizeof(double), hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess)
        e = hipStreamSynchronize(stream);
    (void) hipFree(partials);
    hipCheck(e, "normalization");
    double su = 0, sv = 0, st = 0, mu = 0, mv = 0;
    for (int b = 0; b < STAT_BLOCKS; b++) {
        su += host[STATS*b];
        sv += host[STATS*b + 1];
        st += host[STATS*b + 2];
        mu = std::max(mu, host[STATS*b + 3]);
        mv = std::max(mv, host[STATS*b + 4]);
    }
    lbm_mlp_normalization norm;
    double ru = std::sqrt(su/(81.0*n)), rv = std::sqrt(sv/(3.0*n)), rt = std::sqrt(st/(3.0*n));
    norm.u_scale = ru > 0 ? 1.0/ru : 1.0;
    norm.v_scale = rv > 0 ? 1.0/rv : 1.0;
    norm.out_scale = rt > 0 ? 1.0/rt : 1.0;
    norm.u_bound = mu*norm.u_scale;
    norm.v_bound = mv*norm.v_scale;
    return norm;
}

/* Dataset on the device: normalized inputs and targets. */
struct Dataset {
    int64_t n = 0;
    _Float16* X = nullptr;
    float* T = nullptr;
    /* setNorm: the network's normalization becomes that of these pairs. */
    Dataset(lbm_mlp* m, const float* features, const float* targets, int64_t count, bool setNorm = false) : n(count) {
        float* raw = deviceAlloc<float>((size_t) n*MLP_IN);
        float* rawT = targets ? deviceAlloc<float>((size_t) n*MLP_OUT) : nullptr;
        X = deviceAlloc<_Float16>((size_t) n*MLP_IN_PAD);
        T = deviceAlloc<float>((size_t) n*MLP_OUT);
        hipError_t e = hipMemcpyAsync(raw, features, (size_t) n*MLP_IN*sizeof(float), hipMemcpyHostToDevice, m->stream);
        if (e == hipSuccess && rawT)
            e = hipMemcpyAsync(rawT, targets, (size_t) n*MLP_OUT*sizeof(float), hipMemcpyHostToDevice, m->stream);
        std::string failure = "dataset upload";
        if (e == hipSuccess && setNorm) {
            try {
                m->norm = normalizationOf(raw, rawT, n, m->stream);
            }
            catch (const MlpError& error) {
                e = hipErrorUnknown;
                failure = error.what();
            }
        }
        if (e == hipSuccess) {
            mlpNormalize<<<blocksFor(n*MLP_IN_PAD, 256), 256, 0, m->stream>>>(raw, rawT, n, mlpClosureNorm(m), X, T);
            e = hipStreamSynchronize(m->stream);
        }
        (void) hipStreamSynchronize(m->stream);
        (void) hipFree(raw);
        if (rawT)
            (void) hipFree(rawT);
        if (e != hipSuccess) {
            (void) hipFree(X);
            (void) hipFree(T);
            X = nullptr;
            T = nullptr;
            hipCheck(e, failure.c_str());
        }
    }
    ~Dataset() {
        if (X)
            (void) hipFree(X);
        if (T)
            (void) hipFree(T);
    }
};

/* One minibatch: rows[0 .. count) of the dataset (rows padded with valid indices to a multiple of CHUNK). */
void minibatch(lbm_mlp* m, const Dataset& data, const int* rows, int count, TrainBuffers& buf, bool apply, float lr,
        float* gradOut) {
    int chunks = (count + CHUNK - 1)/CHUNK;
    mlpTrainForward<<<chunks*(CHUNK/16), 64*WAVES, 0, m->stream>>>(m->dev, data.X, data.T, rows, count, buf.act, buf.loss);
    float c1 = 1.0f, c2 = 1.0f;
    if (apply) {
        m->adamStep++;
        c1 = (float) (1.0/(1.0 - std::pow(0.9, (double) m->adamStep)));
        c2 = (float) (1.0/(1.0 - std::pow(0.999, (double) m->adamStep)));
    }
    const UpdateArgs u = {m->master, m->mom1, m->mom2, 1.0f/count, lr, c1, c2, m->dev, gradOut, apply ? 1 : 0};
    const bool split = chunks > GRAD_ONE_LAUNCH;
    const unsigned groups = split ? blocksFor(chunks, GRAD_WAVES) : 1u;
    mlpGradUpdate<<<dim3(GRAD_JOBS, groups), 64*GRAD_WAVES, 0, m->stream>>>(buf.act, chunks, u, split ? buf.partials : nullptr);
    if (split)
        mlpUpdate<<<blocksFor(MLP_PARAMS, 256), 256, 0, m->stream>>>(buf.partials, chunks, u);
    hipCheck(hipGetLastError(), "training launch");
}

int failMlp(const std::exception& e, int status) {
    setLastError(e.what());
    return status;
}

void destroyMlp(lbm_mlp* m) {
    if (m->stream)
        (void) hipStreamSynchronize(m->stream);
    void* all[] = {m->dev, m->master, m->mom1, m->mom2};
    for (void* p : all)
        if (p)
            (void) hipFree(p);
    if (m->stream)
        (void) hipStreamDestroy(m->stream);
    delete m;
}

void uploadParameters(lbm_mlp* m, const float* params) {
    hipCheck(hipMemcpyAsync(m->master, params, MLP_PARAMS*sizeof(float), hipMemcpyHostToDevice, m->stream), "upload");
    hipCheck(hipMemsetAsync(m->mom1, 0, MLP_PARAMS*sizeof(float), m->stream), "memset");
    hipCheck(hipMemsetAsync(m->mom2, 0, MLP_PARAMS*sizeof(float), m->stream), "memset");
    mlpPack<<<blocksFor(MLP_PARAMS, 256), 256, 0, m->stream>>>(m->master, m->dev);
    hipCheck(hipGetLastError(), "pack");
    hipCheck(hipStreamSynchronize(m->stream), "sync");
    m->adamStep = 0;
}

/* The padding entries of a parameter vector must be zero (they multiply padded inputs or feed padded outputs). */
void checkPadding(const float* params) {
    for (int i = MLP_IN; i < MLP_IN_PAD; i++)
        for (int o = 0; o < MLP_H; o++)
            if (params[MLP_OFF_W1 + i*MLP_H + o] != 0.0f)
                throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_set_parameters: rows 87-95 of W1 (input padding) must be zero");
    for (int i = 0; i < MLP_H; i++)
        for (int o = MLP_OUT; o < MLP_OUT_PAD; o++)
            if (params[MLP_OFF_W3 + i*MLP_OUT_PAD + o] != 0.0f)
                throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_set_parameters: columns 3-15 of W3 (output padding) must be zero");
    for (int o = MLP_OUT; o < MLP_OUT_PAD; o++)
        if (params[MLP_OFF_B3 + o] != 0.0f)
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_set_parameters: entries 3-15 of b3 (output padding) must be zero");
}

}  // namespace

#define MLP_TRY(...) \
    try { __VA_ARGS__; setLastError(""); return LBM_OK; } \
    catch (const MlpError& e) { return failMlp(e, e.status); } \
    catch (const std::exception& e) { return failMlp(e, LBM_ERROR_RUNTIME); }

extern "C" {

int lbm_mlp_create(uint64_t seed, lbm_mlp** out) {
    if (!out) {
        setLastError("lbm_mlp_create: null argument");
        return LBM_ERROR_INVALID;
    }
    lbm_mlp* m = new lbm_mlp();
    try {
        hipCheck(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "stream");
        m->scratch = scratchOnCurrentDevice();
        m->dev = deviceAlloc<MlpDevice>(1);
        m->master = deviceAlloc<float>(MLP_PARAMS);
        m->mom1 = deviceAlloc<float>(MLP_PARAMS);
        m->mom2 = deviceAlloc<float>(MLP_PARAMS);
        std::vector<float> p(MLP_PARAMS, 0.0f);
        std::mt19937_64 rng(seed);
        std::normal_distribution<double> normal(0.0, 1.0);
        for (int i = 0; i < MLP_IN; i++)
            for (int o = 0; o < MLP_H; o++)
                p[MLP_OFF_W1 + i*MLP_H + o] = (float) (normal(rng)/std::sqrt((double) MLP_IN));
        for (int i = 0; i < MLP_H; i++)
            for (int o = 0; o < MLP_H; o++)
                p[MLP_OFF_W2 + i*MLP_H + o] = (float) (normal(rng)/std::sqrt((double) MLP_H));
        for (int i = 0; i < MLP_H; i++)
            for (int o = 0; o < MLP_OUT; o++)
                p[MLP_OFF_W3 + i*MLP_OUT_PAD + o] = (float) (normal(rng)/std::sqrt((double) MLP_H));
        hipCheck(hipMemsetAsync(m->dev, 0, sizeof(MlpDevice), m->stream), "memset");
        uploadParameters(m, p.data());
    }
    catch (const MlpError& e) {
        destroyMlp(m);
        return failMlp(e, e.status);
    }
    catch (const std::exception& e) {
        destroyMlp(m);
        return failMlp(e, LBM_ERROR_RUNTIME);
    }
    *out = m;
    setLastError("");
    return LBM_OK;
}

int lbm_mlp_destroy(lbm_mlp* m) {
    if (m)
        destroyMlp(m);
    return LBM_OK;
}

int lbm_mlp_get_parameters(lbm_mlp* m, float* params, size_t count) {
    MLP_TRY({
        if (count != (size_t) MLP_PARAMS)
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_get_parameters: count must be LBM_MLP_NUM_PARAMS");
        hipCheck(hipStreamSynchronize(m->stream), "sync");
        hipCheck(hipMemcpy(params, m->master, MLP_PARAMS*sizeof(float), hipMemcpyDeviceToHost), "download");
    })
}

int lbm_mlp_set_parameters(lbm_mlp* m, const float* params, size_t count) {
    MLP_TRY({
        if (count != (size_t) MLP_PARAMS)
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_set_parameters: count must be LBM_MLP_NUM_PARAMS");
        checkPadding(params);
        uploadParameters(m, params);
    })
}

int lbm_mlp_get_normalization(lbm_mlp* m, lbm_mlp_normalization* norm) {
    MLP_TRY(*norm = m->norm)
}

int lbm_mlp_set_normalization(lbm_mlp* m, const lbm_mlp_normalization* norm) {
    MLP_TRY({
        if (!(norm->u_scale > 0 && norm->v_scale > 0 && norm->out_scale > 0) || !(norm->u_bound >= 0 && norm->v_bound >= 0))
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_set_normalization: scales must be positive and bounds non-negative");
        m->norm = *norm;
    })
}

int lbm_mlp_train(lbm_mlp* m, const float* features, const float* targets, int64_t n, int epochs, int batch,
        double lr, double decay, uint64_t seed, double* epochLoss) {
    MLP_TRY({
        if (n <= 0 || n > (int64_t) 0x7FFFFFFF - (1 << 20) || epochs <= 0 || batch < 16 || batch > (1 << 20) || !(lr > 0))
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_train: invalid n, epochs, batch or learning rate");
        Dataset data(m, features, targets, n, true);
        int padded = (batch + CHUNK - 1)/CHUNK*CHUNK;
        TrainBuffers buf;
        buf.allocate(padded);
        int* order = deviceAlloc<int>((size_t) n + padded);
        // The rows' order of an epoch, drawn while the device works on the one before.
        std::vector<int> orders[2] = {std::vector<int>((size_t) n + padded, 0), std::vector<int>((size_t) n + padded, 0)};
        std::mt19937_64 rng(seed);
        auto shuffled = [&](int epoch) {
            std::vector<int>& perm = orders[epoch & 1];
            std::iota(perm.begin(), perm.begin() + n, 0);
            std::shuffle(perm.begin(), perm.begin() + n, rng);
        };
        shuffled(0);
        try {
            for (int epoch = 0; epoch < epochs; epoch++) {
                const std::vector<int>& perm = orders[epoch & 1];
                hipCheck(hipMemcpyAsync(order, perm.data(), perm.size()*sizeof(int), hipMemcpyHostToDevice, m->stream), "upload");
                hipCheck(hipMemsetAsync(buf.loss, 0, sizeof(double), m->stream), "memset");
                float rate = (float) (lr*std::pow(decay, (double) epoch));
                for (int64_t b0 = 0; b0 < n; b0 += batch) {
                    int count = (int) std::min<int64_t>(batch, n - b0);
                    minibatch(m, data, order + b0, count, buf, true, rate, nullptr);
                }
                if (epoch + 1 < epochs)
                    shuffled(epoch + 1);
                double loss = 0;
                hipCheck(hipMemcpyAsync(&loss, buf.loss, sizeof(double), hipMemcpyDeviceToHost, m->stream), "download");
                hipCheck(hipStreamSynchronize(m->stream), "sync");
                if (epochLoss)
                    epochLoss[epoch] = loss/(double) n;
            }
        }
        catch (...) {
            (void) hipStreamSynchronize(m->stream);
            (void) hipFree(order);
            throw;
        }
        (void) hipFree(order);
    })
}

int lbm_mlp_forward(lbm_mlp* m, const float* features, int64_t n, float* out) {
    MLP_TRY({
        if (n <= 0 || n > 0x7FFFFFFF)
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_forward: invalid n");
        Dataset data(m, features, nullptr, n);
        float* du = deviceAlloc<float>((size_t) n*MLP_OUT);
        launchMlpInfer(m->dev, data.X, (int) n, (float) m->norm.out_scale, du, m->stream);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess)
            e = hipMemcpyAsync(out, du, (size_t) n*MLP_OUT*sizeof(float), hipMemcpyDeviceToHost, m->stream);
        if (e == hipSuccess)
            e = hipStreamSynchronize(m->stream);
        (void) hipStreamSynchronize(m->stream);
        (void) hipFree(du);
        hipCheck(e, "forward");
    })
}

int lbm_mlp_forward_noalloc(lbm_mlp* m, const float* features, int64_t n, float* out) {
    MLP_TRY({
        if (n <= 0 || n > LBM_MLP_NOALLOC_MAX_ROWS) {
            std::stringstream msg;
            msg << "lbm_mlp_forward_noalloc: n = " << n << " is outside [1, LBM_MLP_NOALLOC_MAX_ROWS = "
                << LBM_MLP_NOALLOC_MAX_ROWS << "]";
            throw MlpError(LBM_ERROR_INVALID, msg.str());
        }
        char* base = (char*) m->scratch;
        float* raw = (float*) base;
        _Float16* X = (_Float16*) (base + NOALLOC_RAW_BYTES);
        float* du = (float*) (base + NOALLOC_RAW_BYTES + NOALLOC_X_BYTES);
        hipCheck(hipMemcpyAsync(raw, features, (size_t) n*MLP_IN*sizeof(float), hipMemcpyHostToDevice, m->stream),
                "forward upload");
        mlpNormalize<<<blocksFor(n*MLP_IN_PAD, 256), 256, 0, m->stream>>>(raw, nullptr, n, mlpClosureNorm(m), X,
                nullptr);
        launchMlpInfer(m->dev, X, (int) n, (float) m->norm.out_scale, du, m->stream);
        hipCheck(hipGetLastError(), "forward launch");
        hipCheck(hipMemcpyAsync(out, du, (size_t) n*MLP_OUT*sizeof(float), hipMemcpyDeviceToHost, m->stream),
                "forward download");
        hipCheck(hipStreamSynchronize(m->stream), "forward");
    })
}

int lbm_mlp_gradients(lbm_mlp* m, const float* features, const float* targets, int64_t n, float* grad, double* loss) {
    MLP_TRY({
        if (n <= 0 || n > (1 << 20))
            throw MlpError(LBM_ERROR_INVALID, "lbm_mlp_gradients: n must be in [1, 2^20]");
        Dataset data(m, features, targets, n);
        int padded = (int) ((n + CHUNK - 1)/CHUNK*CHUNK);
        TrainBuffers buf;
        buf.allocate(padded);
        std::vector<int> rows(padded, 0);
        std::iota(rows.begin(), rows.begin() + n, 0);
        int* dRows = deviceAlloc<int>(padded);
        float* dGrad = deviceAlloc<float>(MLP_PARAMS);
        double lossSum = 0;
        hipError_t e = hipMemcpyAsync(dRows, rows.data(), padded*sizeof(int), hipMemcpyHostToDevice, m->stream);
        if (e == hipSuccess)
            e = hipMemsetAsync(buf.loss, 0, sizeof(double), m->stream);
        if (e == hipSuccess) {
            minibatch(m, data, dRows, (int) n, buf, false, 0.0f, dGrad);
            e = hipMemcpyAsync(grad, dGrad, MLP_PARAMS*sizeof(float), hipMemcpyDeviceToHost, m->stream);
        }
        if (e == hipSuccess)
            e = hipMemcpyAsync(&lossSum, buf.loss, sizeof(double), hipMemcpyDeviceToHost, m->stream);
        if (e == hipSuccess)
            e = hipStreamSynchronize(m->stream);
        (void) hipStreamSynchronize(m->stream);
        (void) hipFree(dRows);
        (void) hipFree(dGrad);
        hipCheck(e, "gradients");
        if (loss)
            *loss = lossSum/(double) n;
    })
}

}  // extern "C"
