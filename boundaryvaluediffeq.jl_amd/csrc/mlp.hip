// mlp.hip -- training and inference kernels of the warm-start network (mlp.h).
//
// A training workgroup of 16 waves handles a tile of 64 points and keeps the whole
// tile on chip: inputs, the three BF16 activation layers and one BF16 gradient
// layer live in LDS (about 137 KB), the hidden 256 x 256 products run on the
// gfx950 matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation; each wave
// owns 16 output columns of the 64-row tile), the 4-wide input layer and the
// 2-wide output layer run on the vector ALUs.  The tile goes forward and
// backward in the same workgroup; it writes the small FP32 gradients to a
// per-tile slot and the BF16 operands of the hidden matrices' gradients, which a
// second kernel forms over ranges of points; a third one sums slots and ranges,
// applies Adam to the FP32 master parameters and re-rounds them to BF16 in the
// two layouts the products read (output-major for the forward pass, input-major
// for the backward pass).  The step counter lives in device memory so that a
// captured step replays unchanged.
//
// Rounding points (the CPU oracle of the gradient check rounds at the same
// places): parameters to BF16 (round to nearest even), every activation to
// BF16 after tanh, every hidden-layer gradient dL/dz to BF16; all sums in FP32.
#include "mlp.h"

#include <math.h>

#include "anchors.h"
#include "mirk_device.h"

namespace mlp {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (gfx950: one v_cvt_pk_bf16_f32)
__device__ inline uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ inline float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// tanh z = 1 - 2 / (1 + e^{2z}) with the hardware exponential (absolute error
// ~1e-7, far below the BF16 rounding the activations then get)
__device__ inline float tanh_f(float z) { return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __expf(2.f * z)); }

struct __align__(16) Tile {
    uint16_t h[3][T][HP];   // activations of the hidden layers (BF16)
    uint16_t dz[T][HP];     // dL/dz of the layer being back-propagated (BF16)
    float x[T][NIN];        // normalised inputs
    float out[T][NOUT];     // network output (normalised units), then dL/dout
    float tgt[T][NOUT];
    int valid[T];
};

// Training runs a tile with 16 waves (TW threads, four per SIMD): a tile is a chain of short
// phases, each bound by the latency of its LDS and L2 reads, and a batch of 8,192 points has
// only 128 tiles.  Tile kernel at that batch, the hidden gradients included: 63 us with 4
// waves, 48 us with 16.
constexpr int TW = 1024;

// acc[rt] (rows 16rt.., columns 16*wave..) = A (LDS, T x H) times the matrix whose column
// c is row c of G (global BF16, H x H, row-major).  All of the wave's operands of G are
// loaded at once, before the products.
__device__ inline void gemm_tile(const uint16_t *A, const uint16_t *G, int wave, int lane, f4 acc[4]) {
    const int i = lane & 15, g = lane >> 4;
    bf8 b[H / 32];
#pragma unroll
    for (int ks = 0; ks < H / 32; ++ks) b[ks] = *(const bf8 *)(G + (size_t)(16 * wave + i) * H + 32 * ks + 8 * g);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) acc[rt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < H / 32; ++ks)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
            acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                *(const bf8 *)(A + (size_t)(16 * rt + i) * HP + 32 * ks + 8 * g), b[ks], acc[rt], 0, 0, 0);
}

typedef unsigned int u2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

// The tile's rows of the operands of k_wgrad: act + array a of tile t, [H][T]
__device__ inline uint16_t *act_tile(const Work &wk, int a, int t) {
    return wk.act + ((size_t)a * wk.tiles + t) * (H * T);
}
// four consecutive points of a unit
__device__ inline void store4(uint16_t *p, const uint16_t (&v)[4]) {
    *(u2 *)p = u2{(unsigned)v[0] | ((unsigned)v[1] << 16), (unsigned)v[2] | ((unsigned)v[3] << 16)};
}

// Gradients of the hidden matrices, dW[k][n] = sum_p h[p][k] dz[p][n]: a workgroup forms
// a 64 x 64 block of one matrix over one range of the points.  The tile kernel leaves both
// operands with a unit's points contiguous, which is what an MFMA lane reads (16 bytes);
// each of the eight waves takes an eighth of the range, four steps of 32 points loaded at
// once (the loads' latency bounds it), and their sums meet in LDS.  At 8,192 points: tile
// kernel 35.9 us and 12.2 us here, against 48 us with the products in the tile kernel,
// which then wrote 0.5 MB of gradient per tile for k_adam to sum (15.3 us; now 6.7 us).
constexpr int GW = 8;
__global__ __launch_bounds__(64 * GW) void k_wgrad(Work wk) {
    __shared__ f4 red[GW][16][64];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
    // consecutive workgroups go to different XCDs: with eight ranges, each XCD's L2 holds one
    const int z = blockIdx.x % wk.splits, x = blockIdx.x / wk.splits;
    const int k0 = 64 * (x & 3), n0 = 64 * ((x >> 2) & 3), l = x >> 4;
    const long long steps = 2LL * wk.tiles, parts = (long long)GW * wk.splits, part = (long long)GW * z + wave;
    const int s0 = (int)(steps * part / parts), s1 = (int)(steps * (part + 1) / parts);
    f4 acc[4][4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) acc[rt][ct] = f4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int s, bf8 (&a)[4], bf8 (&b)[4]) {
        const int o = 32 * (s & 1) + 8 * g;
        const uint16_t *hp = act_tile(wk, l, s >> 1) + (k0 + i) * T + o;
        const uint16_t *dp = act_tile(wk, 2 + l, s >> 1) + (n0 + i) * T + o;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = *(const bf8 *)(dp + 16 * q * T);
            b[q] = *(const bf8 *)(hp + 16 * q * T);
        }
    };
    auto mul = [&](const bf8 (&a)[4], const bf8 (&b)[4]) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rt], b[ct], acc[rt][ct], 0, 0, 0);
    };
    int s = s0;
    for (; s + 4 <= s1; s += 4) {
        bf8 a[4][4], b[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) load(s + u, a[u], b[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u) mul(a[u], b[u]);
    }
    for (; s < s1; ++s) {
        bf8 a[4], b[4];
        load(s, a, b);
        mul(a, b);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) red[wave][4 * rt + ct][lane] = acc[rt][ct];
    __syncthreads();
    float *out = wk.hidden + ((size_t)z * 2 + l) * (H * H);
#pragma unroll
    for (int q = 0; q < 16 / GW; ++q) {
        const int f = wave * (16 / GW) + q, rt = f / 4, ct = f % 4;
        f4 v = red[0][f][lane];
#pragma unroll
        for (int w = 1; w < GW; ++w) v += red[w][f][lane];
        *(f4 *)(out + (size_t)(k0 + 16 * ct + i) * H + n0 + 16 * rt + 4 * g) = v;
    }
}

// Forward pass of the tile (S.x filled): hidden activations into S.h, output into S.out.
__device__ void forward_tile(Tile &S, const Net &net, int tid, const Work &wk) {
    const int wave = tid >> 6, lane = tid & 63;
    {  // layer 1 (4 -> 256): a thread owns column n and 16 points
        const int n = tid & (H - 1), p0 = (tid / H) * 16;
        float w[NIN];
#pragma unroll
        for (int i = 0; i < NIN; ++i) w[i] = net.q[OW1 + i * H + n];
        const float b = net.q[OB1 + n];
        uint16_t *act = act_tile(wk, 0, blockIdx.x) + n * T;
#pragma unroll
        for (int p1 = 0; p1 < 16; p1 += 8) {
            uint16_t v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int p = p0 + p1 + e;
                float z = b;
#pragma unroll
                for (int i = 0; i < NIN; ++i) z += S.x[p][i] * w[i];
                v[e] = f2bf(tanh_f(z));
                S.h[0][p][n] = v[e];
            }
            *(u4 *)(act + p0 + p1) = u4{(unsigned)v[0] | ((unsigned)v[1] << 16), (unsigned)v[2] | ((unsigned)v[3] << 16),
                                        (unsigned)v[4] | ((unsigned)v[5] << 16), (unsigned)v[6] | ((unsigned)v[7] << 16)};
        }
    }
    __syncthreads();
    const int i = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int l = 0; l < 2; ++l) {  // layers 2 and 3 (256 -> 256) on the matrix cores
        f4 acc[4];
        const int n = 16 * wave + i;
        const float bn = net.q[(l == 0 ? OB2 : OB3) + n];
        gemm_tile(&S.h[l][0][0], l == 0 ? net.w2f : net.w3f, wave, lane, acc);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            uint16_t v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = f2bf(tanh_f(acc[rt][j] + bn));
                S.h[l + 1][16 * rt + 4 * g + j][n] = v[j];
            }
            if (l == 0) store4(act_tile(wk, 1, blockIdx.x) + n * T + 16 * rt + 4 * g, v);
        }
        __syncthreads();
    }
    {  // output layer (256 -> 2): sixteen threads per point, every sixteenth input each
        const int p = tid >> 4, part = tid & 15;
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int it = 0; it < H / 16; ++it) {
            const int k = 16 * it + part;
            const float hk = bf2f(S.h[2][p][k]);
            o0 += hk * net.q[OW4 + 2 * k];
            o1 += hk * net.q[OW4 + 2 * k + 1];
        }
#pragma unroll
        for (int m = 1; m < 16; m *= 2) {
            o0 += __shfl_xor(o0, m);
            o1 += __shfl_xor(o1, m);
        }
        if (part == 0) {
            S.out[p][0] = o0 + net.q[OB4];
            S.out[p][1] = o1 + net.q[OB4 + 1];
        }
    }
    __syncthreads();
}

// Backward pass of the tile after forward_tile; inv_b = 1 / (points in the step).
// Writes the operands of k_wgrad, and the tile's other gradients and loss into its slot.  Sums over the tile's points: four
// threads per unit, every fourth point each (pt = 4 it + sub), combined by shuffles.
__device__ void backward_tile(Tile &S, const Net &net, int tid, float inv_b, const Work &wk) {
    float *part = wk.slots + (size_t)blockIdx.x * NSLOT;
    const int wave = tid >> 6, lane = tid & 63;
    const int i = lane & 15, g = lane >> 4;
    const int unit = tid >> 2, sub = tid & 3;
    auto sum4 = [](float v) {
        v += __shfl_xor(v, 1);
        return v + __shfl_xor(v, 2);
    };
    // dL/dout and the loss (L = sum 0.5 (out - y)^2 / B): one wave, a point per lane
    if (tid < T) {
        const int p = tid;
        float l = 0.f, d[NOUT];
#pragma unroll
        for (int o = 0; o < NOUT; ++o) {
            d[o] = S.valid[p] ? (S.out[p][o] - S.tgt[p][o]) : 0.f;
            l += 0.5f * d[o] * d[o];
            d[o] *= inv_b;
            S.out[p][o] = d[o];
        }
        l *= inv_b;
#pragma unroll
        for (int m = 1; m < T; m *= 2) {
            l += __shfl_xor(l, m);
#pragma unroll
            for (int o = 0; o < NOUT; ++o) d[o] += __shfl_xor(d[o], m);
        }
        if (p == 0) {
            part[SLOSS] = l;
#pragma unroll
            for (int o = 0; o < NOUT; ++o) part[SB4 + o] = d[o];
        }
    }
    __syncthreads();
    {  // output layer: dW4, and dz3 = (dout W4^T) * (1 - h3^2)
        const float w0 = net.q[OW4 + 2 * unit], w1 = net.q[OW4 + 2 * unit + 1];
        float g0 = 0.f, g1 = 0.f;
        // points in fours, so that their dz leave as one store
        uint16_t *act = act_tile(wk, 3, blockIdx.x) + unit * T;
#pragma unroll
        for (int r = 0; r < T / 16; ++r) {
            uint16_t v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int p = 16 * r + 4 * sub + e;
                const float hk = bf2f(S.h[2][p][unit]);
                const float d0 = S.out[p][0], d1 = S.out[p][1];
                g0 += hk * d0;
                g1 += hk * d1;
                v[e] = f2bf((d0 * w0 + d1 * w1) * (1.f - hk * hk));
                S.dz[p][unit] = v[e];
            }
            store4(act + 16 * r + 4 * sub, v);
        }
        g0 = sum4(g0);
        g1 = sum4(g1);
        if (sub < NOUT) part[SW4 + 2 * unit + sub] = sub == 0 ? g0 : g1;
    }
    __syncthreads();
#pragma unroll 1
    for (int l = 1; l >= 0; --l) {  // hidden layer l + 2 (weights W3 for l = 1, W2 for l = 0)
        {
            float s = 0.f;
#pragma unroll
            for (int it = 0; it < T / 4; ++it) s += bf2f(S.dz[4 * it + sub][unit]);
            s = sum4(s);
            if (sub == 0) part[(l == 1 ? SB3 : SB2) + unit] = s;
        }
        f4 acc[4];
        gemm_tile(&S.dz[0][0], l == 1 ? net.w3b : net.w2b, wave, lane, acc);
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            uint16_t v[4];
            const int k = 16 * wave + i;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int p = 16 * rt + 4 * g + j;
                const float hk = bf2f(S.h[l][p][k]);
                v[j] = f2bf(acc[rt][j] * (1.f - hk * hk));
                S.dz[p][k] = v[j];
            }
            if (l == 1) store4(act_tile(wk, 2, blockIdx.x) + k * T + 16 * rt + 4 * g, v);
        }
        __syncthreads();
    }
    {  // input layer: dW1, db1
        float gw[NIN] = {0.f, 0.f, 0.f, 0.f}, gb = 0.f;
#pragma unroll 8
        for (int it = 0; it < T / 4; ++it) {
            const int p = 4 * it + sub;
            const float d = bf2f(S.dz[p][unit]);
            gb += d;
#pragma unroll
            for (int q = 0; q < NIN; ++q) gw[q] += S.x[p][q] * d;
        }
#pragma unroll
        for (int q = 0; q < NIN; ++q) gw[q] = sum4(gw[q]);
        gb = sum4(gb);
#pragma unroll
        for (int q = 0; q < NIN; ++q)
            if (sub == q) part[OW1 + q * H + unit] = gw[q];
        if (sub == 0) part[OB1 + unit] = gb;
    }
}
static_assert(NIN == 4 && TW == 4 * H && TW == 16 * T, "the thread splits of a training tile");

__device__ inline void load_point(Tile &S, const Net &net, int p, bool valid, const float *xr, const float *yr) {
#pragma unroll
    for (int q = 0; q < NIN; ++q) S.x[p][q] = valid ? (xr[q] - net.in_shift[q]) * net.in_scale[q] : 0.f;
#pragma unroll
    for (int o = 0; o < NOUT; ++o)
        S.tgt[p][o] = (valid && yr) ? (yr[o] - net.out_shift[o]) / net.out_scale[o] : 0.f;
    S.valid[p] = valid ? 1 : 0;
}

// ------------------------------------------------------------------ kernels
__global__ __launch_bounds__(TW) void k_train_tile(Net net, TrainDev td) {
    __shared__ Tile S;
    const int tid = threadIdx.x;
    const int step = td.step[0];
    if (blockIdx.x == 0 && tid == 0) td.step[1] = step;  // for k_adam
    const int epoch = step / td.steps_per_epoch, sin = step % td.steps_per_epoch;
    const unsigned long long a = td.perm[2 * epoch], c = td.perm[2 * epoch + 1];
    const long long bsz = (long long)td.work.tiles * T;
    if (tid < T) {
        const unsigned long long gidx = (unsigned long long)sin * bsz + (unsigned long long)blockIdx.x * T + tid;
        const long long j = (long long)((a * gidx + c) % (unsigned long long)td.n);
        load_point(S, net, tid, true, td.x + j * NIN, td.y + j * NOUT);
    }
    __syncthreads();
    forward_tile(S, net, tid, td.work);
    backward_tile(S, net, tid, 1.0f / (float)bsz, td.work);
}

__global__ __launch_bounds__(TW) void k_grad_tile(Net net, const float *x, const float *y, int n, Work wk) {
    __shared__ Tile S;
    const int tid = threadIdx.x;
    if (tid < T) {
        const long long j = (long long)blockIdx.x * T + tid;
        const bool v = j < n;
        load_point(S, net, tid, v, x + (v ? j : 0) * NIN, y + (v ? j : 0) * NOUT);
    }
    __syncthreads();
    forward_tile(S, net, tid, wk);
    backward_tile(S, net, tid, 1.0f / (float)n, wk);
}

// Gradient of parameter j = 256 blockIdx + threadIdx (the loss for j = NPARAM): the sum over
// the tiles' slots, or over the ranges for the hidden matrices, in a fixed order (the same
// bits on every run).  Each of the block's four waves sums a quarter for all 256 values, 16
// bytes per lane and sixteen loads in flight.
__device__ inline float sum_grad(const Work &wk) {
    static_assert(OW2 % 256 == 0 && OB2 % 256 == 0 && OW3 % 256 == 0 && OB3 % 256 == 0 && (H * H) % 256 == 0,
                  "a block of 256 parameters lies within a hidden matrix or outside");
    __shared__ f4 red[4][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j0 = blockIdx.x * 256;
    const bool w2 = j0 >= OW2 && j0 < OB2, w3 = j0 >= OW3 && j0 < OB3;
    const float *src;
    int cnt, stride;
    bool in = true;
    if (w2 || w3) {
        src = wk.hidden + (w2 ? j0 - OW2 : H * H + j0 - OW3) + 4 * lane;
        cnt = wk.splits;
        stride = 2 * H * H;
    } else {
        src = wk.slots + slot_of(j0) + 4 * lane;
        in = slot_of(j0) + 4 * lane < NSLOT;
        cnt = wk.tiles;
        stride = NSLOT;
    }
    const int per = (cnt + 3) / 4, t0 = min(cnt, wave * per), t1 = min(cnt, t0 + per);
    f4 s = f4{0.f, 0.f, 0.f, 0.f};
    if (in) {
        constexpr int U = 16;
        f4 a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = s;
        for (int t = t0; t < t1; t += U) {
            f4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (t + u < t1) v[u] = *(const f4 *)(src + (size_t)(t + u) * stride);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (t + u < t1) a[u] += v[u];
        }
#pragma unroll
        for (int o = U / 2; o > 0; o /= 2)
#pragma unroll
            for (int u = 0; u < o; ++u) a[u] += a[u + o];
        s = a[0];
    }
    red[wave][lane] = s;
    __syncthreads();
    const float *r = (const float *)red + threadIdx.x;
    return (r[0] + r[256]) + (r[512] + r[768]);
}

__global__ __launch_bounds__(256) void k_sum_grad(Work wk, float *grad) {
    const float g = sum_grad(wk);
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j <= NPARAM) grad[j] = g;
}

__device__ inline void requant(const NetBufs &nb, int j, float w) {
    const uint16_t b = f2bf(w);
    nb.q[j] = bf2f(b);
    if (j >= OW2 && j < OW2 + H * H) {
        const int k = (j - OW2) / H, o = (j - OW2) % H;
        nb.w2b[k * H + o] = b;
        nb.w2f[o * H + k] = b;
    } else if (j >= OW3 && j < OW3 + H * H) {
        const int k = (j - OW3) / H, o = (j - OW3) % H;
        nb.w3b[k * H + o] = b;
        nb.w3f[o * H + k] = b;
    }
}

__global__ void k_quantize(NetBufs nb) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < NPARAM) requant(nb, j, nb.w[j]);
}

// Adam on the summed tile gradients (decoupled weight decay on matrices only),
// learning rate: linear warm-up then cosine decay to lr_min.
// The step it works on is step[1], written by k_train_tile; the thread of the loss advances
// step[0], which nothing else reads meanwhile.
__global__ __launch_bounds__(256) void k_adam(NetBufs nb, TrainDev td) {
    const int step = td.step[1];
    const int j = blockIdx.x * 256 + threadIdx.x;
    float m = 0.f, v = 0.f, w = 0.f;  // read before the sums, so that one wait covers both
    if (j < NPARAM) {
        m = nb.m[j];
        v = nb.v[j];
        w = nb.w[j];
    }
    const float g = sum_grad(td.work);
    if (j > NPARAM) return;
    if (j == NPARAM) {
        td.loss[step - td.step0] = g;
        td.step[0] = step + 1;
        return;
    }
    float lr;
    if (step < td.warmup) lr = td.lr * (float)(step + 1) / (float)td.warmup;
    else {
        const float f = (float)(step - td.warmup) / (float)max(1, td.total_steps - td.warmup);
        lr = td.lr_min + 0.5f * (td.lr - td.lr_min) * (1.f + cosf(3.14159265358979f * fminf(f, 1.f)));
    }
    const float t = (float)(step + 1);
    m = nb.m[j] = td.beta1 * m + (1.f - td.beta1) * g;
    v = nb.v[j] = td.beta2 * v + (1.f - td.beta2) * g * g;
    const float mh = m / (1.f - powf(td.beta1, t)), vh = v / (1.f - powf(td.beta2, t));
    const bool matrix = (j < OB1) || (j >= OW2 && j < OB2) || (j >= OW3 && j < OB3) || (j >= OW4 && j < OB4);
    if (matrix) w -= lr * td.weight_decay * w;
    w -= lr * mh / (sqrtf(vh) + td.eps);
    nb.w[j] = w;
    requant(nb, j, w);
}

// last instance whose first node is <= gidx
__device__ inline int instance_of_node(const BatchDev &B, long long gidx) {
    int lo = 0, hi = B.n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (B.init_off[mid] <= gidx) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// ------------------------------------------------------------------ inference
// Persistent inference: each workgroup keeps its waves' column slices of both
// hidden weight matrices in registers (2 x CT x 8 operands of 8 BF16 per lane)
// and streams 64-point tiles through two LDS activation buffers, so that the
// weights are read from memory once per workgroup instead of once per tile.
// what a source keeps of a point between reading its features and storing its
// output (the anchor source: the instance's parameters, time and family)
constexpr int kStash = 8;
// threads of an inference workgroup: two waves per SIMD, each with 32 columns of both hidden
// matrices (128 registers), so that one wave's LDS reads and exponentials hide the other's
// (262,144 points: 270 us with one wave per SIMD and 64 columns, 151 us)
constexpr int TI = 512;
constexpr int CT = H / (16 * (TI / 64));
// the features of kAhead tiles are read together, by all threads
constexpr int kAhead = TI / T;
struct InferTile {
    uint16_t h[2][T][HP];
    float w4[H][NOUT];
    float x[kAhead][T][NIN];
    float out[T][NOUT];
    double stash[kAhead][T][kStash];
    int valid[kAhead][T];
};

__device__ inline void hidden_reg(const uint16_t *A, uint16_t *Hout, const bf8 (&w)[CT][8], const float (&bias)[CT],
                                  int wave, int lane) {
    const int i = lane & 15, g = lane >> 4;
    f4 acc[4][CT];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        bf8 a[4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) a[rt] = *(const bf8 *)(A + (size_t)(16 * rt + i) * HP + 32 * ks + 8 * g);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rt], w[ct][ks], acc[rt][ct], 0, 0, 0);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                Hout[(size_t)(16 * rt + 4 * g + j) * HP + 16 * CT * wave + 16 * ct + i] =
                    f2bf(tanh_f(acc[rt][ct][j] + bias[ct]));
}

template <class Src>
__global__ __launch_bounds__(TI) void k_infer(Net net, Src src, long long npts) {
    __shared__ InferTile S;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
    bf8 w2[CT][8], w3[CT][8];
    float b2[CT], b3[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int n = 16 * CT * wave + 16 * ct + i;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            w2[ct][ks] = *(const bf8 *)(net.w2f + (size_t)n * H + 32 * ks + 8 * g);
            w3[ct][ks] = *(const bf8 *)(net.w3f + (size_t)n * H + 32 * ks + 8 * g);
        }
        b2[ct] = net.q[OB2 + n];
        b3[ct] = net.q[OB3 + n];
    }
    float w1[NIN];
#pragma unroll
    for (int q = 0; q < NIN; ++q) w1[q] = net.q[OW1 + q * H + (tid & (H - 1))];
    const float b1 = net.q[OB1 + (tid & (H - 1))];
    static_assert(NOUT * H == TI, "one output weight per thread");
    S.w4[tid / NOUT][tid % NOUT] = net.q[OW4 + tid];
    const float b40 = net.q[OB4], b41 = net.q[OB4 + 1];
    const long long ntiles = (npts + T - 1) / T;
    static_assert(kAhead * T == TI, "one feature point per thread");
    for (long long tile0 = blockIdx.x; tile0 < ntiles; tile0 += (long long)kAhead * gridDim.x) {
        {  // features of this workgroup's next kAhead tiles (tile0 + qa * gridDim.x)
            const int qa = tid / T, pa = tid % T;
            const long long tile = tile0 + (long long)qa * gridDim.x;
            const long long gi = tile * T + pa;
            const bool v = tile < ntiles && gi < npts;
            float xr[NIN] = {0.f, 0.f, 0.f, 0.f};
            if (v) src.features(gi, xr, &S.stash[qa][pa][0]);
#pragma unroll
            for (int q = 0; q < NIN; ++q) S.x[qa][pa][q] = v ? (xr[q] - net.in_shift[q]) * net.in_scale[q] : 0.f;
            S.valid[qa][pa] = v;
        }
        __syncthreads();
        for (int qa = 0; qa < kAhead; ++qa) {
        const long long tile = tile0 + (long long)qa * gridDim.x;
        if (tile >= ntiles) break;
        // layer 1: a thread owns a column and a half of the points
        const int n1 = tid & (H - 1), p0 = (tid / H) * (T * H / TI);
#pragma unroll 8
        for (int it = 0; it < T * H / TI; ++it) {
            const int p = p0 + it;
            float z = b1;
#pragma unroll
            for (int q = 0; q < NIN; ++q) z += S.x[qa][p][q] * w1[q];
            S.h[0][p][n1] = f2bf(tanh_f(z));
        }
        __syncthreads();
        hidden_reg(&S.h[0][0][0], &S.h[1][0][0], w2, b2, wave, lane);
        __syncthreads();
        hidden_reg(&S.h[1][0][0], &S.h[0][0][0], w3, b3, wave, lane);
        __syncthreads();
        {
            // output layer: eight threads per point, every eighth input each
            constexpr int TP = TI / T;
            const int p = tid / TP, part = tid % TP;
            float o0 = 0.f, o1 = 0.f;
#pragma unroll 16
            for (int it = 0; it < H / TP; ++it) {
                const int k = TP * it + part;
                const float hk = bf2f(S.h[0][p][k]);
                o0 += hk * S.w4[k][0];
                o1 += hk * S.w4[k][1];
            }
#pragma unroll
            for (int m = 1; m < TP; m *= 2) {
                o0 += __shfl_xor(o0, m);
                o1 += __shfl_xor(o1, m);
            }
            if (part == 0) {
                S.out[p][0] = (o0 + b40) * net.out_scale[0] + net.out_shift[0];
                S.out[p][1] = (o1 + b41) * net.out_scale[1] + net.out_shift[1];
            }
        }
        __syncthreads();
        if (tid < T && S.valid[qa][tid]) src.store(tile * T + tid, S.out[tid], &S.stash[qa][tid][0]);
        }
        __syncthreads();  // the next feature round overwrites x, stash and valid
    }
}

struct PredictSrc {
    const float *x;
    float *y;
    __device__ void features(long long gi, float *xr, double *) const {
#pragma unroll
        for (int q = 0; q < NIN; ++q) xr[q] = x[gi * NIN + q];
    }
    __device__ void store(long long gi, const float *o, const double *) const {
        y[gi * NOUT] = o[0];
        y[gi * NOUT + 1] = o[1];
    }
};

__device__ inline void batch_features(const BatchDev &B, int b, double t, int kind, float *xr) {
    const double p0 = B.params[B.param_off[b]];
    xr[0] = (float)(kind == FEAT_LOG10_PARAM ? log10(p0) : p0);
    xr[1] = (float)B.bc_val[(size_t)b * B.M];
    xr[2] = (float)B.bc_val[(size_t)b * B.M + 1];
    xr[3] = (float)t;
}

// every node of the initial meshes of a batch -> out[node][2]
struct NodeSrc {
    BatchDev B;
    double *out;
    int kind;
    __device__ void features(long long gi, float *xr, double *) const {
        batch_features(B, instance_of_node(B, gi), B.init_mesh[gi], kind, xr);
    }
    __device__ void store(long long gi, const float *o, const double *) const {
        out[gi * 2] = (double)o[0];
        out[gi * 2 + 1] = (double)o[1];
    }
};

// K anchors per instance -> anc[b][j] = (y1, y2, f1, f2) with f = f(t_j, y)
struct AnchorSrc {
    BatchDev B;
    double *anc;
    int K;
    int kind;
    // the stash keeps the instance's parameters (5), the anchor time and the family
    __device__ void features(long long gi, float *xr, double *st) const {
        const int b = (int)(gi / K);
        const double t = anchor_t(B, b, (int)(gi % K), K);
        batch_features(B, b, t, kind, xr);
        const int po = B.param_off[b], pn = B.param_cnt[b];
#pragma unroll
        for (int k = 0; k < bvpdev::Params<2>::MAXP; ++k) st[k] = k < pn ? B.params[po + k] : 0.0;
        st[5] = t;
        st[6] = (double)B.family[b];
    }
    __device__ void store(long long gi, const float *o, const double *st) const {
        bvpdev::Params<2> P;
#pragma unroll
        for (int k = 0; k < bvpdev::Params<2>::MAXP; ++k) P.p[k] = st[k];
        const double y[2] = {(double)o[0], (double)o[1]};
        double f[2];
        bvpdev::f_eval<2, double>((int)st[6], P, st[5], y, f);
        anc[gi * 4] = y[0];
        anc[gi * 4 + 1] = y[1];
        anc[gi * 4 + 2] = f[0];
        anc[gi * 4 + 3] = f[1];
    }
};

// the guess at every node from the anchors (materialised for inspection; a solve
// interpolates on the fly)
__global__ void k_anchor_fill(BatchDev B, const double *anc, int K, double *init_y) {
    const int b = blockIdx.x;
    const long long first = B.init_off[b];
    const int nodes = B.N0[b] + 1;
    for (int k = threadIdx.x; k < nodes; k += blockDim.x)
        anchor_hermite(anc, K, b, B.t0[b], B.t1[b], B.init_mesh[first + k], init_y + (first + k) * 2);
}

// ------------------------------------------------------------------ host side
Net NetBufs::view() const {
    Net n{};
    n.q = q;
    n.w2f = w2f;
    n.w3f = w3f;
    n.w2b = w2b;
    n.w3b = w3b;
    return n;
}

hipError_t launch_quantize(const NetBufs &nb, hipStream_t s) {
    k_quantize<<<(NPARAM + 255) / 256, 256, 0, s>>>(nb);
    return hipGetLastError();
}

// ranges of points of the hidden matrices' gradients: sixteen tiles each at least, so that a
// wave of k_wgrad has its four steps, and at most eight (8 x 32 blocks fill the chip)
static int splits_of(int tiles) { return tiles < 16 ? 1 : tiles < 128 ? tiles / 16 : 8; }

size_t work_floats(int tiles) {
    return (size_t)tiles * NSLOT + (size_t)splits_of(tiles) * 2 * H * H + (size_t)tiles * (4 * H * T / 2);
}

Work work_of(float *base, int tiles) {
    Work w;
    w.tiles = tiles;
    w.splits = splits_of(tiles);
    w.slots = base;
    w.hidden = base + (size_t)tiles * NSLOT;
    w.act = (uint16_t *)(w.hidden + (size_t)w.splits * 2 * H * H);
    return w;
}

constexpr int kGradBlocks = (NPARAM + 1 + 255) / 256;

hipError_t launch_train_step(const NetBufs &nb, const Net &net, const TrainDev &td, hipStream_t s) {
    k_train_tile<<<td.work.tiles, TW, 0, s>>>(net, td);
    k_wgrad<<<32 * td.work.splits, 64 * GW, 0, s>>>(td.work);
    k_adam<<<kGradBlocks, 256, 0, s>>>(nb, td);
    return hipGetLastError();
}

hipError_t launch_grad(const Net &net, const float *x, const float *y, int n, float *work, float *grad,
                       hipStream_t s) {
    const Work wk = work_of(work, (n + T - 1) / T);
    k_grad_tile<<<wk.tiles, TW, 0, s>>>(net, x, y, n, wk);
    k_wgrad<<<32 * wk.splits, 64 * GW, 0, s>>>(wk);
    k_sum_grad<<<kGradBlocks, 256, 0, s>>>(wk, grad);
    return hipGetLastError();
}

static unsigned infer_grid(long long npts, int num_cus) {
    const long long tiles = (npts + T - 1) / T;
    return (unsigned)(tiles < num_cus ? (tiles > 0 ? tiles : 1) : num_cus);
}

hipError_t launch_predict(const Net &net, const float *x, int n, float *out, int num_cus, hipStream_t s) {
    k_infer<PredictSrc><<<infer_grid(n, num_cus), TI, 0, s>>>(net, PredictSrc{x, out}, n);
    return hipGetLastError();
}

hipError_t launch_batch_guess(const Net &net, const BatchDev &B, double *init_y, long long total_nodes,
                              int feature_kind, int anchors, double *anc, int num_cus, hipStream_t s) {
    if (anchors == 0) {
        k_infer<NodeSrc><<<infer_grid(total_nodes, num_cus), TI, 0, s>>>(net, NodeSrc{B, init_y, feature_kind},
                                                                          total_nodes);
        return hipGetLastError();
    }
    const long long pts = (long long)B.n * anchors;
    k_infer<AnchorSrc><<<infer_grid(pts, num_cus), TI, 0, s>>>(net, AnchorSrc{B, anc, anchors, feature_kind}, pts);
    return hipGetLastError();
}

hipError_t launch_anchor_fill(const BatchDev &B, const double *anc, int anchors, double *init_y, hipStream_t s) {
    k_anchor_fill<<<B.n, 256, 0, s>>>(B, anc, anchors, init_y);
    return hipGetLastError();
}

}  // namespace mlp
