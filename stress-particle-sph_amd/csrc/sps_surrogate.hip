// sps_surrogate.hip - learned Drucker-Prager stress update (no counterpart in
// the reference).
//
// A multilayer perceptron 10 -> 128 -> 128 -> 128 -> 4 with SiLU activations
// maps (stress before the step, strain increment of the step expressed as the
// elastic stress increment D:de, cohesion, friction) to the correction that
// the exact return map (adapt_stress2, code/3_SPH_material_2018.f90:2066-2140)
// applies to the elastic trial stress.  Weights and activations are bfloat16,
// every product is accumulated in single precision by the matrix cores
// (v_mfma_f32_16x16x16_bf16); master weights, Adam moments and gradients are
// single precision.
//
// Features (all scaled by the stress scale S and the cohesion scale Sc given
// at set-up):
//   x[0:4] = sigma_n / S        x[4:8] = (sigma_trial - sigma_n) / S
//   x[8]   = c / Sc             x[9]   = tan(phi)
// Output y[0:4] = (R(sigma_trial) - sigma_trial) / F(sigma_trial), with F the
// yield function, positive at every plastic trial state: the correction per
// unit overstress, of order one, so that the network's relative error scales
// the correction, not the stress.
//
// In a step (SPS_MODE_FAST with a network attached) the final stress update
// of the stress points (k_rk_final) logs every plastic trial state; the
// network corrects them in one batch and each result is kept only if it is
// consistent, each residual at most the tolerance relative to the trial
// state's size (sqrt(J2) + |3 alpha p| + k_c): the yield function |F|, and
// the flow rule of the return map -- the mean stress unchanged (or at the
// apex beyond the tension cutoff) and the deviator parallel to the trial
// one.  Otherwise the exact return map's result stays.  Elastic trial states
// never reach the network (R is the identity there).
namespace sps {

typedef unsigned short bf16_t;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int MLP_NIN = SURR_NIN, MLP_NOUT = 4;
// smallest overstress F / (sqrt(J2) + |3 alpha p| + k_c) a state needs for the
// network to correct it (and for a training tuple)
constexpr double OVERSTRESS_MIN = 1e-9;
constexpr int MLP_IN = 16, MLP_H = 128, MLP_OUT = 16;   // padded to the 16-wide matrix tiles
// parameter blocks, weights as [in][out]
constexpr int PW1 = 0, PB1 = PW1 + MLP_IN * MLP_H, PW2 = PB1 + MLP_H, PB2 = PW2 + MLP_H * MLP_H,
              PW3 = PB2 + MLP_H, PB3 = PW3 + MLP_H * MLP_H, PW4 = PB3 + MLP_H, PB4 = PW4 + MLP_H * MLP_OUT,
              MLP_NPARAM = PB4 + MLP_OUT;

__device__ __forceinline__ bf16_t f2bf(float f) {   // round to nearest even
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float((unsigned)b << 16); }
__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu_grad(float z) {
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

// ---------------------------------------------------------- the network
// Layout of the matrix instruction (16 x 16 x 16, bfloat16 in, single
// precision out): lane l holds A[l % 16][4 (l / 16) + q] and
// B[4 (l / 16) + q][l % 16], q = 0..3, and gets C[4 (l / 16) + q][l % 16].
// A "tile word" below is a lane's four bfloat16 of a 16 x 16 tile, 8 bytes;
// tiles are stored as 64 consecutive words, so every load and store of one is
// a coalesced 512 bytes.
typedef unsigned long long tword_t;

__device__ __forceinline__ tword_t pack4(const bf16_t (&h)[4]) {
    return (tword_t)h[0] | (tword_t)h[1] << 16 | (tword_t)h[2] << 32 | (tword_t)h[3] << 48;
}
__device__ __forceinline__ v4s unpack4(tword_t u) {
    v4s r;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = (short)(u >> (16 * q));
    return r;
}

// Parameter i's bfloat16 value into the two tile orders of the weights: wf as
// the B operand of H W, wt as that of dZ W^T.  Biases are not packed.
__device__ __forceinline__ void put_weight(bf16_t *__restrict__ wf, bf16_t *__restrict__ wt, int i, bf16_t v) {
    const int base = i < PB1 ? PW1 : i < PW2 ? -1 : i < PB2 ? PW2 : i < PW3 ? -1 : i < PB3 ? PW3 : i < PW4 ? -1
                   : i < PB4 ? PW4 : -1;
    if (base < 0) return;
    const int fin = base == PW1 ? MLP_IN : MLP_H, fout = base == PW4 ? MLP_OUT : MLP_H;
    const int r = (i - base) / fout, c = (i - base) % fout;
    auto at = [](int k, int j, int nj) { return (((k / 16) * (nj / 16) + j / 16) * 64 + (k % 16) / 4 * 16 + j % 16) * 4 + k % 4; };
    wf[base + at(r, c, fout)] = v;
    wt[base + at(c, r, fin)] = v;
}

// Forward pass of one 64-row block a workgroup, 16 rows a wave, and with GRAD
// the backward pass down to the gradients at every layer's output.  The rows'
// activations stay in the wave: a layer's result is laid out for the next
// product through 4 KiB of LDS of the wave's own, the pre-activations keep
// their registers for the way back (256 registers, 12 of them in scratch), and only what k_gemm_bf16_dw contracts
// over the rows is stored, as tile words (four consecutive rows of a column
// are what a lane holds of a result and what it needs as an operand there).
// The weights of a layer (32 KiB, in operand order) are fetched into registers
// while the layer before multiplies.  A launch per product with its operands
// gathered two bytes at a time took 530 us for 58 k rows, with 46 us for the
// activation's derivative and 390 us for the bias gradients; this takes 62 us,
// k_gemm_bf16_dw 22 us.  What is left here is mostly the activation: two
// exponentials and two correctly rounded divisions a value.
// Rows past nb (or *nbdev) count as zero inputs and have zero gradients.
struct NetPass {
    const float *feat, *targ;        // n x 10 and n x 4
    const unsigned *idx;             // row r of the batch is row idx[r] of the set (null: r)
    int nb;
    const int *nbdev;                // when set: nb = min(nb, *nbdev)
    const bf16_t *wf, *wt;
    const float *w;                  // single-precision parameters (the biases)
    float *Y;                        // rows x 16
    tword_t *X, *H[3], *dZ[3], *dY;  // GRAD: tiles of 16 rows
};

constexpr int NET_ROWS = 64;         // rows of a workgroup
constexpr int NET_TS = MLP_H + 8;    // LDS row of a wave's transposition (16-byte steps, banks apart)

template <bool GRAD> __global__ __launch_bounds__(256, 2) void k_gemm_bf16_chain(NetPass g) {
    __shared__ __align__(16) tword_t sW[64 * 64];
    __shared__ __align__(16) bf16_t sT[4][16 * NET_TS];
    int nb = g.nb;
    if (g.nbdev) nb = min(nb, *g.nbdev);
    if ((int)blockIdx.x * NET_ROWS >= nb) return;   // the whole workgroup
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, li = lane & 15, lg = lane >> 4;
    const int rb = blockIdx.x * (NET_ROWS / 16) + wave, r0 = 16 * rb;
    bf16_t *const mine = sT[wave];
    auto source = [&](int row) { return row < nb ? (g.idx ? (long long)g.idx[row] : (long long)row) : -1ll; };

    // weights on their way, 16 bytes (two tile words) at a time
    v4f pre[8];
    auto fetch = [&](const bf16_t *src, auto nw) {
        constexpr int N = decltype(nw)::value / 512;
#pragma unroll
        for (int k = 0; k < N; ++k) pre[k] = reinterpret_cast<const v4f *>(src)[t + 256 * k];
    };
    auto commit = [&](auto nw) {
        constexpr int N = decltype(nw)::value / 512;
#pragma unroll
        for (int k = 0; k < N; ++k) reinterpret_cast<v4f *>(sW)[t + 256 * k] = pre[k];
    };
    using Small = std::integral_constant<int, 8 * 64>;
    using Large = std::integral_constant<int, 64 * 64>;
    // acc = (the wave's 16 rows in LDS) x (the layer in sW)
    v4f acc[8];
    auto multiply = [&](auto kt_, auto nt_) {
        constexpr int KT = decltype(kt_)::value, NT = decltype(nt_)::value;
        v4s a[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k)
            a[k] = unpack4(*reinterpret_cast<const tword_t *>(mine + li * NET_TS + 16 * k + 4 * lg));
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KT; ++k)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[k], unpack4(sW[(k * NT + n) * 64 + lane]), acc[n],
                                                                   0, 0, 0);
    };
    using T1 = std::integral_constant<int, 1>;
    using T8 = std::integral_constant<int, 8>;
    auto put = [&](int n, const bf16_t (&h)[4]) {   // a result tile's words to the wave's rows
#pragma unroll
        for (int q = 0; q < 4; ++q) mine[(4 * lg + q) * NET_TS + 16 * n + li] = h[q];
    };

    // inputs
    fetch(g.wf + PW1, Small{});
    {
        const long long src = source(r0 + li);
        bf16_t h[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = 4 * lg + q;
            h[q] = f2bf(src >= 0 && c < MLP_NIN ? g.feat[src * MLP_NIN + c] : 0.0f);
        }
        *reinterpret_cast<tword_t *>(mine + li * NET_TS + 4 * lg) = pack4(h);
    }
    if (GRAD) {
        bf16_t h[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const long long src = source(r0 + 4 * lg + q);
            h[q] = f2bf(src >= 0 && li < MLP_NIN ? g.feat[src * MLP_NIN + li] : 0.0f);
        }
        g.X[(size_t)rb * 64 + lane] = pack4(h);
    }
    commit(Small{});
    __syncthreads();
    fetch(g.wf + PW2, Large{});
    multiply(T1{}, T8{});

    // hidden layers
    v4f Z[3][8];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const float *bias = g.w + (l == 0 ? PB1 : l == 1 ? PB2 : PB3);
        __syncthreads();   // every wave has read the weights and its rows
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const float bc = bias[16 * n + li];
            bf16_t h[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float z = acc[n][q] + bc;
                if (GRAD) Z[l][n][q] = z;
                h[q] = f2bf(silu(z));
            }
            put(n, h);
            if (GRAD) g.H[l][((size_t)rb * 8 + n) * 64 + lane] = pack4(h);
        }
        if (l < 2) commit(Large{});
        else commit(Small{});
        __syncthreads();
        if (l == 0) fetch(g.wf + PW3, Large{});
        if (l == 1) fetch(g.wf + PW4, Small{});
        if (l == 2 && GRAD) fetch(g.wt + PW4, Small{});
        if (l < 2) multiply(T8{}, T8{});
        else multiply(T8{}, T1{});
    }

    // output, and the gradient of the mean squared error at it
    const float inv = 1.0f / (float)(nb * MLP_NOUT);
    const float b4 = g.w[PB4 + li];
    __syncthreads();
    {
        bf16_t h[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = r0 + 4 * lg + q;
            const float y = acc[0][q] + b4;
            g.Y[(size_t)row * MLP_OUT + li] = y;
            if (GRAD) {
                const long long src = source(row);
                const float d = src >= 0 && li < MLP_NOUT ? y - g.targ[src * MLP_NOUT + li] : 0.0f;
                h[q] = f2bf(2.0f * d * inv);
            }
        }
        if (!GRAD) return;
        put(0, h);
        g.dY[(size_t)rb * 64 + lane] = pack4(h);
    }
    commit(Small{});
    __syncthreads();
    fetch(g.wt + PW3, Large{});
    multiply(T1{}, T8{});
#pragma unroll
    for (int l = 2; l >= 0; --l) {   // dZ = dH * SiLU'(Z), then dH of the layer below
        if (l > 0) __syncthreads();
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            bf16_t h[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) h[q] = f2bf((acc[n][q] + 0.0f) * silu_grad(Z[l][n][q]));
            if (l > 0) put(n, h);
            g.dZ[l][((size_t)rb * 8 + n) * 64 + lane] = pack4(h);
        }
        if (l == 0) break;
        commit(Large{});
        __syncthreads();
        if (l == 2) fetch(g.wt + PW2, Large{});
        multiply(T8{}, T8{});
    }
}

// Weight gradients: dW = H^T dZ of the layers and the bias gradients (a row
// of ones in the place of H^T), over a chunk of 16-row tiles a workgroup;
// blockIdx.y: 0 the second layer, 1 the third, 2 the first and the last.
// Its sums are part[chunk], which k_mlp_loss_reduce adds up: with atomics on the
// 37 k gradients every chunk had to be long to keep their number down.
// A wave takes two rows of 16 x 16 tiles of dW (64 registers of sums).
__global__ __launch_bounds__(256) void k_gemm_bf16_dw(NetPass g, int nrb, int chunk, float *__restrict__ part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
    const int lo = blockIdx.x * chunk, hi = min(lo + chunk, nrb);
    float *const out = part + (size_t)blockIdx.x * MLP_NPARAM;
    const v4s ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    auto mm = [](const v4s &a, const v4s &b, const v4f &c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
    };
    auto store = [&](const v4f &c, int pw, int fout, int it, int jt) {
#pragma unroll
        for (int q = 0; q < 4; ++q) out[pw + (16 * it + 4 * lg + q) * fout + 16 * jt + li] = c[q];
    };
    auto store_bias = [&](const v4f &c, int pb, int jt) {   // every row holds the sum
        if (lg == 0) out[pb + 16 * jt + li] = c[0];
    };
    if (blockIdx.y < 2) {
        const tword_t *__restrict__ A = g.H[blockIdx.y], *__restrict__ B = g.dZ[blockIdx.y + 1];
        v4f acc[2][8], bias[2] = {zero, zero};
#pragma unroll
        for (int n = 0; n < 8; ++n) acc[0][n] = acc[1][n] = zero;
        for (int rb = lo; rb < hi; ++rb) {
            const size_t at = (size_t)rb * 8 * 64 + lane;
            const v4s a0 = unpack4(A[at + 128 * wave]), a1 = unpack4(A[at + 128 * wave + 64]);
            const v4s c0 = unpack4(B[at + 128 * wave]), c1 = unpack4(B[at + 128 * wave + 64]);
            v4s b[8];
#pragma unroll
            for (int n = 0; n < 8; ++n) b[n] = unpack4(B[at + 64 * n]);
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                acc[0][n] = mm(a0, b[n], acc[0][n]);
                acc[1][n] = mm(a1, b[n], acc[1][n]);
            }
            bias[0] = mm(ones, c0, bias[0]);
            bias[1] = mm(ones, c1, bias[1]);
        }
        const int pw = blockIdx.y ? PW3 : PW2, pb = blockIdx.y ? PB3 : PB2;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            store(acc[0][n], pw, MLP_H, 2 * wave, n);
            store(acc[1][n], pw, MLP_H, 2 * wave + 1, n);
        }
        store_bias(bias[0], pb, 2 * wave);
        store_bias(bias[1], pb, 2 * wave + 1);
    } else {
        v4f w1[2] = {zero, zero}, b1[2] = {zero, zero}, w4[2] = {zero, zero}, b4 = zero;
        for (int rb = lo; rb < hi; ++rb) {
            const size_t at = (size_t)rb * 8 * 64 + lane, at1 = (size_t)rb * 64 + lane;
            const v4s x = unpack4(g.X[at1]), dy = unpack4(g.dY[at1]);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const v4s d = unpack4(g.dZ[0][at + 64 * (2 * wave + k)]), h = unpack4(g.H[2][at + 64 * (2 * wave + k)]);
                w1[k] = mm(x, d, w1[k]);
                b1[k] = mm(ones, d, b1[k]);
                w4[k] = mm(h, dy, w4[k]);
            }
            b4 = mm(ones, dy, b4);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            store(w1[k], PW1, MLP_H, 0, 2 * wave + k);
            store_bias(b1[k], PB1, 2 * wave + k);
            store(w4[k], PW4, MLP_OUT, 2 * wave + k, 0);
        }
        if (wave == 0) store_bias(b4, PB4, 0);
    }
}

// The first blocks: g = the chunks' gradients added up (a parameter a
// thread).  The rest: the squared-error loss (mean over rows and the 4
// outputs), 256 rows a block, added to *loss.
constexpr int REDUCE_BLOCKS = (MLP_NPARAM + 255) / 256;
__global__ void k_mlp_loss_reduce(NetPass g, const float *__restrict__ part, int nchunk, float *__restrict__ grad,
                                  float *__restrict__ loss) {
    if ((int)blockIdx.x < REDUCE_BLOCKS) {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if (i >= MLP_NPARAM) return;
        float s = 0.0f;
#pragma unroll 8
        for (int c = 0; c < nchunk; ++c) s += part[(size_t)c * MLP_NPARAM + i];
        grad[i] = s;
        return;
    }
    __shared__ float s[256];
    const int r = ((int)blockIdx.x - REDUCE_BLOCKS) * 256 + threadIdx.x;
    float l = 0.0f;
    if (r < g.nb) {
        const long long src = g.idx ? (long long)g.idx[r] : (long long)r;
        const float inv = 1.0f / (float)(g.nb * MLP_NOUT);
#pragma unroll
        for (int c = 0; c < MLP_NOUT; ++c) {
            const float d = g.Y[(size_t)r * MLP_OUT + c] - g.targ[src * MLP_NOUT + c];
            l += d * d * inv;
        }
    }
    s[threadIdx.x] = l;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, s[0]);
}

// Adam (Kingma & Ba 2015) on the single-precision masters, then the weights'
// bfloat16 copies in operand order.
__global__ void k_mlp_adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                           const float *__restrict__ g, bf16_t *__restrict__ wf, bf16_t *__restrict__ wt,
                           int n, float lr, float b1,
                           float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    put_weight(wf, wt, i, f2bf(wi));
}

__global__ void k_mlp_to_bf16(const float *__restrict__ w, bf16_t *__restrict__ wf, bf16_t *__restrict__ wt, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) put_weight(wf, wt, i, f2bf(w[i]));
}

// ------------------------------------------------------- use in the step
// Drucker-Prager yield function of the reference's return map:
// F = sqrt(J2) + 3 alpha p - k_c (adapt_stress2, 3_...:2082-2134).
__device__ __forceinline__ double dp_yield(const double4 &s, double alpha2, double kc, double &sj2) {
    const double p = (s.x + s.y + s.w) / 3.0;
    const double d0 = s.x - p, d1 = s.y - p, d3 = s.w - p;
    sj2 = sqrt(s.z * s.z + 0.5 * (d0 * d0 + d1 * d1 + d3 * d3));
    return sj2 + 3 * alpha2 * p - kc;
}

// The network's corrections of the recorded states, kept where consistent.
__global__ void k_surrogate_apply(SurrogateDev G, const float *__restrict__ Y, double4 *__restrict__ stress,
                                  double tol) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int n = min((int)*G.count, G.cap);
    bool kept = false;
    if (k < n) {
        const double sc = G.stress_scale;
        const double4 t = G.s_tr[k];
        const double tanfi = G.mat[k].x, coh = G.mat[k].y;
        const float *y = Y + (long long)k * MLP_OUT;
        const double alpha2 = tanfi / (sqrt(9 + 12 * (tanfi * tanfi)));
        const double kc = (3 * coh) / (sqrt(9 + 12 * (tanfi * tanfi)));
        double sj2_t, sj2;
        const double ft = dp_yield(t, alpha2, kc, sj2_t);   // > 0: the state is plastic
        const double4 s = make_double4(t.x + ft * y[0], t.y + ft * y[1], t.z + ft * y[2], t.w + ft * y[3]);
        const double f = dp_yield(s, alpha2, kc, sj2);
        const double size = sj2_t + fabs(3 * alpha2 * (t.x + t.y + t.w) / 3.0) + kc;
        (void)sc;
        // consistency with the return map's flow rule: the returned deviator
        // is the trial one scaled down, at the trial mean stress, or at the
        // apex kc / (3 alpha) where the trial state is beyond the tension cutoff
        const double pt = (t.x + t.y + t.w) / 3.0, po = (s.x + s.y + s.w) / 3.0;
        const double p_exp = kc - 3 * alpha2 * pt < 0 ? kc / (3 * alpha2) : pt;
        const double a0 = t.x - pt, a1 = t.y - pt, a3 = t.w - pt;
        const double b0 = s.x - po, b1 = s.y - po, b3 = s.w - po;
        const double dot = t.z * s.z + 0.5 * (a0 * b0 + a1 * b1 + a3 * b3);   // the J2 inner product
        const double cross = sj2_t * sj2 - dot;                               // >= 0, 0 when parallel
        // left to the return map: an overstress at rounding level (it moved a few
        // bits), and sqrt(J2) <= 1e-5, where it zeroes the deviator whatever
        // the overstress (3_...:2122)
        kept = ft > OVERSTRESS_MIN * size && sj2_t > (double)10e-06f && fabs(f) <= tol * size &&
               fabs(po - p_exp) <= tol * size && cross <= tol * sj2_t * sj2_t;
        if (kept) stress[G.slot[k]] = s;
    }
    // per-wave counts, one atomic per wave
    const unsigned long long ev = __ballot(k < n), kp = __ballot(kept);
    if ((threadIdx.x & 63) == 0) {
        if (ev) atomicAdd(&G.stats[0], (unsigned long long)__popcll(ev));
        if (kp) atomicAdd(&G.stats[1], (unsigned long long)__popcll(kp));
    }
}

// The exact return map of n stresses, each with its own material (labels of
// training tuples).
__global__ void k_return_map(const double4 *__restrict__ in, const double2 *__restrict__ mat,
                             double4 *__restrict__ out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 s = in[i];
    const double2 m = mat[i];   // tan(phi), c
    adapt_stress(s, m.x, m.y);
    out[i] = s;
}

}  // namespace sps
