/*
 * mg_mlp.hip — the learned coarse-step correction (no counterpart in the reference).
 *
 * A per-particle MLP 64 -> 128 -> 128 -> 16 (SiLU hidden layers; 53 real inputs, 6 real
 * outputs, the rest zero padding to MFMA tile sizes) predicts two velocity corrections for
 * one coarse step of 4 dt, each the fine segment's value minus the plain coarse step's:
 *   drift c_d: the position moves by (v_next + c_d) 4 dt, as four fine steps move it;
 *   veval c_e: veval is the plain step's (v + v_next) / 2 + c_e, the fine segment's last.
 * The plain coarse step overshoots four fine steps by about 6 dt^2 a per step in position,
 * because the leapfrog drift uses the end-of-step velocity, and its veval lags by about
 * 1.5 dt a; the stored velocity itself agrees with the fine one to a difference that the
 * local state does not predict, so it keeps the plain step's value.
 * Inputs, from the particle's sorted state after the step's pressure and force passes:
 *   8 bonded neighbours (live own bond slots in slot order, then incoming bonds in CSR
 *   order): (x_j - x_i) and (v_j - v_i), 48 values; density and pressure; the coarse step's
 *   acceleration (FFORCE with walls, gravity and the acceleration limit, as the advance
 *   applies it), 3 values; zeros to 64.
 * Each input is normalised as (x - mu) * inv_sigma; output c is y_c * out_scale[c].
 *
 * Weights are bf16, accumulation fp32, on gfx950 MFMA (v_mfma_f32_16x16x32_bf16): for a
 * 16 x 32 A tile lane l holds A[l % 16][8 (l / 16) + e], for a 32 x 16 B tile lane l holds
 * B[8 (l / 16) + e][l % 16] (e = 0..7), and the 16 x 16 fp32 result lane l holds
 * D[4 (l / 16) + r][l % 16] (r = 0..3).
 *
 * Training runs a minibatch forward and backward in one kernel (bf16 operands, fp32
 * accumulation, gradient partials reduced in a fixed order) with fp32 Adam on fp32 master
 * weights; inference is two kernels per step.
 */

#define MLP_IN 64
#define MLP_IN_REAL 53
/* a correction that would move a particle farther than this in one step (world units, a
 * thousandth of the unit smoothing radius) is refused: the particle takes the plain step */
#define MLP_MAX_SHIFT 1e-3f
#define MLP_H 128
#define MLP_OUT 16
#define MLP_OUT_REAL 6
#define MLP_NBR 8

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }

/* sigmoid with the hardware exp2 and reciprocal (a few ulp; the network runs in bf16). The
 * same function serves training and inference. */
__device__ __forceinline__ float sigmoid_fast(float z)
{
    const float e = __builtin_amdgcn_exp2f(-1.44269504f * z);
    return __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float silu(float z) { return z * sigmoid_fast(z); }

/* d silu / dz = s (1 + z (1 - s)), s = sigmoid(z) */
__device__ __forceinline__ float silu_grad(float z)
{
    const float s = sigmoid_fast(z);
    return s * (1.0f + z * (1.0f - s));
}

/* Everything the inference kernel reads, device resident. Weight fragments are laid out so
 * that each lane's 8 bf16 of a B operand are contiguous:
 *   W?f[ntile][kchunk][col 0..15][k 0..31] = W[kchunk * 32 + k][ntile * 16 + col]. */
struct MlpDev {
    __bf16 w1f[(MLP_IN / 32) * (MLP_H / 16) * 16 * 32];
    __bf16 w2f[(MLP_H / 32) * (MLP_H / 16) * 16 * 32];
    __bf16 w3f[(MLP_H / 32) * (MLP_OUT / 16) * 16 * 32];
    float b1[MLP_H], b2[MLP_H], b3[MLP_OUT];
    float mu[MLP_IN], inv_sigma[MLP_IN];
    float out_scale[MLP_OUT];
    float in_limit;  /* |normalised input| above this -> fallback (plain coarse step) */
    float out_limit; /* |y| above this -> fallback */
};

/* ------------------------------------------------------------------ features
 * The 64 raw inputs of active particle i (sorted state after the pressure and force passes;
 * FFORCE in d.F). Neighbours: the live own bond slots in slot order, then the incoming bonds
 * in CSR order, skipping partners outside the active range and broken bonds (rest length
 * below 1e-9), up to MLP_NBR. Candidates are examined MLP_NBR at a time, each group's
 * records loaded together (partner, rest length, then slot), and the chosen neighbours'
 * positions and velocities loaded together at the end. */
__device__ __forceinline__ void mlp_features(const DS& d, const MgParams& p, uint32_t i, uint32_t na,
                                             float x[MLP_IN])
{
    const int N = d.N, B = d.B;
    const float* BPARf = (const float*)d.BPAR;
#pragma unroll
    for (int k = 0; k < MLP_IN; k++) x[k] = 0.0f;
    const uint32_t h = d.HOME[i];
    const float4 Pi = d.P[i], Vi = d.VEL[i];
    uint32_t sel[MLP_NBR];
    int m = 0;
    auto push = [&](uint32_t j) {
#pragma unroll
        for (int q = 0; q < MLP_NBR; q++)
            if (q == m) sel[q] = j;
        m++;
    };
    /* own live slots (LIVE: partner present; B <= 64) */
    uint64_t live = d.LIVE[h];
    while (live != 0ull && m < MLP_NBR) {
        uint32_t a[MLP_NBR], jh[MLP_NBR], jj[MLP_NBR];
        float rest[MLP_NBR];
        bool has[MLP_NBR];
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++) {
            has[k] = live != 0ull;
            a[k] = has[k] ? (uint32_t)__builtin_ctzll(live) : 0u;
            live &= live - 1ull;
        }
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++) {
            jh[k] = MG_NONE;
            rest[k] = 0.0f;
            if (has[k]) {
                const size_t bi = (size_t)a[k] * N + h;
                jh[k] = d.BPARTNER[bi];
                rest[k] = BPARf[bi * 4 + 1];
            }
        }
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++) jj[k] = (has[k] && jh[k] < (uint32_t)N) ? d.SLOT[jh[k]] : MG_NONE;
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++)
            if (m < MLP_NBR && jj[k] < na && !((double)rest[k] < 0.000000001)) push(jj[k]);
    }
    /* incoming bonds */
    const uint32_t e0 = d.INC_OFF[h], e1 = d.INC_OFF[h + 1];
    for (uint32_t e = e0; e < e1 && m < MLP_NBR; e += MLP_NBR) {
        uint32_t kh[MLP_NBR], kk[MLP_NBR];
        float rest[MLP_NBR];
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++) {
            kh[k] = MG_NONE;
            rest[k] = 0.0f;
            if (e + (uint32_t)k < e1) {
                const uint32_t packed = d.INC[e + (uint32_t)k];
                kh[k] = packed / (uint32_t)B;
                const uint32_t b = packed - kh[k] * (uint32_t)B;
                rest[k] = BPARf[((size_t)b * N + kh[k]) * 4 + 1];
            }
        }
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++) kk[k] = kh[k] < (uint32_t)N ? d.SLOT[kh[k]] : MG_NONE;
#pragma unroll
        for (int k = 0; k < MLP_NBR; k++)
            if (m < MLP_NBR && kk[k] < na && !((double)rest[k] < 0.000000001)) push(kk[k]);
    }
#pragma unroll
    for (int q = 0; q < MLP_NBR; q++) {
        if (q < m) {
            const float4 Pj = d.P[sel[q]], Vj = d.VEL[sel[q]];
            x[6 * q + 0] = Pj.x - Pi.x;
            x[6 * q + 1] = Pj.y - Pi.y;
            x[6 * q + 2] = Pj.z - Pi.z;
            x[6 * q + 3] = Vj.x - Vi.x;
            x[6 * q + 4] = Vj.y - Vi.y;
            x[6 * q + 5] = Vj.z - Vi.z;
        }
    }
    const float4 Vi_eval = d.V[i];
    x[48] = 1.0f / Vi_eval.w; /* density */
    x[49] = Pi.w;             /* pressure */
    const f3 a = advance_accel(p, xyz(Pi), xyz(Vi_eval), xyz(d.F[i]));
    x[50] = a.x;
    x[51] = a.y;
    x[52] = a.z;
}

/* raw features of every active slot (rows of inactive slots are zero), for training data */
__global__ LAUNCH_BOUNDS_256 void k_mlp_features(DS d, MgParams p, float* __restrict__ X)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint32_t)d.N) return;
    float x[MLP_IN];
    const uint32_t na = d.ctr[MG_C_ACTIVE];
    if (i < na && d.GCELL[i] != MG_GRID_UNDEF) {
        mlp_features(d, p, i, na, x);
    } else {
#pragma unroll
        for (int k = 0; k < MLP_IN; k++) x[k] = 0.0f;
    }
    float4* o = (float4*)(X + (size_t)i * MLP_IN);
#pragma unroll
    for (int k = 0; k < MLP_IN / 4; k++) o[k] = make_float4(x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]);
}

/* --------------------------------------------------------------- inference
 * Two kernels per learned step.
 *
 * k_mlp_gather, one thread per slot: the particle's inputs, normalised and rounded to bf16,
 * into X[i][0..63] (128 bytes), and flags[i] = active | (every normalised input within
 * in_limit) << 1.
 *
 * k_mlp_apply, one wavefront per group of 32 particles (two 16-particle tiles): the three
 * layers as transposed products, H^T = W^T X^T, so the weights are the MFMA A operand and the
 * particles the B operand. The 16 x 16 result of a layer leaves lane l holding neurons
 * 16 mt + 4 (l / 16) + r of particle l % 16, which is a B operand of the next layer for the
 * K order nu(32 kc + 8 q + e) = 32 kc + (e < 4 ? 4 q + e : 16 + 4 q + e - 4) (q = l / 16);
 * W2 and W3 are packed with their input rows in that order (k_pack_frag with perm), so the
 * activations never leave registers. Weight fragments and biases are staged in LDS once per
 * block. DV[2i] = (c_d, 1), DV[2i + 1] = (c_e, 0) for corrected particles, zeros for inactive
 * or fallback ones (a normalised input beyond in_limit, an output beyond out_limit, or a
 * drift correction that would move the particle more than MLP_MAX_SHIFT in the step of
 * length dt); fallbacks of active particles are counted in *fallbacks. */
__global__ LAUNCH_BOUNDS_256 void k_mlp_gather(DS d, MgParams p, const MlpDev* __restrict__ net,
                                               uint4* __restrict__ X, uint32_t* __restrict__ flags)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint32_t)d.N) return;
    const uint32_t na = d.ctr[MG_C_ACTIVE];
    const bool act = i < na && d.GCELL[i] != MG_GRID_UNDEF;
    float x[MLP_IN];
    if (act) {
        mlp_features(d, p, i, na, x);
    } else {
#pragma unroll
        for (int k = 0; k < MLP_IN; k++) x[k] = 0.0f;
    }
    bool ok = act;
    uint32_t w[MLP_IN / 2];
#pragma unroll
    for (int k = 0; k < MLP_IN; k += 2) {
        const float v0 = act ? (x[k] - net->mu[k]) * net->inv_sigma[k] : 0.0f;
        const float v1 = act ? (x[k + 1] - net->mu[k + 1]) * net->inv_sigma[k + 1] : 0.0f;
        if (!(fabsf(v0) <= net->in_limit) || !(fabsf(v1) <= net->in_limit)) ok = false;
        const __bf16 b0 = to_bf16(v0), b1 = to_bf16(v1);
        w[k / 2] = (uint32_t)__builtin_bit_cast(uint16_t, b0) | ((uint32_t)__builtin_bit_cast(uint16_t, b1) << 16);
    }
    uint4* o = X + (size_t)i * (MLP_IN / 8);
#pragma unroll
    for (int k = 0; k < MLP_IN / 8; k++) o[k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
    flags[i] = (act ? 1u : 0u) | (ok ? 2u : 0u);
}

#define MLP_WAVES 4
struct MlpLds {
    __bf16 w1f[(MLP_IN / 32) * (MLP_H / 16) * 16 * 32];
    __bf16 w2f[(MLP_H / 32) * (MLP_H / 16) * 16 * 32];
    __bf16 w3f[(MLP_H / 32) * (MLP_OUT / 16) * 16 * 32];
    float b1[MLP_H], b2[MLP_H], b3[MLP_OUT], out_scale[MLP_OUT];
};

__device__ __forceinline__ bf16x8_t lds8(const __bf16* p) { return *(const bf16x8_t*)p; }

/* bias + SiLU of a layer's results (neuron 16 mt + 4 q + r in acc[mt][r]) packed as the next
 * layer's B operands: op[kc] holds neurons nu(32 kc + 8 q + e), e = 0..7 */
__device__ __forceinline__ void silu_pack(const f32x4_t acc[MLP_H / 16], const float* bias, int q,
                                          bf16x8_t op[MLP_H / 32])
{
#pragma unroll
    for (int kc = 0; kc < MLP_H / 32; kc++) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int mt = 2 * kc + (e >> 2), r = e & 3;
            op[kc][e] = to_bf16(silu(acc[mt][r] + bias[16 * mt + 4 * q + r]));
        }
    }
}

__global__ __launch_bounds__(256) void k_mlp_apply(const MlpDev* __restrict__ net, const uint4* __restrict__ X,
                                                   const uint32_t* __restrict__ flags, float4* __restrict__ DV,
                                                   uint32_t* __restrict__ fallbacks, float dt, uint32_t N)
{
    extern __shared__ float4 mg_lds[];
    MlpLds& L = *(MlpLds*)mg_lds;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    {
        const uint4* s1 = (const uint4*)net->w1f;
        uint4* d1 = (uint4*)L.w1f;
        for (int k = t; k < (int)(sizeof(L.w1f) / 16); k += 256) d1[k] = s1[k];
        const uint4* s2 = (const uint4*)net->w2f;
        uint4* d2 = (uint4*)L.w2f;
        for (int k = t; k < (int)(sizeof(L.w2f) / 16); k += 256) d2[k] = s2[k];
        const uint4* s3 = (const uint4*)net->w3f;
        uint4* d3 = (uint4*)L.w3f;
        for (int k = t; k < (int)(sizeof(L.w3f) / 16); k += 256) d3[k] = s3[k];
        for (int k = t; k < MLP_H; k += 256) {
            L.b1[k] = net->b1[k];
            L.b2[k] = net->b2[k];
        }
        if (t < MLP_OUT) {
            L.b3[t] = net->b3[t];
            L.out_scale[t] = net->out_scale[t];
        }
    }
    __syncthreads();
    const int q = l >> 4, col = l & 15;
    const uint32_t ngroups = (N + 31u) / 32u;
    uint32_t nfall = 0;
    for (uint32_t grp = blockIdx.x * MLP_WAVES + (uint32_t)w; grp < ngroups; grp += gridDim.x * MLP_WAVES) {
        /* layer-1 B operands: particle col of tile tt, inputs 32 kc + 8 q .. + 7 */
        bf16x8_t xb[2][MLP_IN / 32];
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            const uint32_t i = grp * 32u + (uint32_t)(16 * tt + col);
#pragma unroll
            for (int kc = 0; kc < MLP_IN / 32; kc++) {
                uint4 v = make_uint4(0u, 0u, 0u, 0u);
                if (i < N) v = X[(size_t)i * (MLP_IN / 8) + (size_t)(4 * kc + q)];
                xb[tt][kc] = __builtin_bit_cast(bf16x8_t, v);
            }
        }
        /* layer 1: [128 x 64] x [64 x 16] per tile */
        f32x4_t acc[2][MLP_H / 16];
#pragma unroll
        for (int mt = 0; mt < MLP_H / 16; mt++) {
            acc[0][mt] = acc[1][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kc = 0; kc < MLP_IN / 32; kc++) {
                const bf16x8_t a = lds8(&L.w1f[((mt * (MLP_IN / 32) + kc) * 16 + col) * 32 + 8 * q]);
                acc[0][mt] = mfma16(a, xb[0][kc], acc[0][mt]);
                acc[1][mt] = mfma16(a, xb[1][kc], acc[1][mt]);
            }
            __builtin_amdgcn_sched_barrier(0); /* one tile's weight fragments live at a time */
        }
        bf16x8_t hb[2][MLP_H / 32];
        silu_pack(acc[0], L.b1, q, hb[0]);
        silu_pack(acc[1], L.b1, q, hb[1]);
        /* layer 2: [128 x 128] x [128 x 16] per tile */
#pragma unroll
        for (int mt = 0; mt < MLP_H / 16; mt++) {
            acc[0][mt] = acc[1][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kc = 0; kc < MLP_H / 32; kc++) {
                const bf16x8_t a = lds8(&L.w2f[((mt * (MLP_H / 32) + kc) * 16 + col) * 32 + 8 * q]);
                acc[0][mt] = mfma16(a, hb[0][kc], acc[0][mt]);
                acc[1][mt] = mfma16(a, hb[1][kc], acc[1][mt]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        silu_pack(acc[0], L.b2, q, hb[0]);
        silu_pack(acc[1], L.b2, q, hb[1]);
        /* layer 3: [16 x 128] x [128 x 16] per tile */
        f32x4_t y[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kc = 0; kc < MLP_H / 32; kc++) {
            const bf16x8_t a = lds8(&L.w3f[(kc * 16 + col) * 32 + 8 * q]);
            y[0] = mfma16(a, hb[0][kc], y[0]);
            y[1] = mfma16(a, hb[1][kc], y[1]);
        }
        /* lane l holds outputs 4 q + r of particle col; lanes q = 0 take outputs 4 and 5 from
         * lane l + 16 and write the particle's corrections */
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            float o[4];
            bool lim = true;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int c = 4 * q + r;
                const float v = y[tt][r] + L.b3[c];
                if (c < MLP_OUT_REAL && !(fabsf(v) <= net->out_limit)) lim = false;
                o[r] = v * L.out_scale[c];
            }
            const float o4 = __shfl(o[0], l + 16), o5 = __shfl(o[1], l + 16);
            const bool lim_hi = __shfl((int)lim, l + 16) != 0;
            if (q == 0) {
                const uint32_t i = grp * 32u + (uint32_t)(16 * tt + col);
                if (i < N) {
                    const uint32_t fl = flags[i];
                    const f3 cd = mk3(o[0], o[1], o[2]), ce = mk3(o[3], o4, o5);
                    /* the residual the network may apply: a shift of at most MLP_MAX_SHIFT */
                    const bool use = (fl & 2u) != 0u && lim && lim_hi && sqrtf(dot3(cd, cd)) * dt <= MLP_MAX_SHIFT;
                    if (use) {
                        DV[2 * (size_t)i] = make_float4(cd.x, cd.y, cd.z, 1.0f);
                        DV[2 * (size_t)i + 1] = make_float4(ce.x, ce.y, ce.z, 0.0f);
                    } else {
                        DV[2 * (size_t)i] = make_float4(0.f, 0.f, 0.f, 0.f);
                        DV[2 * (size_t)i + 1] = make_float4(0.f, 0.f, 0.f, 0.f);
                    }
                    if ((fl & 1u) && !use) nfall++;
                }
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) nfall += (uint32_t)__shfl_xor((int)nfall, o);
    if (l == 0 && nfall) atomicAdd(fallbacks, nfall);
}

/* ------------------------------------------------------------ training
 * A step of Adam is three launches: k_net_pass takes a minibatch forward and backward, k_net_grad
 * multiplies out the gradients, k_net_reduce adds their partials and updates the weights. (The
 * layer-by-layer form they replaced, a GEMM with elementwise and column-sum kernels over
 * intermediates in memory, took 21 launches and 316 us per step of 16,384 rows; its sums over
 * rows are kept in their order, because a last-bit difference in a gradient grows, through the
 * bf16 rounding of the weights, to 1e-4 of them within 60 steps.) Now 22 + 14 + 7 us at 16,384
 * rows, 2.6 GFLOP: the pass is bound by its chain of six layers with a barrier each (one workgroup
 * of four wavefronts per CU), the other two by the 55 MB of operands and partials.
 *
 * k_net_pass: a workgroup takes 64 rows through all layers, the activations in LDS and the
 * pre-activations in registers. Products are transposed, D[neuron][row] = W^T[neuron][k]
 * X^T[k][row], so wavefront w owns the 32 neurons from 32 w of each hidden layer for all 64 rows:
 * the weights are read once per workgroup, straight from memory in fragments of 16 contiguous
 * bytes per lane ([out][in] order forward, [in][out] backward), the rows' operands from LDS. The
 * weight gradients sum over rows, so their operands are kept transposed ([neuron][row]) and leave
 * in tiles of 16 neurons by 32 rows (1 KB), which k_net_grad reads whole. */
#define NET_ROWS 64
#define NET_LD(k) ((k) + 8) /* row stride of an LDS operand with k columns (bf16) */
struct NetLds {
    __bf16 Xr[NET_ROWS][NET_LD(MLP_IN)];
    __bf16 XT[MLP_IN][NET_LD(NET_ROWS)];
    union {
        __bf16 A1r[NET_ROWS][NET_LD(MLP_H)];   /* dead after layer 2 */
        __bf16 dZ1T[MLP_H][NET_LD(NET_ROWS)];
    };
    __bf16 A1T[MLP_H][NET_LD(NET_ROWS)];
    union {
        __bf16 A2r[NET_ROWS][NET_LD(MLP_H)];   /* dead after layer 3 */
        __bf16 dZ2r[NET_ROWS][NET_LD(MLP_H)];
    };
    __bf16 A2T[MLP_H][NET_LD(NET_ROWS)];
    __bf16 dZ2T[MLP_H][NET_LD(NET_ROWS)];
    __bf16 dYr[NET_ROWS][NET_LD(32)];          /* columns 16 .. 31 zero (K padding) */
    __bf16 dYT[MLP_OUT][NET_LD(NET_ROWS)];
    float loss[4];
};

/* What a pass leaves for the gradients: operand tiles [row chunk][neuron tile][16][32] in bf16, and
 * dZ1, dZ2 [rows][128], dY [rows][16] in fp32 for the bias gradients */
struct NetOps {
    __bf16 *x, *a1, *a2, *dz1, *dz2, *dy;
    float *fz1, *fz2, *fy;
};

/* bf16 weights of a pass: [out][in] (forward) and [in][out] (backward) */
struct NetWeights {
    const __bf16 *w1t, *w2t, *w3t; /* [128][64], [128][128], [16][128] */
    const __bf16 *w2, *w3;         /* [128][128], [128][16] */
    const float *b1, *b2, *b3;
    const float *mu, *inv_sigma;
};

typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;

/* four neurons n .. n + 3 of a row into the row-major and the transposed operand */
template <int KR, int KT>
__device__ __forceinline__ void net_put(__bf16 (*rows)[KR], __bf16 (*cols)[KT], int row, int n, const float v[4])
{
    bf16x4_t b;
#pragma unroll
    for (int r = 0; r < 4; r++) b[r] = to_bf16(v[r]);
    if (rows) *(bf16x4_t*)&rows[row][n] = b;
#pragma unroll
    for (int r = 0; r < 4; r++) cols[n + r][row] = b[r];
}

/* the block's operand tiles (TILES x 16 neurons, 64 rows: two chunks of 32) to memory */
template <int TILES>
__device__ __forceinline__ void net_tiles(const __bf16 (*T)[NET_LD(NET_ROWS)], __bf16* __restrict__ out, size_t blk, int t)
{
    uint4* o = (uint4*)out + blk * (size_t)(2 * TILES * 64);
#pragma unroll
    for (int k = t; k < 2 * TILES * 64; k += 256) {
        const int l = k & 63, nt = (k >> 6) % TILES, kc = (k >> 6) / TILES;
        o[k] = *(const uint4*)&T[16 * nt + (l & 15)][32 * kc + 8 * (l >> 4)];
    }
}

/* offsets of the parameter vector: W1 b1 W2 b2 W3 b3 */
#define NET_W1 0
#define NET_B1 (NET_W1 + MLP_IN * MLP_H)
#define NET_W2 (NET_B1 + MLP_H)
#define NET_B2 (NET_W2 + MLP_H * MLP_H)
#define NET_W3 (NET_B2 + MLP_H)
#define NET_B3 (NET_W3 + MLP_H * MLP_OUT)
#define NET_PARAMS (NET_B3 + MLP_OUT)

/* BACK: the operands of the gradients into O and the loss into lpart[block] (times inv_count);
 * else the outputs into Y [rows][16] */
template <bool BACK>
__global__ __launch_bounds__(256, 1) void k_net_pass(NetWeights W, const float* __restrict__ X,
                                                     const float* __restrict__ T, const float* __restrict__ mask,
                                                     size_t rows, float inv_count, NetOps O, float* __restrict__ lpart,
                                                     float* __restrict__ Y)
{
    extern __shared__ float4 mg_lds[];
    NetLds& L = *(NetLds*)mg_lds;
    const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63, q = l >> 4, col = l & 15;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    float lsum = 0.0f;
    if (BACK)
        for (int k = t; k < NET_ROWS * 16; k += 256) L.dYr[k >> 4][16 + (k & 15)] = to_bf16(0.0f);
    const size_t blk = blockIdx.x, r0 = blk * NET_ROWS;
    /* inputs: chunk c of 4 columns of row c / 16 */
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int c = t + 256 * k, row = c >> 4, k0 = 4 * (c & 15);
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        const bool in = r0 + (size_t)row < rows;
        if (in) x = *(const float4*)(X + (r0 + (size_t)row) * MLP_IN + k0);
        const float4 m = *(const float4*)(W.mu + k0), s = *(const float4*)(W.inv_sigma + k0);
        const float v[4] = {in ? (x.x - m.x) * s.x : 0.f, in ? (x.y - m.y) * s.y : 0.f,
                            in ? (x.z - m.z) * s.z : 0.f, in ? (x.w - m.w) * s.w : 0.f};
        net_put(L.Xr, L.XT, row, k0, v);
    }
    __syncthreads();
    /* layer 1 */
    f32x4_t z1[2][4], z2[2][4];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int mt = 2 * w + a;
        bf16x8_t wf[2];
#pragma unroll
        for (int kc = 0; kc < 2; kc++) wf[kc] = lds8(W.w1t + (size_t)(16 * mt + col) * MLP_IN + 32 * kc + 8 * q);
        const float4 bias = *(const float4*)(W.b1 + 16 * mt + 4 * q);
#pragma unroll
        for (int rt = 0; rt < 4; rt++) {
            f32x4_t acc = zero;
#pragma unroll
            for (int kc = 0; kc < 2; kc++) acc = mfma16(wf[kc], lds8(&L.Xr[16 * rt + col][32 * kc + 8 * q]), acc);
            acc[0] += bias.x; acc[1] += bias.y; acc[2] += bias.z; acc[3] += bias.w;
            z1[a][rt] = acc;
            const float v[4] = {silu(acc[0]), silu(acc[1]), silu(acc[2]), silu(acc[3])};
            net_put(L.A1r, L.A1T, 16 * rt + col, 16 * mt + 4 * q, v);
        }
    }
    __syncthreads();
    /* layer 2 */
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int mt = 2 * w + a;
        bf16x8_t wf[4];
#pragma unroll
        for (int kc = 0; kc < 4; kc++) wf[kc] = lds8(W.w2t + (size_t)(16 * mt + col) * MLP_H + 32 * kc + 8 * q);
        const float4 bias = *(const float4*)(W.b2 + 16 * mt + 4 * q);
#pragma unroll
        for (int rt = 0; rt < 4; rt++) {
            f32x4_t acc = zero;
#pragma unroll
            for (int kc = 0; kc < 4; kc++) acc = mfma16(wf[kc], lds8(&L.A1r[16 * rt + col][32 * kc + 8 * q]), acc);
            acc[0] += bias.x; acc[1] += bias.y; acc[2] += bias.z; acc[3] += bias.w;
            z2[a][rt] = acc;
            const float v[4] = {silu(acc[0]), silu(acc[1]), silu(acc[2]), silu(acc[3])};
            net_put(L.A2r, L.A2T, 16 * rt + col, 16 * mt + 4 * q, v);
        }
    }
    __syncthreads();
    /* layer 3: wavefront w the rows 16 w .. 16 w + 15, lane outputs 4 q .. 4 q + 3 */
    {
        f32x4_t y = zero;
#pragma unroll
        for (int kc = 0; kc < 4; kc++)
            y = mfma16(lds8(W.w3t + (size_t)col * MLP_H + 32 * kc + 8 * q), lds8(&L.A2r[16 * w + col][32 * kc + 8 * q]), y);
        const float4 bias = *(const float4*)(W.b3 + 4 * q);
        y[0] += bias.x; y[1] += bias.y; y[2] += bias.z; y[3] += bias.w;
        const size_t row = r0 + (size_t)(16 * w + col);
        const bool in = row < rows;
        if (!BACK) {
            if (in) *(float4*)(Y + row * MLP_OUT + 4 * q) = make_float4(y[0], y[1], y[2], y[3]);
        } else {
            /* loss = sum over masked-in rows of |Y - T|^2 / count; dY = 2 (Y - T) / count */
            float g[4] = {0.f, 0.f, 0.f, 0.f};
            if (in && mask[row] != 0.f) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int c = 4 * q + r;
                    if (c >= MLP_OUT_REAL) continue;
                    const float e = y[r] - T[row * MLP_OUT_REAL + c];
                    lsum += e * e;
                    g[r] = 2.0f * e * inv_count;
                }
            }
            if (in) *(float4*)(O.fy + row * MLP_OUT + 4 * q) = make_float4(g[0], g[1], g[2], g[3]);
            net_put(L.dYr, L.dYT, 16 * w + col, 4 * q, g);
        }
    }
    if (!BACK) return;
    __syncthreads();
    /* dZ2 = (W3 dY) silu'(Z2); K = 16 outputs, padded to 32 with zeros */
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int mt = 2 * w + a;
        bf16x8_t wf = __builtin_bit_cast(bf16x8_t, make_uint4(0u, 0u, 0u, 0u));
        if (q < 2) wf = lds8(W.w3 + (size_t)(16 * mt + col) * MLP_OUT + 8 * q);
#pragma unroll
        for (int rt = 0; rt < 4; rt++) {
            const f32x4_t acc = mfma16(wf, lds8(&L.dYr[16 * rt + col][8 * q]), zero);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = acc[r] * silu_grad(z2[a][rt][r]);
            const size_t row = r0 + (size_t)(16 * rt + col);
            if (row < rows) *(float4*)(O.fz2 + row * MLP_H + 16 * mt + 4 * q) = make_float4(v[0], v[1], v[2], v[3]);
            net_put(L.dZ2r, L.dZ2T, 16 * rt + col, 16 * mt + 4 * q, v);
        }
    }
    __syncthreads();
    /* dZ1 = (W2 dZ2) silu'(Z1) */
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int mt = 2 * w + a;
        bf16x8_t wf[4];
#pragma unroll
        for (int kc = 0; kc < 4; kc++) wf[kc] = lds8(W.w2 + (size_t)(16 * mt + col) * MLP_H + 32 * kc + 8 * q);
#pragma unroll
        for (int rt = 0; rt < 4; rt++) {
            f32x4_t acc = zero;
#pragma unroll
            for (int kc = 0; kc < 4; kc++) acc = mfma16(wf[kc], lds8(&L.dZ2r[16 * rt + col][32 * kc + 8 * q]), acc);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = acc[r] * silu_grad(z1[a][rt][r]);
            const size_t row = r0 + (size_t)(16 * rt + col);
            if (row < rows) *(float4*)(O.fz1 + row * MLP_H + 16 * mt + 4 * q) = make_float4(v[0], v[1], v[2], v[3]);
            net_put((__bf16(*)[NET_LD(MLP_H)]) nullptr, L.dZ1T, 16 * rt + col, 16 * mt + 4 * q, v);
        }
    }
    __syncthreads();
    net_tiles<MLP_IN / 16>(L.XT, O.x, blk, t);
    net_tiles<MLP_H / 16>(L.A1T, O.a1, blk, t);
    net_tiles<MLP_H / 16>(L.A2T, O.a2, blk, t);
    net_tiles<MLP_H / 16>(L.dZ1T, O.dz1, blk, t);
    net_tiles<MLP_H / 16>(L.dZ2T, O.dz2, blk, t);
    net_tiles<MLP_OUT / 16>(L.dYT, O.dy, blk, t);
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
    if (l == 0) L.loss[w] = lsum;
    __syncthreads();
    if (t == 0) lpart[blk] = (((L.loss[0] + L.loss[1]) + L.loss[2]) + L.loss[3]) * inv_count;
}

/* Gradients of the weights, W[m][n] = sum over rows of A[row][m] dZ[row][n], in splits of `kper`
 * rows (a multiple of 32) that k_net_reduce adds in order, into part[split][NET_PARAMS]. One
 * wavefront per (split, 16-row tile of W, four column tiles): a chain of MFMAs over the split's
 * rows, 32 at a time, its operand tiles read whole from memory (1 KB per load) four chunks ahead.
 * Tasks of a split: W2 8 x 2, W1 4 x 2, W3 8. The blocks past the splits' tasks sum the bias
 * gradients' columns, rows t, t + 256, ... for each of 256 values of t, into bpart[t][272]
 * (b1, b2, b3); k_net_reduce adds the 256. */
#define NET_TASKS 32
#define NET_BIASES (2 * MLP_H + MLP_OUT)
#define NET_BIAS_BLOCKS (2 * 2 * 64 + 16)
__global__ LAUNCH_BOUNDS_256 void k_net_grad(NetOps O, size_t rows, int splits, int kper, float* __restrict__ part,
                                             float* __restrict__ bpart)
{
    const int t = threadIdx.x, l = t & 63, q = l >> 4, col = l & 15;
    const int tasks = (splits * NET_TASKS) / 4; /* blocks of four wavefronts */
    if ((int)blockIdx.x >= tasks) {
        int b = (int)blockIdx.x - tasks;
        const float* G;
        int cols, c, tt, to;
        if (b < 256) { /* 64 columns x 4 values of t */
            G = b < 128 ? O.fz1 : O.fz2;
            to = b < 128 ? 0 : MLP_H;
            b &= 127;
            cols = MLP_H;
            c = (b & 1) * 64 + l;
            tt = (b >> 1) * 4 + (t >> 6);
        } else { /* 16 columns x 16 values of t */
            G = O.fy;
            to = 2 * MLP_H;
            cols = MLP_OUT;
            c = t & 15;
            tt = (b - 256) * 16 + (t >> 4);
        }
        float s = 0.0f;
        size_t r = (size_t)tt;
        for (; r + 7 * 256 < rows; r += 8 * 256) {
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; k++) x[k] = G[(r + (size_t)k * 256) * cols + c];
#pragma unroll
            for (int k = 0; k < 8; k++) s += x[k];
        }
        for (; r < rows; r += 256) s += G[r * cols + c];
        bpart[(size_t)tt * NET_BIASES + to + c] = s;
        return;
    }
    const int task = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + (t >> 6));
    const int split = task / NET_TASKS, k = task % NET_TASKS;
    const bf16x8_t *A, *B;
    int ta, tb, mt, nt, nn, off, ld; /* tiles per chunk of A and B, the task's tiles, W's offset and row */
    if (k < 16) {
        A = (const bf16x8_t*)O.a1; B = (const bf16x8_t*)O.dz2;
        ta = tb = MLP_H / 16; mt = k >> 1; nt = (k & 1) * 4; nn = 4; off = NET_W2; ld = MLP_H;
    } else if (k < 24) {
        A = (const bf16x8_t*)O.x; B = (const bf16x8_t*)O.dz1;
        ta = MLP_IN / 16; tb = MLP_H / 16; mt = (k - 16) >> 1; nt = (k & 1) * 4; nn = 4; off = NET_W1; ld = MLP_H;
    } else {
        A = (const bf16x8_t*)O.a2; B = (const bf16x8_t*)O.dy;
        ta = MLP_H / 16; tb = 1; mt = k - 24; nt = 0; nn = 1; off = NET_W3; ld = MLP_OUT;
    }
    const size_t c0 = (size_t)split * (kper / 32), c1 = min(c0 + (size_t)(kper / 32), (rows + 31) / 32);
    A += (size_t)mt * 64 + l;
    B += (size_t)nt * 64 + l;
    f32x4_t acc[4];
#pragma unroll
    for (int n = 0; n < 4; n++) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (size_t c = c0; c < c1; c += 4) {
        bf16x8_t a[4], b[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const size_t cu = min(c + (size_t)u, c1 - 1);
            a[u] = A[cu * ta * 64];
#pragma unroll
            for (int n = 0; n < 4; n++)
                if (n < nn) b[u][n] = B[(cu * tb + n) * 64];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (c + (size_t)u < c1)
#pragma unroll
                for (int n = 0; n < 4; n++)
                    if (n < nn) acc[n] = mfma16(a[u], b[u][n], acc[n]);
    }
    float* out = part + (size_t)split * NET_PARAMS + off;
#pragma unroll
    for (int n = 0; n < 4; n++)
        if (n < nn)
#pragma unroll
            for (int r = 0; r < 4; r++) out[(16 * mt + 4 * q + r) * ld + 16 * (nt + n) + col] = acc[n][r];
}

/* Adam's constants of one step (Kingma & Ba, 2015); update = 0: gradients only */
struct AdamStep {
    int update;
    float lr, b1, b2, eps, c1, c2;
};

/* the [out][in] index of parameter i, or -1 where no bf16 [out][in] copy is kept (biases) */
__device__ __forceinline__ int net_transposed(int i)
{
    if (i < NET_B1) return NET_W1 + (i % MLP_H) * MLP_IN + i / MLP_H;
    if (i >= NET_W2 && i < NET_B2) return NET_W2 + ((i - NET_W2) % MLP_H) * MLP_H + (i - NET_W2) / MLP_H;
    if (i >= NET_W3 && i < NET_B3) return NET_W3 + ((i - NET_W3) % MLP_OUT) * MLP_H + (i - NET_W3) / MLP_OUT;
    return -1;
}

/* Gradients: a weight's is its splits' partials added in order (blocks of 256 weights), a bias's
 * the tree sum of its 256 columns' sums (a block each, after those); with a.update the Adam update
 * of fp32 master weights w and their bf16 copies. Block 0 also adds the loss partials (in double). */
__global__ LAUNCH_BOUNDS_256 void k_net_reduce(const float* __restrict__ part, int splits,
                                               const float* __restrict__ bpart, const float* __restrict__ lpart,
                                               int lparts, float* __restrict__ grads, float* __restrict__ loss,
                                               AdamStep a, float* __restrict__ w, float* __restrict__ m,
                                               float* __restrict__ v, __bf16* __restrict__ wb, __bf16* __restrict__ wt)
{
    __shared__ float red[256];
    const int t = threadIdx.x, nw = (NET_PARAMS + 255) / 256;
    int i = (int)blockIdx.x * 256 + t;
    float gi;
    if ((int)blockIdx.x < nw) {
        if (blockIdx.x == 0 && t < 64 && loss) {
            double d = 0.0;
            for (int p = t; p < lparts; p += 64) d += lpart[p];
            for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o);
            if (t == 0) *loss = (float)d;
        }
        const bool bias = (i >= NET_B1 && i < NET_W2) || (i >= NET_B2 && i < NET_W3) || i >= NET_B3;
        if (bias) return;
        gi = part[i];
        for (int p = 1; p < splits; p++) gi += part[(size_t)p * NET_PARAMS + i];
    } else {
        const int b = (int)blockIdx.x - nw;
        red[t] = bpart[(size_t)t * NET_BIASES + b];
        __syncthreads();
        for (int k = 128; k > 0; k >>= 1) {
            if (t < k) red[t] += red[t + k];
            __syncthreads();
        }
        if (t != 0) return;
        gi = red[0];
        i = b < MLP_H ? NET_B1 + b : b < 2 * MLP_H ? NET_B2 + b - MLP_H : NET_B3 + b - 2 * MLP_H;
    }
    grads[i] = gi;
    if (!a.update) return;
    const float mi = a.b1 * m[i] + (1.0f - a.b1) * gi;
    const float vi = a.b2 * v[i] + (1.0f - a.b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float x = w[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
    w[i] = x;
    wb[i] = to_bf16(x);
    const int j = net_transposed(i);
    if (j >= 0) wt[j] = to_bf16(x);
}

/* the bf16 copies of the fp32 weights: wb as they are, wt the matrices in [out][in] order */
__global__ LAUNCH_BOUNDS_256 void k_net_weights(const float* __restrict__ w, __bf16* __restrict__ wb,
                                                __bf16* __restrict__ wt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NET_PARAMS) return;
    wb[i] = to_bf16(w[i]);
    const int j = net_transposed(i);
    if (j >= 0) wt[j] = to_bf16(w[i]);
}

/* W [K x N] fp32 row-major -> fragment layout (ntile, kchunk, col, k) in bf16 */
/* Fragment kk of chunk kc, column col of tile nt takes W[k][n] with k = 32 kc + kk, or with
 * perm the row whose neuron the previous layer's result leaves at that position:
 * nu(32 kc + 8 q + e) = 32 kc + (e < 4 ? 4 q + e : 16 + 4 q + e - 4). */
__global__ LAUNCH_BOUNDS_256 void k_pack_frag(const float* __restrict__ W, int K, int N, __bf16* __restrict__ F,
                                              int perm)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= K * N) return;
    const int k = i / N, n = i % N;
    const int nt = n / 16, col = n % 16, kc = k / 32;
    int kk = k % 32;
    if (perm) {
        /* the inverse of nu inside the chunk: neuron offset o = kk -> position 8 q + e */
        const int o = kk, hi = o >= 16 ? 1 : 0, rem = o - 16 * hi;
        kk = 8 * (rem / 4) + 4 * hi + rem % 4;
    }
    F[(((size_t)nt * (K / 32) + kc) * 16 + col) * 32 + kk] = to_bf16(W[i]);
}
