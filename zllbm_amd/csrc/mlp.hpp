// mlp.hpp -- learned sub-grid closure: a 9 -> 32 -> 32 -> 1 MLP (SiLU, softplus) predicting the
// eddy viscosity from local non-equilibrium invariants.  No counterpart in the reference; it
// replaces the Smagorinsky relaxation time (les_models/lbm_les_smagorinsky.cpp:22-94) where its
// inputs lie inside the training range and falls back to Smagorinsky elsewhere.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>
#include <type_traits>

namespace zlh {

constexpr int kMlpF = 9;
constexpr int kMlpH = 32;
constexpr int kMlpParams = kMlpH * kMlpF + kMlpH + kMlpH * kMlpH + kMlpH + kMlpH + 1;   // 1409

// Output row held in accumulator r by lanes of half h (lane / 32) of a 32x32 MFMA result
// (v_mfma_f32_32x32x16_bf16: lane l holds C[i][l % 32] for i = 8 (r / 4) + 4 h + r % 4).
__host__ __device__ constexpr int mfma_row(int h, int r) { return (r >> 2) * 8 + h * 4 + (r & 3); }

// Per-lane operand images of the wavefront MFMA network, as BF16 and as FP16 bit patterns (built
// on the host; w1a/w2a BF16, h1a/h2a the same entries in FP16):
//   w1a[l][e]    = layer-1 A operand, K slot k = 8 (l / 32) + e of row l % 32: W1[l % 32][k] for
//                  the 9 features, b1[l % 32] in slot 9 (its B slot holds 1), zero above
//   w2a[s][l][e] = layer-2 A operand, K step s < 2: W2[l % 32][mfma_row(l / 32, 8 s + e)] (the
//                  layer-1 accumulator order, so activations stay in their registers)
//   w3r[h][r]    = w3[mfma_row(h, r)] (FP32)
//   b2r[h][r]    = b2[mfma_row(h, r)] (FP32): the layer-2 accumulators start from it
// plus the input normalisation, training range, output scale and b3, so that the fused kernel
// reads nothing of the network from global memory after its first store; and the operand images
// of the MRT moment transform on the matrix cores (moments_mfma, populations_mfma):
//   mfwd[s][l] = M[l % 32][2 s + l / 32]   (moment row, population column; zero outside Q x Q)
//   mbwd[s][l] = M[2 s + l / 32][l % 32]   (M^T)
constexpr int kMrtSteps = 10;   // K steps of two: (19 + 1) / 2 for D3Q19, 5 used for D2Q9
struct alignas(16) MlpOps {
    uint16_t w1a[64][8];
    uint16_t w2a[2][64][8];
    uint16_t h1a[64][8];
    uint16_t h2a[2][64][8];
    float w3r[2][16];
    float b2r[2][16];
    float mean[kMlpF];
    float inv_std[kMlpF];
    float fmin[kMlpF];
    float fmax[kMlpF];
    float nu_scale;
    float b3;
    float pad[2];
    float mfwd[kMrtSteps][64];   // last: only the kernels with the transform on the matrix cores stage them
    float mbwd[kMrtSteps][64];
};

// device-resident closure: operand images, parameters (flat order W1, b1, W2, b2, w3, b3), input
// normalisation, training range of the raw features and the output scale
struct MlpDev {
    MlpOps ops;
    float p[kMlpParams];
    float mean[kMlpF];
    float inv_std[kMlpF];
    float fmin[kMlpF];
    float fmax[kMlpF];
    float nu_scale;
};

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + __expf(-z)); }
__device__ __forceinline__ float softplusf_(float z) { return z > 20.f ? z : log1pf(__expf(z)); }

// 1 / x: exact division in FP64; in FP32 the hardware reciprocal (about 1 ulp, one instruction
// where the IEEE-rounded division takes about ten)
template <typename C>
__device__ __forceinline__ C recip(C x) {
    if constexpr (std::is_same<C, float>::value) return __builtin_amdgcn_rcpf(x);
    else return C(1) / x;
}

// square root: correctly rounded in FP64; in FP32 the hardware square root (about 1 ulp, one
// instruction where the correctly rounded sqrtf takes about fifteen)
template <typename C>
__device__ __forceinline__ C root(C x) {
    if constexpr (std::is_same<C, float>::value) return __builtin_amdgcn_sqrtf(x);
    else return sqrt(x);
}

// raw closure inputs from the non-equilibrium stress Pi (xx, yy, zz, xy, xz, yz), density and
// velocity: P = Pi / rho, a = sqrt(2 P:P), I1 = tr P, I2 = (I1^2 - P:P) / 2, I3 = det P, |u|^2,
// rho - 1, tau0, a tau0, a^2
template <typename C>
__device__ __forceinline__ void closure_features(const C *pi, C rho, C drho, const C *u, C tau0, float *x) {
    const C ir = recip(rho);
    const C pxx = pi[0] * ir, pyy = pi[1] * ir, pzz = pi[2] * ir, pxy = pi[3] * ir, pxz = pi[4] * ir, pyz = pi[5] * ir;
    const C pp = pxx * pxx + pyy * pyy + pzz * pzz + C(2) * (pxy * pxy + pxz * pxz + pyz * pyz);
    const C a = root(C(2) * pp);
    const C i1 = pxx + pyy + pzz;
    const C i2 = C(0.5) * (i1 * i1 - pp);
    const C i3 = pxx * (pyy * pzz - pyz * pyz) - pxy * (pxy * pzz - pyz * pxz) + pxz * (pxy * pyz - pyy * pxz);
    x[0] = float(a);
    x[1] = float(i1);
    x[2] = float(i2);
    x[3] = float(i3);
    x[4] = float(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    x[5] = float(drho);
    x[6] = float(tau0);
    x[7] = float(a * tau0);
    x[8] = float(a * a);
}

// network output nu_t / nu_scale for normalised inputs (FP32 on the vector units)
__device__ __forceinline__ float mlp_forward(const MlpDev &m, const float *xn) {
    const float *W1 = m.p, *b1 = W1 + kMlpH * kMlpF, *W2 = b1 + kMlpH, *b2 = W2 + kMlpH * kMlpH;
    const float *w3 = b2 + kMlpH, b3 = w3[kMlpH];
    float h1[kMlpH];
#pragma unroll
    for (int j = 0; j < kMlpH; ++j) {
        float z = b1[j];
#pragma unroll
        for (int i = 0; i < kMlpF; ++i) z += W1[j * kMlpF + i] * xn[i];
        h1[j] = z * sigmoidf_(z);
    }
    float out = b3;
#pragma unroll 4
    for (int j = 0; j < kMlpH; ++j) {
        float z = b2[j];
#pragma unroll
        for (int i = 0; i < kMlpH; ++i) z += W2[j * kMlpH + i] * h1[i];
        out += w3[j] * (z * sigmoidf_(z));
    }
    return softplusf_(out);
}

// relaxation-time increment of the closure; Smagorinsky (with the physical tau mode) where any
// raw input lies outside the training range
template <typename C>
__device__ __forceinline__ C mlp_tau_t(const MlpDev &m, const C *pi, C rho, C drho, const C *u, C tau0, C cs18,
                                      bool *fallback) {
    float x[kMlpF];
    closure_features<C>(pi, rho, drho, u, tau0, x);
    bool inside = true;
#pragma unroll
    for (int i = 0; i < kMlpF; ++i) inside = inside && x[i] >= m.fmin[i] && x[i] <= m.fmax[i];
    if (!inside) {
        *fallback = true;
        const C q = root(C(2) * (pi[0] * pi[0] + pi[1] * pi[1] + pi[2] * pi[2] +
                                 C(2) * (pi[3] * pi[3] + pi[4] * pi[4] + pi[5] * pi[5])));
        return C(0.5) * (root(tau0 * tau0 + cs18 * q) - tau0);
    }
    *fallback = false;
    float xn[kMlpF];
#pragma unroll
    for (int i = 0; i < kMlpF; ++i) xn[i] = (x[i] - m.mean[i]) * m.inv_std[i];
    return C(3) * C(m.nu_scale * mlp_forward(m, xn));
}

// ---------------------------------------------------------------------------------------------
// FP32 solver: the network of 64 nodes (one per lane) as matrix-core products with BF16 or FP16
// operands and FP32 accumulation.  Layer l computes H_l^T [32 x 64 nodes] = W_l [32 x K] *
// H_{l-1}^T in two 32-node column blocks; every lane of the wavefront must call it (EXEC all
// ones).  v_mfma_f32_32x32x16_bf16 and _f16 share one lane layout.
// ---------------------------------------------------------------------------------------------
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// kernel variants: VAR = 2 sub-grid code + forced (+ kVarMrtMfma); sub-grid codes of the learned
// closure: 2 with BF16 operands, 4 with FP16
constexpr int kVarMrtMfma = 16;   // the FP32 learned-closure kernels' MRT transform on the matrix cores
template <typename C, int VAR>
__host__ __device__ constexpr bool mlp_on_mfma() {
    return std::is_same<C, float>::value && (VAR < 0 || ((VAR & 15) >> 1) == 2 || ((VAR & 15) >> 1) == 4);
}
template <typename C, int VAR>
__host__ __device__ constexpr bool mrt_on_mfma() {
    return VAR >= 0 && (VAR & kVarMrtMfma) != 0 && mlp_on_mfma<C, VAR>();
}

struct OperandsBf16 {
    typedef bf16x8_t vec;
    typedef __bf16 elem;
    static __device__ __forceinline__ vec load(const MlpOps &o, const uint16_t *bits) {
        return __builtin_bit_cast(vec, *reinterpret_cast<const u16x8_t *>(bits));
    }
    static __device__ __forceinline__ const uint16_t *w1(const MlpOps &o, int lane) { return o.w1a[lane]; }
    static __device__ __forceinline__ const uint16_t *w2(const MlpOps &o, int s, int lane) { return o.w2a[s][lane]; }
    static __device__ __forceinline__ f32x16_t mfma(vec a, vec b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
struct OperandsF16 {
    typedef f16x8_t vec;
    typedef _Float16 elem;
    static __device__ __forceinline__ vec load(const MlpOps &o, const uint16_t *bits) {
        return __builtin_bit_cast(vec, *reinterpret_cast<const u16x8_t *>(bits));
    }
    static __device__ __forceinline__ const uint16_t *w1(const MlpOps &o, int lane) { return o.h1a[lane]; }
    static __device__ __forceinline__ const uint16_t *w2(const MlpOps &o, int s, int lane) { return o.h2a[s][lane]; }
    static __device__ __forceinline__ f32x16_t mfma(vec a, vec b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

// SiLU of the matrix-core form, on pre-activations scaled by c = -log2(e) (the host scales W1, b1
// and b2 in the operand images): for t = c z, t / (1 + 2^t) = c silu(z).  Hardware exp2 and
// reciprocal, about 1 ulp each, far below the operands' rounding; a large t gives 2^t -> inf,
// rcp -> 0.  The next layer takes the scaled activations as they are (its weights are unscaled;
// the output weights carry 1/c).
constexpr double kSiluScale = -1.4426950408889634;
__device__ __forceinline__ float silu_scaled(float t) {
    return t * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(t));
}

// softplus of the matrix-core form: max(z, 0) + ln 2 log2(1 + 2^(-|z| log2 e)) with the hardware
// exp2 and log2 (about 1 ulp each).  Rounding 1 + e to FP32 costs at most 2^-24 absolute where
// e is small, far below the operands' rounding; the library log1pf takes about 110 instructions.
__device__ __forceinline__ float softplus_fast(float z) {
    const float e = __builtin_amdgcn_exp2f(-1.4426950408889634f * __builtin_fabsf(z));
    return __builtin_fmaxf(z, 0.f) + 0.6931471805599453f * __builtin_amdgcn_logf(1.f + e);
}

// The MRT moment transform m = M f and its inverse f = M^T y as batched 19 x 19 contractions on
// the matrix cores (v_mfma_f32_32x32x2f32, FP32 operands, products exact, FP32 sums): the 64 nodes
// of the wavefront are two 32-node column blocks, a K step takes populations 2s and 2s + 1.  The
// B operand of block 0 holds population 2s of node l (lanes 0..31) and 2s + 1 of node l - 32
// (lanes 32..63); block 1 the same for nodes 32..63: v_permlane32_swap(f[2s], f[2s + 1]) gives
// both.  The results (rows in the accumulator order of a 32 x 32 product) return to one node per
// lane by v_permlane32_swap(block 0, block 1) of each accumulator register: then register r of
// the first result holds row 8 (r / 4) + r % 4 and of the second row 8 (r / 4) + 4 + r % 4.
// Every lane of the wavefront must call them (EXEC all ones).
__device__ __forceinline__ constexpr int mrt_reg(int k) { return 4 * (k >> 3) + (k & 3); }
__device__ __forceinline__ constexpr bool mrt_upper(int k) { return (k & 4) != 0; }

template <int Q>
__device__ __forceinline__ void rows_to_lanes(const f32x16_t &d0, const f32x16_t &d1, float (&out)[Q]) {
    float lo[16], hi[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        // only the registers that carry rows below Q
        const bool need = 8 * (r >> 2) + (r & 3) < Q;
        if (!need) { lo[r] = hi[r] = 0.f; continue; }
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(d0[r]), __float_as_uint(d1[r]), false, false);
        lo[r] = __uint_as_float(s[0]);
        hi[r] = __uint_as_float(s[1]);
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) out[k] = mrt_upper(k) ? hi[mrt_reg(k)] : lo[mrt_reg(k)];
}

template <int Q>
__device__ __forceinline__ void contract_mfma(const float (&x)[Q], const float (*a)[64], float (&out)[Q]) {
    constexpr int NK = (Q + 1) / 2;
    static_assert(NK <= kMrtSteps, "transform operand images cover the lattice");
    const int lane = __lane_id();
    f32x16_t d0 = {}, d1 = {};
#pragma unroll
    for (int s = 0; s < NK; ++s) {
        const float lo = x[2 * s];
        const float hi = 2 * s + 1 < Q ? x[2 * s + 1] : 0.f;
        const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
        const float av = a[s][lane];
        d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(av, __uint_as_float(b[0]), d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(av, __uint_as_float(b[1]), d1, 0, 0, 0);
    }
    rows_to_lanes<Q>(d0, d1, out);
}

// m = M f of this lane's node (shifted populations give shifted moments)
template <int Q>
__device__ __forceinline__ void moments_mfma(const MlpOps &o, const float (&f)[Q], float (&m)[Q]) {
    contract_mfma<Q>(f, o.mfwd, m);
}
// f = M^T y of this lane's node
template <int Q>
__device__ __forceinline__ void populations_mfma(const MlpOps &o, const float (&y)[Q], float (&f)[Q]) {
    contract_mfma<Q>(y, o.mbwd, f);
}

// value held by lane l ^ 32 (v_permlane32_swap exchanges the halves of a register pair; unlike
// ds_bpermute it is no LDS instruction, so it never waits on direct-to-LDS loads in flight)
__device__ __forceinline__ float swap_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(__lane_id() < 32 ? r[1] : r[0]);
}

// network output (nu_t / nu_scale) of this lane's normalised inputs; o may live in LDS
template <typename OT>
__device__ __forceinline__ float mlp_forward_wave(const MlpOps &o, const float *xn, float b3) {
    typedef typename OT::vec vec;
    typedef typename OT::elem elem;
    const int lane = __lane_id();
    const int h = lane >> 5;
    // layer-1 B operands: column block 0 = nodes 0..31, block 1 = nodes 32..63; lane l carries
    // K slots 8 h .. 8 h + 7 of node l % 32 (block 0) or 32 + l % 32 (block 1); slot 9 = 1 (bias).
    // Slot e takes feature e in the lower half and t_e (feature 8, the bias 1, zeros) in the upper
    // half: v_permlane32_swap(xn[e], t_e) leaves exactly block 0's operand in the first register
    // and block 1's in the second.
    vec x0, x1;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float t = e == 0 ? xn[8] : (e == 1 ? 1.f : 0.f);
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(xn[e]), __float_as_uint(t), false, false);
        x0[e] = (elem)__uint_as_float(r[0]);
        x1[e] = (elem)__uint_as_float(r[1]);
    }
    const f32x16_t zero = {};
    f32x16_t z0, z1;
    {
        const vec a1 = OT::load(o, OT::w1(o, lane));
        z0 = OT::mfma(a1, x0, zero);
        z1 = OT::mfma(a1, x1, zero);
    }
    // SiLU; accumulator r of this lane is hidden unit mfma_row(h, r), which is also the K slot
    // 8 h + r % 8 of layer-2 K step r / 8, so the activations stay in place
    vec g0[2], g1[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        g0[r >> 3][r & 7] = (elem)silu_scaled(z0[r]);
        g1[r >> 3][r & 7] = (elem)silu_scaled(z1[r]);
    }
    // layer 2: the accumulators start from the (FP32, scaled) bias of their rows
    f32x16_t y0, y1;
#pragma unroll
    for (int r = 0; r < 16; ++r) y0[r] = y1[r] = o.b2r[h][r];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        const vec a2 = OT::load(o, OT::w2(o, st, lane));
        y0 = OT::mfma(a2, g0[st], y0);
        y1 = OT::mfma(a2, g1[st], y1);
    }
    float p0 = 0.f, p1 = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float ww = o.w3r[h][r];
        p0 += ww * silu_scaled(y0[r]);
        p1 += ww * silu_scaled(y1[r]);
    }
    // node l % 32 + 32 h sums the two halves of its block: after v_permlane32_swap(p0, p1) the
    // lower lanes hold block 0's halves (p0 of lanes l and l + 32) and the upper lanes block 1's
    const auto pr = __builtin_amdgcn_permlane32_swap(__float_as_uint(p0), __float_as_uint(p1), false, false);
    return softplus_fast(__uint_as_float(pr[0]) + __uint_as_float(pr[1]) + b3);
}

// mlp_tau_t for the FP32 solver, evaluated by the whole wavefront
template <typename OT>
__device__ __forceinline__ float mlp_tau_t_wave(const MlpOps &o, const float *pi, float rho, float drho,
                                                const float *u, float tau0, float cs18) {
    float x[kMlpF], xn[kMlpF];
    closure_features<float>(pi, rho, drho, u, tau0, x);
    bool inside = true;
#pragma unroll
    for (int i = 0; i < kMlpF; ++i) {
        inside = inside && x[i] >= o.fmin[i] && x[i] <= o.fmax[i];
        xn[i] = (x[i] - o.mean[i]) * o.inv_std[i];
    }
    const float net = mlp_forward_wave<OT>(o, xn, o.b3);
    // the Smagorinsky fallback only where some lane of the wavefront needs it
    float smag = 0.f;
    if (__ballot(!inside)) {
        const float q = root(2.f * (pi[0] * pi[0] + pi[1] * pi[1] + pi[2] * pi[2] +
                                    2.f * (pi[3] * pi[3] + pi[4] * pi[4] + pi[5] * pi[5])));
        smag = 0.5f * (root(tau0 * tau0 + cs18 * q) - tau0);
    }
    return inside ? 3.f * o.nu_scale * net : smag;
}

// copy of the operand images into LDS by one workgroup (followed by a barrier)
// Copies into LDS the parts of the operand images a kernel reads: one operand form's network
// images (BF16 w1a, w2a or FP16 h1a, h2a), the scalars, and with MRT the transform's images; the
// other parts of dst stay unwritten and are never read.
template <bool FP16, bool MRT>
__device__ __forceinline__ void stage_mlp_ops(MlpOps &dst, const MlpOps &src) {
    static_assert(sizeof(MlpOps) % 16 == 0 && offsetof(MlpOps, w3r) % 16 == 0 && offsetof(MlpOps, mfwd) % 16 == 0,
                  "operand images are copied in 16-byte units");
    static_assert(offsetof(MlpOps, w2a) == offsetof(MlpOps, w1a) + sizeof(src.w1a) &&
                  offsetof(MlpOps, h2a) == offsetof(MlpOps, h1a) + sizeof(src.h1a), "each form's images are adjacent");
    constexpr int img0 = (int)((FP16 ? offsetof(MlpOps, h1a) : offsetof(MlpOps, w1a)) / 16);
    constexpr int nimg = (int)((sizeof(src.w1a) + sizeof(src.w2a)) / 16);
    constexpr int sc0 = (int)(offsetof(MlpOps, w3r) / 16);
    constexpr int nsc = (int)(((MRT ? sizeof(MlpOps) : offsetof(MlpOps, mfwd)) - offsetof(MlpOps, w3r)) / 16);
    const uint4 *s = reinterpret_cast<const uint4 *>(&src);
    uint4 *d = reinterpret_cast<uint4 *>(&dst);
    for (int i = threadIdx.x; i < nimg + nsc; i += blockDim.x) {
        const int j = i < nimg ? img0 + i : sc0 + (i - nimg);
        d[j] = s[j];
    }
    __syncthreads();
}

// batch inference on the MFMA network (FP32 solver form); every lane runs, inactive ones on zeros
template <typename OT>
__global__ __launch_bounds__(256) void k_mlp_eval_wave(const MlpDev *m, const float *X, int64_t n, float *y) {
    __shared__ MlpOps ops;
    stage_mlp_ops<std::is_same<OT, OperandsF16>::value, false>(ops, m->ops);
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float xn[kMlpF];
    for (int i = 0; i < kMlpF; ++i) xn[i] = k < n ? X[k * kMlpF + i] : 0.f;
    const float out = mlp_forward_wave<OT>(ops, xn, ops.b3);
    if (k < n) y[k] = out;
}

// ---------------------------------------------------------------------------------------------
// training: gradient kernels, their reduction, and the Adam update over the flat parameter vector.
// A gradient workgroup writes the sums of its samples as one row of `part` ([workgroup][kGradRow]:
// the gradient in parameter order, then the loss); k_grad_reduce adds the rows in workgroup order,
// so a gradient depends on its inputs alone (no floating-point atomics between workgroups) and no
// accumulator has to be cleared first.
// ---------------------------------------------------------------------------------------------
constexpr int kGradRow = 1412;       // kMlpParams + 1, rounded up to 16 bytes
// Rows: one workgroup per CU, which loops over a larger batch.  The gradient kernels' registers (291 and
// 323 of a SIMD's 512) leave one wavefront per SIMD, so a second workgroup would only queue behind the
// first.  256 rows against 512, us: FP32 17.2 / 21.6 on 65,536 samples, 27.9 / 31.9 on 131,072, 174.7 / 178.7
// on 2^20; BF16 operands 15.3 / 15.5, 21.0 / 27.8, 94.7 / 100.2.
constexpr int kGradMaxBlocks = 256;
static_assert(kGradRow >= kMlpParams + 1, "a row holds the gradient and the loss");

__device__ __forceinline__ float wave_sum_f(float v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ uint32_t hash32(uint32_t x) {
    x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
    return x;
}

// sample k of a batch: k itself, or with `random` (hash(seed, k) mod n); n <= 2^26
__device__ __forceinline__ int64_t batch_sample(int k, uint32_t seed, int random, int64_t n) {
    return random ? (int64_t)(hash32(seed * 2654435761u + (uint32_t)k) % (uint32_t)n) : (int64_t)k;
}

__device__ __forceinline__ float dsilu(float z, float sg) { return sg * (1.f + z * (1.f - sg)); }

// orders a wavefront's LDS writes before its later LDS reads of other lanes' values
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Gradient of mean((softplus(net(x)) - t)^2) in FP32: products and sums of every layer as
// v_mfma_f32_32x32x2f32 (exact FP32 products, FP32 accumulation), activations in FP32.  A
// wavefront takes 32 samples, one per column; lane l = 32 h + c holds rows mfma_row(h, r) of
// column c.
//   forward    H^T[32 x 32 samples] = W . (...)^T: K step r of layer 2 takes units mfma_row(0, r)
//              and mfma_row(1, r), so that accumulators feed the next product from their registers;
//              the accumulators start from the biases
//   backward   D1^T = W2^T . D2 the same way
//   gradients  dW2 = D2 . H1^T and [dW1 | db1] = D1 . [X | 1] contract over the samples: both
//              operands are turned around through a per-wavefront LDS tile (row stride 36 floats:
//              16-byte reads of a row's half); the bias and output-weight gradients are the row
//              sums of the same reads
// 69 products of 64 cycles per 32 samples.  A batch of 4,096 takes 10.8 us (32 workgroups, bound by
// the latency of one tile) and 2^20 samples 175 us (6.0 G samples/s).  The products fill the matrix
// pipe for a third of that; the SiLU arithmetic on the vector units and the turns through LDS take the
// rest, which one wavefront per SIMD does not overlap.  One sample per lane with a wavefront reduction and
// an atomic per parameter (1,409 of each) took 403 us and 8.4 ms.
constexpr int kTileStride = 36;
struct alignas(16) GradTilesF {
    float d[kMlpH][kTileStride];     // layer delta [hidden][sample]: D2, then D1
    float h[kMlpH][kTileStride];     // layer-1 activations [hidden][sample], then dz3 h2
    float x[kMlpF][kTileStride];     // inputs [feature][sample]
};

__global__ __launch_bounds__(256) void k_mlp_grad(const float *__restrict__ params, const float *__restrict__ X,
                                                  const float *__restrict__ T, int64_t n, int batch, uint32_t seed,
                                                  int random, float *__restrict__ part) {
    __shared__ union {
        GradTilesF tiles[4];
        float sums[4][kGradRow];   // after the loop
    } sh;
    const int lane = __lane_id(), h = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    GradTilesF &tl = sh.tiles[wave];
    const float *W1 = params, *b1 = W1 + kMlpH * kMlpF, *W2 = b1 + kMlpH, *b2 = W2 + kMlpH * kMlpH;
    const float *w3 = b2 + kMlpH;
    // A operands: row `col` of W1 (K slots 2 s + h), of W2 and of W2^T (K slots mfma_row(h, r))
    float a1[5], a2[16], at[16], w3r[16];
    f32x16_t z1_0, z2_0;
#pragma unroll
    for (int s = 0; s < 5; ++s) a1[s] = 2 * s + h < kMlpF ? W1[col * kMlpF + 2 * s + h] : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = mfma_row(h, r);
        a2[r] = W2[col * kMlpH + row];
        at[r] = W2[row * kMlpH + col];
        w3r[r] = w3[row];
        z1_0[r] = b1[row];
        z2_0[r] = b2[row];
    }
    const float b3 = w3[kMlpH];
    const float inv_b = 1.f / (float)batch;
    f32x16_t gw2 = {}, gw1 = {};
    float gw3 = 0.f, gb2 = 0.f, gb3 = 0.f, lsum = 0.f;
    // columns past the batch carry zero inputs and a zero output delta, so they add nothing
    for (int64_t base = (int64_t)blockIdx.x * 128 + wave * 32; base < batch; base += (int64_t)gridDim.x * 128) {
        const int64_t k = base + col;
        const bool active = k < batch;
        const int64_t s = active ? batch_sample((int)k, seed, random, n) : 0;
        float xv[5];
#pragma unroll
        for (int e = 0; e < 5; ++e) xv[e] = active && 2 * e + h < kMlpF ? X[s * kMlpF + 2 * e + h] : 0.f;
        const float t = active ? T[s] : 0.f;
        f32x16_t z1 = z1_0;
#pragma unroll
        for (int e = 0; e < 5; ++e) z1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[e], xv[e], z1, 0, 0, 0);
        float s1[16], g1[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s1[r] = sigmoidf_(z1[r]);
            g1[r] = z1[r] * s1[r];
            tl.h[mfma_row(h, r)][col] = g1[r];
        }
#pragma unroll
        for (int e = 0; e < 5; ++e)
            if (2 * e + h < kMlpF) tl.x[2 * e + h][col] = xv[e];
        f32x16_t z2 = z2_0;
#pragma unroll
        for (int r = 0; r < 16; ++r) z2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[r], g1[r], z2, 0, 0, 0);
        float s2[16], p = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s2[r] = sigmoidf_(z2[r]);
            p += w3r[r] * (z2[r] * s2[r]);
        }
        // both halves of a column hold the sample's output
        const float z3 = b3 + (p + swap_halves(p));
        const float y = softplusf_(z3);
        const float dz3 = active ? 2.f * (y - t) * inv_b * sigmoidf_(z3) : 0.f;
        if (h == 0) {
            lsum += active ? (y - t) * (y - t) * inv_b : 0.f;
            gb3 += dz3;
        }
        float d2[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            d2[r] = dz3 * w3r[r] * dsilu(z2[r], s2[r]);
            tl.d[mfma_row(h, r)][col] = d2[r];
        }
        wave_lds_sync();
        // row `col`, samples 16 h .. 16 h + 15 (K slot t of both operands is sample 16 h + t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 A = *reinterpret_cast<const float4 *>(&tl.d[col][16 * h + 4 * q]);
            const float4 B = *reinterpret_cast<const float4 *>(&tl.h[col][16 * h + 4 * q]);
            gb2 += (A.x + A.y) + (A.z + A.w);
            gw2 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.x, B.x, gw2, 0, 0, 0);
            gw2 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.y, B.y, gw2, 0, 0, 0);
            gw2 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.z, B.z, gw2, 0, 0, 0);
            gw2 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.w, B.w, gw2, 0, 0, 0);
        }
        f32x16_t e1 = {};
#pragma unroll
        for (int r = 0; r < 16; ++r) e1 = __builtin_amdgcn_mfma_f32_32x32x2f32(at[r], d2[r], e1, 0, 0, 0);
        wave_lds_sync();   // D2 and H1 read by every lane before others take their place
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            tl.d[mfma_row(h, r)][col] = e1[r] * dsilu(z1[r], s1[r]);
            tl.h[mfma_row(h, r)][col] = dz3 * (z2[r] * s2[r]);
        }
        wave_lds_sync();
        const int xr = col < kMlpF ? col : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 A = *reinterpret_cast<const float4 *>(&tl.d[col][16 * h + 4 * q]);
            const float4 H = *reinterpret_cast<const float4 *>(&tl.h[col][16 * h + 4 * q]);
            const float4 V = *reinterpret_cast<const float4 *>(&tl.x[xr][16 * h + 4 * q]);
            const float o = col == kMlpF ? 1.f : 0.f;   // column 9: the bias; columns 10..31: zero
            const bool in = col < kMlpF;
            gw3 += (H.x + H.y) + (H.z + H.w);
            gw1 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.x, in ? V.x : o, gw1, 0, 0, 0);
            gw1 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.y, in ? V.y : o, gw1, 0, 0, 0);
            gw1 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.z, in ? V.z : o, gw1, 0, 0, 0);
            gw1 = __builtin_amdgcn_mfma_f32_32x32x2f32(A.w, in ? V.w : o, gw1, 0, 0, 0);
        }
        wave_lds_sync();   // tiles read before the next samples overwrite them
    }
    __syncthreads();   // every wavefront is done with its tile
    float *S = sh.sums[wave];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = mfma_row(h, r);
        S[kMlpH * kMlpF + kMlpH + row * kMlpH + col] = gw2[r];
        if (col <= kMlpF) S[col < kMlpF ? row * kMlpF + col : kMlpH * kMlpF + row] = gw1[r];
    }
    gb2 += swap_halves(gb2);
    gw3 += swap_halves(gw3);
    gb3 = wave_sum_f(gb3);
    lsum = wave_sum_f(lsum);
    constexpr int kB2 = kMlpH * kMlpF + kMlpH + kMlpH * kMlpH;
    if (h == 0) {
        S[kB2 + col] = gb2;
        S[kB2 + kMlpH + col] = gw3;
    }
    if (lane == 0) {
        S[kMlpParams - 1] = gb3;
        S[kMlpParams] = lsum;
    }
    __syncthreads();
    for (int i = threadIdx.x; i <= kMlpParams; i += blockDim.x)
        part[(int64_t)blockIdx.x * kGradRow + i] = (sh.sums[0][i] + sh.sums[1][i]) + (sh.sums[2][i] + sh.sums[3][i]);
}

// Sum over the `rows` rows of part: gradient to grad and loss to loss (either may be null), and
// with ADAM the update of the parameters.  A workgroup takes 32 parameters, 8 groups of threads a
// share of the rows each.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_grad_reduce(const float *__restrict__ part, int rows, float *__restrict__ grad,
                                                     float *__restrict__ loss, float *params, float *m, float *v,
                                                     float lr, float b1, float b2, float eps, int t) {
    __shared__ float sh[8][32];
    const int c = threadIdx.x & 31, grp = threadIdx.x >> 5;
    const int i = blockIdx.x * 32 + c;
    float acc = 0.f;
    if (i <= kMlpParams) {
#pragma unroll 4
        for (int b = grp; b < rows; b += 8) acc += part[(int64_t)b * kGradRow + i];
    }
    sh[grp][c] = acc;
    __syncthreads();
    if (grp != 0 || i > kMlpParams) return;
    const float g = ((sh[0][c] + sh[1][c]) + (sh[2][c] + sh[3][c])) + ((sh[4][c] + sh[5][c]) + (sh[6][c] + sh[7][c]));
    if (i == kMlpParams) {
        if (loss) *loss = g;
        return;
    }
    if (grad) grad[i] = g;
    if constexpr (ADAM) {
        const float mi = b1 * m[i] + (1.f - b1) * g;
        const float vi = b2 * v[i] + (1.f - b2) * g * g;
        m[i] = mi;
        v[i] = vi;
        const float mh = mi / (1.f - powf(b1, (float)t));
        const float vh = vi / (1.f - powf(b2, (float)t));
        params[i] -= lr * mh / (sqrtf(vh) + eps);
    }
}

// ---------------------------------------------------------------------------------------------
// The gradient with BF16 operands: forward and backward of 64 samples per wavefront as
// v_mfma_f32_32x32x16_bf16 with FP32 accumulation.  Same gradient, batch selection and loss as
// k_mlp_grad.  The forward has mlp_forward_wave's layout without the SiLU scaling (the parameters
// change every step, so the operands are rounded here from FP32); the accumulators of layer 2
// start from its rounded bias.  The weight gradients contract over samples, which sit on lanes,
// so the backward turns the layer deltas and activations around through LDS:
//   dW2 [32 x 32]        = D2 [32 x 64 samples] . H1^T     4 K steps of 16 samples
//   D1^T [32 x 64]       = W2^T . D2                       D2 kept in accumulator order, as the
//                                                          forward keeps H1 for layer 2
//   [dW1 | db1] [32 x 10] = D1 [32 x 64] . [X | 1]          4 K steps; column 9 is the bias
// Rounded to BF16: X, W1, b1, W2, b2, H1, D2 (as operand of both products) and D1.  db2, dw3,
// db3 and the loss accumulate per lane in FP32 from unrounded values and are summed over the
// lanes once, through the tile.  A wavefront keeps its sums over all the batches it takes; its
// tile is its own, so only the closing sum over the workgroup's wavefronts takes a barrier.  Bound
// by the latency of a tile at one wavefront per SIMD: 70,000 samples (two trips of the grid) take
// 24 us, where four barriers a tile and LDS atomics of 32 lanes to one address in the closing sum
// took 44.5; 2^20 samples take 95 us (122.7).
// ---------------------------------------------------------------------------------------------
constexpr int kGradTileStride = 72;   // LDS row stride of the transposed tiles, BF16 elements (144 B)

struct alignas(16) GradTiles {
    __bf16 d[kMlpH][kGradTileStride];   // layer delta [hidden][sample]: D2, then D1
    __bf16 h[kMlpH][kGradTileStride];   // layer-1 activations [hidden][sample]
    __bf16 x[16][kGradTileStride];      // inputs [feature][sample]; row 9 = 1, rows 10..15 = 0
};

// row sums over the 32 lanes of a half and both halves: v[r] of lane 32 h + c belongs to row
// mfma_row(h, r); returns the sum of row `col`, the same in both halves.  buf: [32][kTileStride]
// floats of this wavefront.
__device__ __forceinline__ float tile_row_sum(float (*buf)[kTileStride], const float (&v)[16], int h, int col) {
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 16; ++r) buf[mfma_row(h, r)][col] = v[r];
    wave_lds_sync();
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 a = *reinterpret_cast<const float4 *>(&buf[col][16 * h + 4 * q]);
        s += (a.x + a.y) + (a.z + a.w);
    }
    return s + swap_halves(s);
}

__global__ __launch_bounds__(256) void k_mlp_grad_mfma(const float *__restrict__ params, const float *__restrict__ X,
                                                       const float *__restrict__ T, int64_t n, int batch,
                                                       uint32_t seed, int random, float *__restrict__ part) {
    __shared__ union {
        GradTiles tiles[4];
        float sums[4][kGradRow];             // then the wavefronts' sums
    } sh;
    static_assert(sizeof(GradTiles) >= sizeof(float) * kMlpH * kTileStride, "row sums fit a wavefront's tile");
    const int lane = __lane_id(), h = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    GradTiles &tl = sh.tiles[wave];
    for (int r = kMlpF; r < 16; ++r) tl.x[r][lane] = (__bf16)(r == kMlpF ? 1.f : 0.f);
    const float *W1 = params, *b1 = W1 + kMlpH * kMlpF, *W2 = b1 + kMlpH, *b2 = W2 + kMlpH * kMlpH;
    const float *w3 = b2 + kMlpH;
    const float b3 = w3[kMlpH];
    // A operands: row `col` of the weight matrix, K slots 8 h + e (the layout of mlp_forward_wave's operand images)
    bf16x8_t a1, a2[2], at[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = 8 * h + e;
        a1[e] = (__bf16)(k < kMlpF ? W1[col * kMlpF + k] : k == kMlpF ? b1[col] : 0.f);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            a2[st][e] = (__bf16)W2[col * kMlpH + mfma_row(h, 8 * st + e)];
            at[st][e] = (__bf16)W2[mfma_row(h, 8 * st + e) * kMlpH + col];   // W2^T
        }
    }
    float w3r[16];
    f32x16_t z2_0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        w3r[r] = w3[mfma_row(h, r)];
        z2_0[r] = (float)(__bf16)b2[mfma_row(h, r)];
    }
    const float inv_b = 1.f / (float)batch;
    const f32x16_t zero = {};
    f32x16_t gw2 = zero, gw1 = zero;
    float gw3[16], gb2[16], gb3 = 0.f, lsum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) gw3[r] = gb2[r] = 0.f;
    // lanes past the batch carry zero inputs and a zero output delta, so they add nothing
    for (int64_t base = (int64_t)blockIdx.x * 256 + wave * 64; base < batch; base += (int64_t)gridDim.x * 256) {
        const int64_t k = base + lane;
        const bool active = k < batch;
        const int64_t s = active ? batch_sample((int)k, seed, random, n) : 0;
        float xn[kMlpF], px[kMlpF];
#pragma unroll
        for (int i = 0; i < kMlpF; ++i) xn[i] = active ? X[s * kMlpF + i] : 0.f;
        const float t = active ? T[s] : 0.f;
#pragma unroll
        for (int i = 0; i < kMlpF; ++i) {
            px[i] = swap_halves(xn[i]);
            tl.x[i][lane] = (__bf16)xn[i];
        }
        // layer 1: column block c holds samples 32 c .. 32 c + 31 of the wavefront
        bf16x8_t xb[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float hi = e == 1 ? 1.f : 0.f;
            xb[0][e] = (__bf16)(e == 0 ? (h ? px[8] : xn[0]) : (h ? hi : xn[e]));
            xb[1][e] = (__bf16)(e == 0 ? (h ? xn[8] : px[0]) : (h ? hi : px[e]));
        }
        f32x16_t z1[2], z2[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            z1[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, xb[c], zero, 0, 0, 0);
            bf16x8_t g[2];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const __bf16 v = (__bf16)(z1[c][r] * sigmoidf_(z1[c][r]));
                g[r >> 3][r & 7] = v;
                tl.h[mfma_row(h, r)][32 * c + col] = v;
            }
            z2[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2[0], g[0], z2_0, 0, 0, 0);
            z2[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2[1], g[1], z2[c], 0, 0, 0);
        }
        // output, loss and its derivative for this lane's sample (lane l holds sample l)
        float p[2] = {0.f, 0.f}, s2[2][16];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s2[c][r] = sigmoidf_(z2[c][r]);
                p[c] += w3r[r] * z2[c][r] * s2[c][r];
            }
        const float z3 = (h ? p[1] : p[0]) + swap_halves(h ? p[0] : p[1]) + b3;
        const float y = softplusf_(z3);
        const float dz3 = active ? 2.f * (y - t) * inv_b * sigmoidf_(z3) : 0.f;
        lsum += active ? (y - t) * (y - t) * inv_b : 0.f;
        gb3 += dz3;
        // output delta of the samples of this lane's two columns
        const float other = swap_halves(dz3);
        const float d3[2] = {h ? other : dz3, h ? dz3 : other};
        bf16x8_t bd[2][2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                gw3[r] += d3[c] * z2[c][r] * s2[c][r];
                const float dz = d3[c] * w3r[r] * dsilu(z2[c][r], s2[c][r]);
                gb2[r] += dz;
                const __bf16 db = (__bf16)dz;
                bd[c][r >> 3][r & 7] = db;
                tl.d[mfma_row(h, r)][32 * c + col] = db;
            }
        wave_lds_sync();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const bf16x8_t A = *reinterpret_cast<const bf16x8_t *>(&tl.d[col][16 * ks + 8 * h]);
            const bf16x8_t B = *reinterpret_cast<const bf16x8_t *>(&tl.h[col][16 * ks + 8 * h]);
            gw2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B, gw2, 0, 0, 0);
        }
        f32x16_t e1[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            e1[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(at[0], bd[c][0], zero, 0, 0, 0);
            e1[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(at[1], bd[c][1], e1[c], 0, 0, 0);
        }
        wave_lds_sync();   // D2 read by every lane before D1 takes its place
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                tl.d[mfma_row(h, r)][32 * c + col] = (__bf16)(e1[c][r] * dsilu(z1[c][r], sigmoidf_(z1[c][r])));
        wave_lds_sync();
        const int xr = col < 16 ? col : 15;   // columns 16..31 of [X | 1] are zero (row 15)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const bf16x8_t A = *reinterpret_cast<const bf16x8_t *>(&tl.d[col][16 * ks + 8 * h]);
            const bf16x8_t B = *reinterpret_cast<const bf16x8_t *>(&tl.x[xr][16 * ks + 8 * h]);
            gw1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B, gw1, 0, 0, 0);
        }
        wave_lds_sync();   // tiles read before the next samples overwrite them
    }
    float (*buf)[kTileStride] = reinterpret_cast<float (*)[kTileStride]>(&tl);
    const float w3s = tile_row_sum(buf, gw3, h, col), b2s = tile_row_sum(buf, gb2, h, col);
    gb3 = wave_sum_f(gb3);
    lsum = wave_sum_f(lsum);
    __syncthreads();   // every wavefront is done with its tile
    float *S = sh.sums[wave];
    constexpr int kB2 = kMlpH * kMlpF + kMlpH + kMlpH * kMlpH;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = mfma_row(h, r);
        S[kMlpH * kMlpF + kMlpH + row * kMlpH + col] = gw2[r];
        if (col <= kMlpF) S[col < kMlpF ? row * kMlpF + col : kMlpH * kMlpF + row] = gw1[r];
    }
    if (h == 0) {
        S[kB2 + col] = b2s;
        S[kB2 + kMlpH + col] = w3s;
    }
    if (lane == 0) {
        S[kMlpParams - 1] = gb3;
        S[kMlpParams] = lsum;
    }
    __syncthreads();
    for (int i = threadIdx.x; i <= kMlpParams; i += blockDim.x)
        part[(int64_t)blockIdx.x * kGradRow + i] = (sh.sums[0][i] + sh.sums[1][i]) + (sh.sums[2][i] + sh.sums[3][i]);
}

// batch inference (normalised inputs) for tests and evaluation
__global__ void k_mlp_eval(const MlpDev *m, const float *X, int64_t n, float *y) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    float xn[kMlpF];
    for (int i = 0; i < kMlpF; ++i) xn[i] = X[k * kMlpF + i];
    y[k] = mlp_forward(*m, xn);
}

}  // namespace zlh
