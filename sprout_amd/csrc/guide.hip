// BF16 MFMA inference and training kernels of the path-guiding network.
//
// Matrix products run on gfx950's v_mfma_f32_16x16x32_bf16 (64-wide wave,
// FP32 accumulation).  Operand lanes, for lane l, r = l % 16, q = l / 16:
//   A (16 x 16, rows i, depth k): A[r][4q + t], t = 0..3  (x32: A[r][8q + t], t = 0..7)
//   B (16 x 16, depth k, cols j): B[4q + t][r]            (x32: B[8q + t][r])
//   D (16 x 16):                   D[4q + t][r]
// Weights live in LDS as bf16 W^T [out][in] so a forward B operand is one
// 8-byte read; activations as bf16 [row][feature] so an A operand is one
// 8-byte read.
//
// forward   a wave computes 16 queries: the first layer takes its features
//           (sinpi / cospi of f x) straight from registers, two hidden layers
//           pass through LDS, the output layer stores to memory; weights
//           are loaded once per workgroup and the grid strides over tiles.
// gradient  a workgroup of 4 waves takes 64 samples at a time: each wave runs
//           forward and backward for its 16, whose activations and
//           pre-activation gradients also go to LDS transposed; then the 4
//           waves split the 96 16x16 tiles of the weight gradients (depth =
//           the 64 samples) and keep them in registers across all chunks;
//           partial sums per workgroup are reduced in a fixed order, so
//           gradients are deterministic.
// adam      one thread per parameter; refreshes the bf16 W^T copy.

#include "common.hpp"
#include "device_memory.hpp"
#include "guide.hpp"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstddef>
#include <cstring>
#include <vector>

namespace mi {

namespace {

using namespace guide;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// LDS row strides (elements), padded against bank conflicts; multiples of 4
constexpr int S_feat = Feat_pad + 8;  // 232
constexpr int S_hid  = Hidden + 8;    // 72
constexpr int S_out  = Num_out + 8;   // 40

typedef float  f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// fp32 -> bf16, rounded to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t to_bf16(float f) {
    return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

// two bf16 in one word, lo in the low half (one v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    f32x2_t const f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}

__device__ __forceinline__ float from_bf16(uint16_t h) {
    return __uint_as_float(uint32_t(h) << 16);
}

// Orders this wave's LDS accesses (writes by some lanes, reads by others).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

// gfx950's double-depth product: 16 x 16 x 32, each lane supplying eight
// consecutive depth elements.  Lane (r, q) gives A[r][8q + t] and
// B[8q + t][r], t = 0..7; whatever order the unit adds the 32 depth terms
// in, D is the sum over all of them, so the operands only need the same
// depth index at the same lane and slot.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 load8(uint16_t const* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<uint4 const*>(p));
}

__device__ __forceinline__ bf16x8 gather8(uint16_t const* p, int stride) {
    uint32_t w[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        w[t] = uint32_t(p[2 * t * stride]) | (uint32_t(p[(2 * t + 1) * stride]) << 16);
    }
    return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct Weights {
    alignas(16) uint16_t w1[Hidden * S_feat];
    alignas(16) uint16_t w2[Hidden * S_hid];
    alignas(16) uint16_t w3[Hidden * S_hid];
    alignas(16) uint16_t w4[Num_out * S_hid];
    float    b[3 * Hidden + Num_out];
};

// Rows of `cols` weights to LDS rows of `stride`, 16 bytes a load (2-byte
// loads took 11 us of a workgroup's start).
template <int Rows, int Cols, int Stride>
__device__ __forceinline__ void load_rows(uint16_t* dst, uint16_t const* src) {
    static_assert(Cols % 8 == 0 && Stride % 8 == 0, "16-byte pieces");
    for (int i = threadIdx.x; i < Rows * (Cols / 8); i += blockDim.x) {
        *reinterpret_cast<uint4*>(dst + (i / (Cols / 8)) * Stride + 8 * (i % (Cols / 8))) =
            reinterpret_cast<uint4 const*>(src)[i];
    }
}

__device__ void load_weights(Weights& s, uint16_t const* wt, float const* params) {
    static_assert(T_w1 % 8 == 0 && T_w2 % 8 == 0 && T_w3 % 8 == 0 && T_w4 % 8 == 0, "16-byte pieces");
    load_rows<Hidden, Feat_pad, S_feat>(s.w1, wt + T_w1);
    load_rows<Hidden, Hidden, S_hid>(s.w2, wt + T_w2);
    load_rows<Hidden, Hidden, S_hid>(s.w3, wt + T_w3);
    load_rows<Num_out, Hidden, S_hid>(s.w4, wt + T_w4);
    for (int i = threadIdx.x; i < Hidden; i += blockDim.x) {
        s.b[i]              = params[Off_b1 + i];
        s.b[Hidden + i]     = params[Off_b2 + i];
        s.b[2 * Hidden + i] = params[Off_b3 + i];
    }
    for (int i = threadIdx.x; i < Num_out; i += blockDim.x) {
        s.b[3 * Hidden + i] = params[Off_b4 + i];
    }
}

// Epilogue of a layer: acc[nt][t] is output 16 nt + 4q + t of row r; adds
// the bias and writes, per Mode, ReLU'd bf16 to H (one 8-byte store per
// tile), or fp32 rows r < rows to global F (Mode_out; float4 stores where F
// is 16-byte aligned, sf a multiple of 4).
enum { Mode_relu = 0, Mode_out = 1 };

template <int N, int Mode>
__device__ __forceinline__ void store_layer(f32x4 const (&acc)[N / 16], float const* bias, int r,
                                            int q, uint16_t* H, int sh, float* F, int sf,
                                            int rows) {
#pragma unroll
    for (int nt = 0; nt < N / 16; ++nt) {
        int const j0 = nt * 16 + 4 * q;
        float     v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v[t] = acc[nt][t] + bias[j0 + t];
        }
        if (Mode_relu == Mode) {
            uint2 pk;
            pk.x = pack_bf16(fmaxf(v[0], 0.f), fmaxf(v[1], 0.f));
            pk.y = pack_bf16(fmaxf(v[2], 0.f), fmaxf(v[3], 0.f));
            *reinterpret_cast<uint2*>(H + r * sh + j0) = pk;
        } else if (r < rows) {
            float* const o = F + size_t(r) * sf + j0;
            if (0 == (reinterpret_cast<uintptr_t>(o) & 15u)) {
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    o[t] = v[t];
                }
            }
        }
    }
}

// out[16][N] = act(A[16][K] W + b), formed as its transpose W^T A^T so that a
// lane's four results are four consecutive outputs of one row: MFMA A
// operand = rows of W^T in LDS (stride sw), B operand = activation rows
// (bf16 in LDS, stride sa), D[4q + t][r] = output 16 nt + 4q + t of row r.
// Double-depth products: one 16-byte operand read per lane and step.
// The depth steps run outermost, so each activation operand is read once and
// the N / 16 accumulation chains interleave.
template <int K, int N, int Mode>
__device__ void layer(uint16_t const* A, int sa, uint16_t const* Wt, int sw, float const* bias,
                      uint16_t* H, int sh, float* F, int sf, int rows = 16) {
    int const lane = threadIdx.x & 63;
    int const r    = lane & 15;
    int const q    = lane >> 4;
    f32x4     acc[N / 16];
#pragma unroll
    for (int nt = 0; nt < N / 16; ++nt) {
        acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    static_assert(K % 32 == 0, "depth in steps of 32");
#pragma unroll
    for (int ks = 0; ks < K / 32; ++ks) {
        bf16x8 const b = load8(A + r * sa + ks * 32 + 8 * q);
#pragma unroll
        for (int nt = 0; nt < N / 16; ++nt) {
            acc[nt] = mfma32(load8(Wt + (nt * 16 + r) * sw + ks * 32 + 8 * q), b, acc[nt]);
        }
    }
    store_layer<N, Mode>(acc, bias, r, q, H, sh, F, sf, rows);
}

// First layer of the forward pass with its features formed in registers: the
// B operand of lane (r, q) at depth step ks is features k0 .. k0 + 7, k0 =
// 32 ks + 8q, of query row0 + r, i.e. (sin, cos) of pi f x_i for i = k0 / 24
// and the multipliers j0 .. j0 + 3 with j0 = (k0 % 24) / 2 (zero past the
// 216 features): the values gradient_kernel forms.  half_freq holds
// f / 2, and (f / 2) x equals (f x) / 2 for every normal product.  Rows past
// n run on zero inputs; rows do not mix and theirs are never stored.
__device__ void layer1_direct(float const* x, float const* half_freq, uint32_t row0, uint32_t n,
                              uint16_t const* Wt, float const* bias, uint16_t* H) {
    int const      lane = threadIdx.x & 63;
    int const      r    = lane & 15;
    int const      q    = lane >> 4;
    uint32_t const row  = row0 + r;
    bool const     live = row < n;
    f32x4          acc[Hidden / 16];
#pragma unroll
    for (int nt = 0; nt < Hidden / 16; ++nt) {
        acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    static_assert(Feat_pad % 32 == 0 && 24 % 8 == 0, "eight features of one input per lane");
#pragma unroll
    for (int ks = 0; ks < Feat_pad / 32; ++ks) {
        int const k0 = ks * 32 + 8 * q;
        uint4     pk = make_uint4(0u, 0u, 0u, 0u);
        if (k0 < Num_feat) {
            int const   i  = k0 / 24;
            int const   j0 = (k0 % 24) / 2;
            float const v  = live ? x[size_t(row) * Num_in + i] : 0.f;
            uint32_t    w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float const h   = half_freq[i * Num_freq + j0 + u] * v;
                float const rev = h - floorf(h);
                w[u] = pack_bf16(__builtin_amdgcn_sinf(rev), __builtin_amdgcn_cosf(rev));
            }
            pk = make_uint4(w[0], w[1], w[2], w[3]);
        }
        bf16x8 const b = __builtin_bit_cast(bf16x8, pk);
#pragma unroll
        for (int nt = 0; nt < Hidden / 16; ++nt) {
            acc[nt] = mfma32(load8(Wt + (nt * 16 + r) * S_feat + k0), b, acc[nt]);
        }
    }
    store_layer<Hidden, Mode_relu>(acc, bias, r, q, H, S_hid, nullptr, 0, 16);
}

constexpr int Fwd_waves = 16;

struct alignas(16) Fwd_lds {
    Weights  w;
    float    half_freq[Num_in * Num_freq];
    uint16_t h[Fwd_waves][2][16 * S_hid];
};
static_assert(sizeof(Fwd_lds) <= 160 * 1024, "LDS of a workgroup");
static_assert(offsetof(Fwd_lds, h) % 16 == 0 && (S_hid * sizeof(uint16_t)) % 8 == 0,
              "8-byte aligned activation rows");

// A wave computes 16 queries per tile: layer 1 from register features, two
// hidden layers through LDS, the output layer stored straight to out.
__global__ void __launch_bounds__(Fwd_waves * 64)
    forward_kernel(uint16_t const* wt, float const* params, float const* freq, float const* x,
                   uint32_t n_host, uint32_t const* n_dev, float* out) {
    __shared__ Fwd_lds s;
    uint32_t const n = n_dev ? min(*n_dev, n_host) : n_host;
    load_weights(s.w, wt, params);
    for (int i = threadIdx.x; i < Num_in * Num_freq; i += blockDim.x) {
        s.half_freq[i] = 0.5f * freq[i];
    }
    __syncthreads();

    int const wave  = threadIdx.x >> 6;
    uint16_t* H0    = s.h[wave][0];
    uint16_t* H1    = s.h[wave][1];
    float const* bb = s.w.b;

    for (uint32_t tile = blockIdx.x * Fwd_waves + wave; uint64_t(tile) * 16 < n;
         tile += gridDim.x * Fwd_waves) {
        uint32_t const row0 = tile * 16;
        layer1_direct(x, s.half_freq, row0, n, s.w.w1, bb, H0);
        wave_sync();
        layer<Hidden, Hidden, Mode_relu>(H0, S_hid, s.w.w2, S_hid, bb + Hidden, H1, S_hid, nullptr, 0);
        wave_sync();
        layer<Hidden, Hidden, Mode_relu>(H1, S_hid, s.w.w3, S_hid, bb + 2 * Hidden, H0, S_hid, nullptr, 0);
        wave_sync();
        layer<Hidden, Num_out, Mode_out>(H0, S_hid, s.w.w4, S_hid, bb + 3 * Hidden, nullptr, 0,
                                         out + size_t(row0) * Num_out, Num_out,
                                         int(min(n - row0, 16u)));
        wave_sync();
    }
}

// ---- training ----

constexpr int Grad_waves = 4;
constexpr int Chunk      = 16 * Grad_waves;  // samples per workgroup step
constexpr int Grad_tiles = (Feat_pad / 16) * (Hidden / 16) + 2 * (Hidden / 16) * (Hidden / 16) +
                           (Hidden / 16) * (Num_out / 16);  // 56 + 32 + 8 = 96
constexpr int Tiles_per_wave = Grad_tiles / Grad_waves;      // 24

// Sample-major rows of the transposed operands: the 64 samples of a chunk and
// padding that puts 16 rows on distinct banks (16-byte reads of 16 lanes).
constexpr int S_smp = Chunk + 8;  // 72
constexpr int S_y   = 36;         // fp32 outputs of a row

// The weight gradients multiply over the samples, so every activation and
// pre-activation gradient is stored transposed, [feature][sample]: an operand
// is one 16-byte read.  A wave's own 16 rows pass from layer to layer through
// `row`, one after the other.
struct alignas(16) Grad_lds {
    Weights  w;
    uint16_t xt[Feat_pad * S_smp];
    uint16_t ht[3][Hidden * S_smp];  // post-ReLU activations of the hidden layers
    uint16_t dzt[3][Hidden * S_smp];  // loss gradient at the hidden pre-activations
    uint16_t dyt[Num_out * S_smp];    // loss gradient at the outputs
    alignas(16) uint16_t row[Grad_waves][16 * S_hid];
    alignas(16) float freq[Num_in * Num_freq];
};
static_assert(sizeof(Grad_lds) <= 160 * 1024, "LDS of a workgroup");
static_assert(offsetof(Grad_lds, xt) % 16 == 0 && offsetof(Grad_lds, dyt) % 16 == 0 &&
                  (S_smp * sizeof(uint16_t)) % 16 == 0 && (S_hid * sizeof(uint16_t)) % 16 == 0 &&
                  (S_out * sizeof(uint16_t)) % 16 == 0 && 16 * S_y * sizeof(float) <= 16 * S_hid * sizeof(uint16_t),
              "16-byte reads are aligned and a wave's outputs fit its rows");
constexpr int Num_bias = 3 * Hidden + Num_out;  // 224

// Loss gradient at the outputs of lobes q and q + 4 of one sample (row of
// Y), for g = -t / q: the derivative of -t log q (the reduction divides by
// the batch's weight sum).  The sample's four lanes (q = 0..3, lanes r + 16 q)
// hold two lobes each and share the mixture's sums by lane exchange, so
// every lobe is evaluated once; all 64 lanes must call it.
struct Lobe_terms {
    float v, kap, cosk, sa, sb, d;
    float st, ct, sp, cp;  // sines and cosines of the lobe's angles
    float em;              // expm1(-2 kappa)
};

__device__ Lobe_terms lobe_terms(float const* r, float dirx, float diry, float dirz) {
    Lobe_terms t;
    t.sa  = 1.f / (1.f + expf(-r[0]));
    t.sb  = 1.f / (1.f + expf(-r[1]));
    sincosf(dev::Pi * t.sa, &t.st, &t.ct);
    sincosf(2.f * dev::Pi * t.sb, &t.sp, &t.cp);
    t.cosk = (t.st * t.cp) * dirx + (t.st * t.sp) * diry + t.ct * dirz;
    t.kap  = expf(fminf(fmaxf(r[2], Kappa_lo), Kappa_hi));
    t.em   = expm1f(-2.f * t.kap);
    t.v    = t.kap / (2.f * dev::Pi * -t.em) * expf(t.kap * (t.cosk - 1.f));
    t.d    = r[3];
    return t;
}

__device__ void lobe_gradient(Lobe_terms const& t, float const* r, float g, float q, float wk,
                              float dirx, float diry, float dirz, float out[4]) {
    float const resp = wk * t.v;
    // softmax: dq/dd_k = w_k (v_k - q)
    out[3] = g * wk * (t.v - q);
    // kappa: d log v / d kappa = 1/kappa - 2 e^(-2k) / (1 - e^(-2k)) + (cos - 1)
    float const e2  = expf(-2.f * t.kap);
    float const dlk = 1.f / t.kap - 2.f * e2 / (-t.em) + (t.cosk - 1.f);
    bool const  in  = r[2] > Kappa_lo && r[2] < Kappa_hi;
    out[2]          = in ? g * resp * dlk * t.kap : 0.f;
    // direction: d log v / d mu = kappa w
    float const dth = t.kap * ((t.ct * t.cp) * dirx + (t.ct * t.sp) * diry - t.st * dirz);
    float const dph = t.kap * ((-t.st * t.sp) * dirx + (t.st * t.cp) * diry);
    out[0]          = g * resp * dth * dev::Pi * t.sa * (1.f - t.sa);
    out[1]          = g * resp * dph * 2.f * dev::Pi * t.sb * (1.f - t.sb);
}

__device__ float sum4(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

__device__ void output_gradients(float const* y, float dirx, float diry, float dirz, float tw,
                                 int q, float g0[4], float g1[4]) {
    Lobe_terms const a = lobe_terms(y + 4 * q, dirx, diry, dirz);
    Lobe_terms const b = lobe_terms(y + 4 * (q + 4), dirx, diry, dirz);
    float            dmax = fmaxf(a.d, b.d);
    dmax                  = fmaxf(dmax, __shfl_xor(dmax, 16));
    dmax                  = fmaxf(dmax, __shfl_xor(dmax, 32));
    float const ea        = expf(a.d - dmax);
    float const eb        = expf(b.d - dmax);
    float const esum      = sum4(ea + eb);
    float const wa        = ea / esum;
    float const wb        = eb / esum;
    float const qm        = sum4(wa * a.v + wb * b.v);  // mixture density q
    float const g         = -tw / fmaxf(qm, 1e-30f);
    lobe_gradient(a, y + 4 * q, g, qm, wa, dirx, diry, dirz, g0);
    lobe_gradient(b, y + 4 * (q + 4), g, qm, wb, dirx, diry, dirz, g1);
}

// A layer's results in a wave, acc[nt][t] = output 16 nt + 4q + t of row r:
// to the wave's rows (one 8-byte store per tile) and, transposed, to column
// `sample` of dt.
template <int N>
__device__ __forceinline__ void store_rows(float const (&v)[N / 16][4], int r, int q, uint16_t* row,
                                           int stride, uint16_t* dt, int sample) {
#pragma unroll
    for (int nt = 0; nt < N / 16; ++nt) {
        int const   j0 = nt * 16 + 4 * q;
        uint2 const pk = make_uint2(pack_bf16(v[nt][0], v[nt][1]), pack_bf16(v[nt][2], v[nt][3]));
        if (row) {
            *reinterpret_cast<uint2*>(row + r * stride + j0) = pk;
        }
        dt[(j0 + 0) * S_smp + sample] = uint16_t(pk.x);
        dt[(j0 + 1) * S_smp + sample] = uint16_t(pk.x >> 16);
        dt[(j0 + 2) * S_smp + sample] = uint16_t(pk.y);
        dt[(j0 + 3) * S_smp + sample] = uint16_t(pk.y >> 16);
    }
}

// ReLU of acc + bias, stored as above; bit 4 nt + t of the result: output
// 16 nt + 4q + t of row r is positive (as bf16).
template <int N>
__device__ __forceinline__ uint32_t store_relu(f32x4 const (&acc)[N / 16], float const* bias, int r,
                                               int q, uint16_t* row, uint16_t* dt, int sample) {
    float    v[N / 16][4];
    uint32_t mask = 0;
#pragma unroll
    for (int nt = 0; nt < N / 16; ++nt) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v[nt][t] = fmaxf(acc[nt][t] + bias[nt * 16 + 4 * q + t], 0.f);
            mask |= from_bf16(to_bf16(v[nt][t])) > 0.f ? 1u << (4 * nt + t) : 0u;
        }
    }
    store_rows<N>(v, r, q, row, S_hid, dt, sample);
    return mask;
}

// acc = W^T A^T over a wave's 16 rows like layer().
template <int K, int N>
__device__ __forceinline__ void multiply(uint16_t const* row, int stride, uint16_t const* Wt, int sw,
                                         int r, int q, f32x4 (&acc)[N / 16]) {
#pragma unroll
    for (int nt = 0; nt < N / 16; ++nt) {
        acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int ks = 0; ks < K / 32; ++ks) {
        bf16x8 const b = load8(row + r * stride + ks * 32 + 8 * q);
#pragma unroll
        for (int nt = 0; nt < N / 16; ++nt) {
            acc[nt] = mfma32(load8(Wt + (nt * 16 + r) * sw + ks * 32 + 8 * q), b, acc[nt]);
        }
    }
}

// The operands of a layer's way back, W[16 nt + r][32 ks + 8q ..] =
// Wt[32 ks + 8q ..][16 nt + r], gathered once per workgroup and kept.
template <int K, int N>
struct Back {
    bf16x8 w[K / 32][N / 16];

    __device__ __forceinline__ void load(uint16_t const* Wt, int sw, int r, int q) {
#pragma unroll
        for (int ks = 0; ks < K / 32; ++ks) {
#pragma unroll
            for (int nt = 0; nt < N / 16; ++nt) {
                w[ks][nt] = gather8(Wt + (ks * 32 + 8 * q) * sw + nt * 16 + r, sw);
            }
        }
    }

    // (src[16][K] W^T) * (act > 0), the mask as store_relu gives it
    __device__ __forceinline__ void run(uint16_t const* src, int stride, uint32_t mask, int r, int q,
                                        float (&v)[N / 16][4]) const {
        f32x4 acc[N / 16];
#pragma unroll
        for (int nt = 0; nt < N / 16; ++nt) {
            acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int ks = 0; ks < K / 32; ++ks) {
            bf16x8 const b = load8(src + r * stride + ks * 32 + 8 * q);
#pragma unroll
            for (int nt = 0; nt < N / 16; ++nt) {
                acc[nt] = mfma32(w[ks][nt], b, acc[nt]);
            }
        }
#pragma unroll
        for (int nt = 0; nt < N / 16; ++nt) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v[nt][t] = (mask >> (4 * nt + t)) & 1u ? acc[nt][t] : 0.f;
            }
        }
    }
};

// Weight gradients of one layer over the chunk's samples: tiles (mt, nt) of
// act^T dz for mt = mt0, mt0 + step, ..., accumulated in acc.
template <int Tiles>
__device__ __forceinline__ void weight_gradients(uint16_t const* act, uint16_t const* dz, int mt0,
                                                 int step, int nt, int r, int q, f32x4* acc) {
    bf16x8 b[Chunk / 32];
#pragma unroll
    for (int ks = 0; ks < Chunk / 32; ++ks) {
        // B[k][j] = dz[sample k][j]
        b[ks] = load8(dz + (nt * 16 + r) * S_smp + ks * 32 + 8 * q);
    }
#pragma unroll
    for (int k = 0; k < Tiles; ++k) {
#pragma unroll
        for (int ks = 0; ks < Chunk / 32; ++ks) {
            // A[i][k] = act[sample k][feature i]
            bf16x8 const a = load8(act + ((mt0 + step * k) * 16 + r) * S_smp + ks * 32 + 8 * q);
            acc[k]         = mfma32(a, b[ks], acc[k]);
        }
    }
}

// Bound by the latencies of one wave a SIMD (155 KB of LDS a workgroup).
// 65 536 samples, 4 chunks a workgroup: 81 us with row-major activations,
// whose transposed operands took eight 2-byte reads each; 57.6 us with the
// layout above.
__global__ void __launch_bounds__(Grad_waves * 64)
    gradient_kernel(uint16_t const* wt, float const* params, float const* freq, float const* x,
                    float const* dirs, float const* weights, uint32_t n, uint32_t const* window,
                    float* partial, float* wsum) {
    __shared__ Grad_lds s;
    if (window) {
        // the batch is records [window[0], window[0] + window[1]) of the arrays
        uint32_t const off = window[0];
        n                  = window[1];
        x += 9 * size_t(off);
        dirs += 3 * size_t(off);
        weights += off;
    }
    load_weights(s.w, wt, params);
    for (int i = threadIdx.x; i < Num_in * Num_freq; i += blockDim.x) {
        s.freq[i] = freq[i];
    }
    __syncthreads();

    // thread b < 224 sums the gradient of bias b over the samples, in order
    float bias_acc = 0.f;

    int const wave = threadIdx.x >> 6;
    int const lane = threadIdx.x & 63;
    int const r    = lane & 15;
    int const q    = lane >> 4;
    float     wacc = 0.f;  // weights of this lane's samples (q == 0), in order

    Back<Num_out, Hidden> back4;
    Back<Hidden, Hidden>  back3, back2;
    back4.load(s.w.w4, S_hid, r, q);
    back3.load(s.w.w3, S_hid, r, q);
    back2.load(s.w.w2, S_hid, r, q);

    f32x4 acc[Tiles_per_wave];
#pragma unroll
    for (int k = 0; k < Tiles_per_wave; ++k) {
        acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    uint16_t* const R      = s.row[wave];
    float* const    Y      = reinterpret_cast<float*>(R);
    int const       sample = wave * 16 + r;  // of the chunk

    uint32_t const chunks = (n + Chunk - 1) / Chunk;
    for (uint32_t c = blockIdx.x; c < chunks; c += gridDim.x) {  // block-uniform
        uint32_t const row  = c * Chunk + sample;
        bool const     live = row < n;
        // unnormalized weights: the reduction divides by the batch's weight sum
        float const tw  = live ? weights[row] : 0.f;
        float const dx  = live ? dirs[3 * size_t(row) + 0] : 0.f;
        float const dyv = live ? dirs[3 * size_t(row) + 1] : 0.f;
        float const dz  = live ? dirs[3 * size_t(row) + 2] : 1.f;

        uint32_t mask1, mask2, mask3;
        {
            // Layer 1 with its features formed in registers: the operand of
            // lane (r, q) at depth step ks is features k0 .. k0 + 7 of row r,
            // sin / cos of pi (freq[i][j] x_i), the product rounded to fp32;
            // zero past the 216 features and for rows past n.  sin(pi f) =
            // sin(2 pi (f / 2)): the hardware sine of the fraction of f / 2
            // turns (f / 2 and its fraction are exact).
            f32x4 a1[Hidden / 16];
#pragma unroll
            for (int nt = 0; nt < Hidden / 16; ++nt) {
                a1[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            static_assert(Feat_pad % 32 == 0 && 24 % 8 == 0, "eight features of one input per lane");
#pragma unroll
            for (int ks = 0; ks < Feat_pad / 32; ++ks) {
                int const k0   = ks * 32 + 8 * q;
                uint32_t  w[4] = {0u, 0u, 0u, 0u};
                if (k0 < Num_feat && live) {
                    int const   i  = k0 / 24;
                    int const   j0 = (k0 % 24) / 2;
                    float const v  = x[size_t(row) * Num_in + i];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        float const f   = s.freq[i * Num_freq + j0 + u] * v;
                        float const h   = 0.5f * f;
                        float const rev = h - floorf(h);
                        w[u] = pack_bf16(__builtin_amdgcn_sinf(rev), __builtin_amdgcn_cosf(rev));
                    }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    s.xt[(k0 + 2 * u) * S_smp + sample]     = uint16_t(w[u]);
                    s.xt[(k0 + 2 * u + 1) * S_smp + sample] = uint16_t(w[u] >> 16);
                }
                bf16x8 const b = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
#pragma unroll
                for (int nt = 0; nt < Hidden / 16; ++nt) {
                    a1[nt] = mfma32(load8(s.w.w1 + (nt * 16 + r) * S_feat + k0), b, a1[nt]);
                }
            }
            mask1 = store_relu<Hidden>(a1, s.w.b, r, q, R, s.ht[0], sample);
        }
        wave_sync();
        f32x4 a[Hidden / 16];
        multiply<Hidden, Hidden>(R, S_hid, s.w.w2, S_hid, r, q, a);
        wave_sync();  // the rows are read before they are written
        mask2 = store_relu<Hidden>(a, s.w.b + Hidden, r, q, R, s.ht[1], sample);
        wave_sync();
        multiply<Hidden, Hidden>(R, S_hid, s.w.w3, S_hid, r, q, a);
        wave_sync();
        mask3 = store_relu<Hidden>(a, s.w.b + 2 * Hidden, r, q, R, s.ht[2], sample);
        wave_sync();
        f32x4 ay[Num_out / 16];
        multiply<Hidden, Num_out>(R, S_hid, s.w.w4, S_hid, r, q, ay);
        wave_sync();
#pragma unroll
        for (int nt = 0; nt < Num_out / 16; ++nt) {
            int const j0 = nt * 16 + 4 * q;
            float     o[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                o[t] = ay[nt][t] + s.w.b[3 * Hidden + j0 + t];
            }
            *reinterpret_cast<float4*>(Y + r * S_y + j0) = make_float4(o[0], o[1], o[2], o[3]);
        }
        wave_sync();

        // output gradients: lane handles sample r, lobes q and q + 4
        {
            float g[2][4];
            if (0 == q) {
                wacc += tw;
            }
            output_gradients(Y + r * S_y, dx, dyv, dz, tw, q, g[0], g[1]);
            wave_sync();  // the outputs are read by all lanes before the rows are written
            store_rows<Num_out>(g, r, q, R, S_out, s.dyt, sample);
        }
        wave_sync();
        float v[Hidden / 16][4];
        back4.run(R, S_out, mask3, r, q, v);
        wave_sync();
        store_rows<Hidden>(v, r, q, R, S_hid, s.dzt[2], sample);
        wave_sync();
        back3.run(R, S_hid, mask2, r, q, v);
        wave_sync();
        store_rows<Hidden>(v, r, q, R, S_hid, s.dzt[1], sample);
        wave_sync();
        back2.run(R, S_hid, mask1, r, q, v);
        store_rows<Hidden>(v, r, q, nullptr, 0, s.dzt[0], sample);
        __syncthreads();

        // bias gradients: sums over the chunk's samples
        if (int(threadIdx.x) < Num_bias) {
            int const       b   = threadIdx.x;
            uint16_t const* src = b < 3 * Hidden ? s.dzt[b / Hidden] + (b % Hidden) * S_smp
                                                 : s.dyt + (b - 3 * Hidden) * S_smp;
#pragma unroll
            for (int k = 0; k < Chunk; k += 8) {
                uint4 const    pk   = *reinterpret_cast<uint4 const*>(src + k);
                uint32_t const w[4] = {pk.x, pk.y, pk.z, pk.w};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    bias_acc += from_bf16(uint16_t(w[u]));
                    bias_acc += from_bf16(uint16_t(w[u] >> 16));
                }
            }
        }

        // weight gradients over the chunk's 64 samples: dW = act^T dz, tile
        // wave + 4 k of the 56 + 16 + 16 + 8
        weight_gradients<14>(s.xt, s.dzt[0], 0, 1, wave, r, q, acc);
        weight_gradients<4>(s.ht[0], s.dzt[1], 0, 1, wave, r, q, acc + 14);
        weight_gradients<4>(s.ht[1], s.dzt[2], 0, 1, wave, r, q, acc + 18);
        weight_gradients<2>(s.ht[2], s.dyt, wave / 2, 2, wave % 2, r, q, acc + 22);
        __syncthreads();
    }

    // the workgroup's weight sum, lanes in a fixed order (reusing the rows)
    float* const sums = reinterpret_cast<float*>(s.row);
    sums[threadIdx.x] = wacc;
    __syncthreads();
    if (0 == threadIdx.x) {
        float t = 0.f;
        for (int k = 0; k < Grad_waves * 64; ++k) {
            t += sums[k];
        }
        wsum[blockIdx.x] = t;
    }

    // partial sums of this workgroup, in the parameter layout
    float* out = partial + size_t(blockIdx.x) * Num_params;
#pragma unroll
    for (int k = 0; k < Tiles_per_wave; ++k) {
        int const tile = wave + Grad_waves * k;
        int       base, cols, mt, nt;
        if (tile < 56) {
            base = Off_w1, cols = Hidden, mt = tile / 4, nt = tile % 4;
        } else if (tile < 72) {
            base = Off_w2, cols = Hidden, mt = (tile - 56) / 4, nt = (tile - 56) % 4;
        } else if (tile < 88) {
            base = Off_w3, cols = Hidden, mt = (tile - 72) / 4, nt = (tile - 72) % 4;
        } else {
            base = Off_w4, cols = Num_out, mt = (tile - 88) / 2, nt = (tile - 88) % 2;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int const i = mt * 16 + 4 * q + t;
            int const j = nt * 16 + r;
            out[base + i * cols + j] = acc[k][t];
        }
    }
    if (int(threadIdx.x) < Num_bias) {
        int const b       = threadIdx.x;
        int const offs[4] = {Off_b1, Off_b2, Off_b3, Off_b4};
        out[offs[b < 3 * Hidden ? b / Hidden : 3] + (b < 3 * Hidden ? b % Hidden : b - 3 * Hidden)] =
            bias_acc;
    }
}

// grad = (sum of the workgroups' partials) / (sum of the batch weights).  A
// workgroup covers 64 parameters: wave w sums the partials of workgroups
// w, w + 8, w + 16, ... in order, then the eight sums are added in wave
// order (the weights alike), so gradients are deterministic.
constexpr int Reduce_waves = 8;

__global__ void __launch_bounds__(Reduce_waves * 64)
    reduce_partials(float const* partial, float const* wsum, uint32_t blocks, float* grad) {
    __shared__ float sum_s[Reduce_waves][64];
    __shared__ float sum_t[Reduce_waves];
    uint32_t const lane = threadIdx.x & 63;
    uint32_t const wave = threadIdx.x >> 6;
    uint32_t const p    = blockIdx.x * 64 + lane;
    float          s    = 0.f;
    float          t    = 0.f;
    if (p < uint32_t(Num_params)) {
        for (uint32_t b = wave; b < blocks; b += Reduce_waves) {
            s += partial[size_t(b) * Num_params + p];
            t += wsum[b];
        }
    }
    sum_s[wave][lane] = s;
    if (0 == lane) {
        sum_t[wave] = t;
    }
    __syncthreads();
    if (0 == wave && p < uint32_t(Num_params)) {
        float ss = 0.f;
        float tt = 0.f;
#pragma unroll
        for (int w = 0; w < Reduce_waves; ++w) {
            ss += sum_s[w][lane];
            tt += sum_t[w];
        }
        grad[p] = ss / (tt > 0.f ? tt : 1.f);
    }
}

// W^T bf16 position of parameter p, or -1 for a bias
__device__ __host__ inline int transposed_index(int p) {
    if (p < Off_b1) {
        return T_w1 + (p % Hidden) * Feat_pad + p / Hidden;
    }
    if (p >= Off_w2 && p < Off_b2) {
        int const e = p - Off_w2;
        return T_w2 + (e % Hidden) * Hidden + e / Hidden;
    }
    if (p >= Off_w3 && p < Off_b3) {
        int const e = p - Off_w3;
        return T_w3 + (e % Hidden) * Hidden + e / Hidden;
    }
    if (p >= Off_w4 && p < Off_b4) {
        int const e = p - Off_w4;
        return T_w4 + (e % Num_out) * Hidden + e / Num_out;
    }
    return -1;
}

__global__ void refresh_bf16(float const* params, uint16_t* wt) {
    int const p = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= Num_params) {
        return;
    }
    int const t = transposed_index(p);
    if (t >= 0) {
        wt[t] = to_bf16(params[p]);
    }
}

// Training window of one Adam step: window = {first record, count, step t}.
// Records [k batch mod count, + batch) of the first min(*records, cap); with
// batch 0 the count is split into `steps` slices.  Empty windows take no
// step.  trained (optional) sums the records used.
__global__ void set_window(uint32_t const* records, uint32_t cap, uint32_t fixed_n, uint32_t k,
                           uint32_t steps, uint32_t batch, uint32_t* window, uint32_t* step,
                           unsigned long long* trained) {
    uint32_t off = 0;
    uint32_t nb  = fixed_n;
    if (records) {
        uint32_t const count = min(*records, cap);
        uint32_t const b     = batch ? min(batch, count) : (count + steps - 1) / max(steps, 1u);
        off                  = count ? uint32_t((uint64_t(k) * b) % count) : 0u;
        nb                   = count ? min(b, count - off) : 0u;
    }
    window[0] = off;
    window[1] = nb;
    if (nb) {
        *step += 1;
        if (trained) {
            *trained += nb;
        }
    }
    window[2] = *step;
}

// Adam with the bias corrections of the window's step (no step on an empty window).
__global__ void adam_kernel(float* params, float* m, float* v, float const* grad, float lr,
                            float b1, float b2, uint32_t const* window, float eps, uint16_t* wt) {
    int const p = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= Num_params || 0 == window[1]) {
        return;
    }
    double const step = double(window[2]);
    float const  c1   = float(1.0 - pow(double(b1), step));
    float const  c2   = float(1.0 - pow(double(b2), step));
    float const g  = grad[p];
    float const mm = b1 * m[p] + (1.f - b1) * g;
    float const vv = b2 * v[p] + (1.f - b2) * g * g;
    m[p]           = mm;
    v[p]           = vv;
    float const w  = params[p] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    params[p]      = w;
    int const t    = transposed_index(p);
    if (t >= 0) {
        wt[t] = to_bf16(w);
    }
}

uint32_t blocks_for(uint64_t n, uint32_t b) {
    uint64_t const g = (n + b - 1) / b;
    return uint32_t(g > 0 ? g : 1);
}

struct Pcg {
    uint64_t state, inc;
    uint32_t next() {
        uint64_t const old = state;
        state              = old * 6364136223846793005ull + (inc | 1);
        uint32_t const xrs = uint32_t(((old >> 18u) ^ old) >> 27u);
        uint32_t const rot = uint32_t(old >> 59u);
        return (xrs >> rot) | (xrs << ((0u - rot) & 31u));
    }
    double uniform() { return double(next()) * (1.0 / 4294967296.0); }
};

hipError_t refresh(GuideNet& net, hipStream_t stream) {
    hipLaunchKernelGGL(refresh_bf16, dim3(blocks_for(Num_params, 256)), dim3(256), 0, stream,
                       net.params, net.wt);
    return hipGetLastError();
}

}  // namespace

void GuideNet::release() {
    (void)hipFree(params);
    (void)hipFree(adam_m);
    (void)hipFree(adam_v);
    (void)hipFree(grad);
    (void)hipFree(partial);
    (void)hipFree(wsum);
    (void)hipFree(freq);
    (void)hipFree(wt);
    (void)hipFree(window);
    *this = GuideNet();
}

int32_t guide_create(uint64_t seed, uint32_t num_cus, GuideNet& out) {
    GuideNet n;
    n.partial_blocks = num_cus ? num_cus : 256;
    hipError_t e     = device_malloc(&n.params, Num_params * sizeof(float));
    if (!e) e = device_malloc(&n.adam_m, Num_params * sizeof(float));
    if (!e) e = device_malloc(&n.adam_v, Num_params * sizeof(float));
    if (!e) e = device_malloc(&n.grad, Num_params * sizeof(float));
    if (!e) e = device_malloc(&n.partial, size_t(n.partial_blocks) * Num_params * sizeof(float));
    if (!e) e = device_malloc(&n.wsum, size_t(n.partial_blocks) * sizeof(float));
    if (!e) e = device_malloc(&n.freq, Num_in * Num_freq * sizeof(float));
    if (!e) {
        float f[Num_in * Num_freq];
        guide_default_frequencies(f);
        e = hipMemcpy(n.freq, f, sizeof(f), hipMemcpyHostToDevice);
    }
    if (!e) e = device_malloc(&n.wt, Num_t * sizeof(uint16_t));
    if (!e) e = device_malloc(&n.window, 8 * sizeof(uint32_t));
    if (e) {
        n.release();
        return fail(MI_ERR_HIP, "guide: %s", hipGetErrorString(e));
    }
    n.step_dev     = n.window + 4;
    n.scratch_step = n.window + 5;
    // He-uniform weights (fan-in of the unpadded features), zero biases
    std::vector<float> p(Num_params, 0.f);
    Pcg                rng{0, (seed << 1) | 1};
    rng.next();
    rng.state += seed;
    rng.next();
    struct L {
        int off, in, out, fan;
    } const layers[4] = {{Off_w1, Feat_pad, Hidden, Num_feat},
                         {Off_w2, Hidden, Hidden, Hidden},
                         {Off_w3, Hidden, Hidden, Hidden},
                         {Off_w4, Hidden, Num_out, Hidden}};
    for (L const& l : layers) {
        double const bound = std::sqrt(6.0 / l.fan);
        for (int i = 0; i < l.in; ++i) {
            for (int j = 0; j < l.out; ++j) {
                float const w = float((2.0 * rng.uniform() - 1.0) * bound);
                p[l.off + i * l.out + j] = (l.off == Off_w1 && i >= Num_feat) ? 0.f : w;
            }
        }
    }
    out = n;
    return guide_set_params(out, p.data());
}

void guide_default_frequencies(float* out) {
    for (int i = 0; i < Num_in; ++i) {
        double const step = i < 3 ? 0.5 : 0.25;  // position: half octaves, directions: quarter
        for (int j = 0; j < Num_freq; ++j) {
            out[i * Num_freq + j] = float(std::exp2(step * j));
        }
    }
}

int32_t guide_set_frequencies(GuideNet& net, float const* host_freq) {
    for (int k = 0; k < Num_in * Num_freq; ++k) {
        if (!std::isfinite(host_freq[k]) || std::fabs(host_freq[k]) > 4096.f) {
            return fail(MI_ERR_ARGS, "guide frequencies: entry %d is %g", k, double(host_freq[k]));
        }
    }
    hipError_t const e = hipMemcpy(net.freq, host_freq, Num_in * Num_freq * sizeof(float),
                                   hipMemcpyHostToDevice);
    if (e) {
        return fail(MI_ERR_HIP, "guide frequencies: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

int32_t guide_set_params(GuideNet& net, float const* host_params) {
    hipError_t e = hipMemcpy(net.params, host_params, Num_params * sizeof(float), hipMemcpyHostToDevice);
    if (!e) e = hipMemset(net.adam_m, 0, Num_params * sizeof(float));
    if (!e) e = hipMemset(net.adam_v, 0, Num_params * sizeof(float));
    if (!e) e = hipMemset(net.window, 0, 8 * sizeof(uint32_t));  // step 0
    if (!e) e = refresh(net, nullptr);
    if (!e) e = hipDeviceSynchronize();
    if (e) {
        return fail(MI_ERR_HIP, "guide parameters: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

int32_t guide_get_params(GuideNet const& net, float* host_params) {
    if (hipError_t const e = hipMemcpy(host_params, net.params, Num_params * sizeof(float),
                                       hipMemcpyDeviceToHost);
        e) {
        return fail(MI_ERR_HIP, "guide parameters: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

int32_t guide_forward(GuideNet const& net, float const* x, uint32_t n, float* out,
                      hipStream_t stream) {
    if (0 == n) {
        return MI_OK;
    }
    // one workgroup per CU fits (LDS): more would reload the weights per round
    uint32_t const tiles  = blocks_for(n, 16);
    uint32_t const blocks = std::min<uint32_t>(blocks_for(tiles, Fwd_waves), net.partial_blocks);
    hipLaunchKernelGGL(forward_kernel, dim3(blocks), dim3(Fwd_waves * 64), 0, stream, net.wt,
                       net.params, net.freq, x, n, static_cast<uint32_t const*>(nullptr), out);
    if (hipError_t const e = hipGetLastError(); e) {
        return fail(MI_ERR_HIP, "guide forward: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

int32_t guide_forward_device_count(GuideNet const& net, float const* x, uint32_t const* n,
                                   uint32_t max_n, float* out, hipStream_t stream) {
    if (0 == max_n) {
        return MI_OK;
    }
    uint32_t const tiles  = blocks_for(max_n, 16);
    uint32_t const blocks = std::min<uint32_t>(blocks_for(tiles, Fwd_waves), net.partial_blocks);
    hipLaunchKernelGGL(forward_kernel, dim3(blocks), dim3(Fwd_waves * 64), 0, stream, net.wt,
                       net.params, net.freq, x, max_n, n, out);
    if (hipError_t const e = hipGetLastError(); e) {
        return fail(MI_ERR_HIP, "guide forward: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

namespace {

// gradient of the batch described by net.window (max_n bounds its count)
void enqueue_gradients(GuideNet& net, float const* x, float const* dirs, float const* weights,
                       uint32_t max_n, hipStream_t stream) {
    uint32_t const blocks = std::min(blocks_for(max_n, Chunk), net.partial_blocks);
    hipLaunchKernelGGL(gradient_kernel, dim3(blocks), dim3(Grad_waves * 64), 0, stream, net.wt,
                       net.params, net.freq, x, dirs, weights, 0u,
                       static_cast<uint32_t const*>(net.window), net.partial, net.wsum);
    hipLaunchKernelGGL(reduce_partials, dim3(blocks_for(Num_params, 64)), dim3(Reduce_waves * 64),
                       0, stream, net.partial, net.wsum, blocks, net.grad);
}

void enqueue_adam(GuideNet& net, float lr, hipStream_t stream) {
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(Num_params, 256)), dim3(256), 0, stream,
                       net.params, net.adam_m, net.adam_v, net.grad, lr, 0.9f, 0.99f,
                       static_cast<uint32_t const*>(net.window), 1e-8f, net.wt);
}

}  // namespace

int32_t guide_gradients(GuideNet& net, float const* x, float const* dirs, float const* weights,
                        uint32_t n, hipStream_t stream) {
    if (0 == n) {
        return fail(MI_ERR_ARGS, "guide gradients: empty batch");
    }
    // a fixed window of n records that takes no Adam step
    hipLaunchKernelGGL(set_window, dim3(1), dim3(1), 0, stream, static_cast<uint32_t const*>(nullptr),
                       0u, n, 0u, 1u, 0u, net.window, net.scratch_step,
                       static_cast<unsigned long long*>(nullptr));
    enqueue_gradients(net, x, dirs, weights, n, stream);
    if (hipError_t const e = hipGetLastError(); e) {
        return fail(MI_ERR_HIP, "guide gradients: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

int32_t guide_adam_step(GuideNet& net, float const* x, float const* dirs, float const* weights,
                        uint32_t n, float lr, hipStream_t stream) {
    if (0 == n) {
        return fail(MI_ERR_ARGS, "guide adam: empty batch");
    }
    hipLaunchKernelGGL(set_window, dim3(1), dim3(1), 0, stream, static_cast<uint32_t const*>(nullptr),
                       0u, n, 0u, 1u, 0u, net.window, net.step_dev,
                       static_cast<unsigned long long*>(nullptr));
    enqueue_gradients(net, x, dirs, weights, n, stream);
    enqueue_adam(net, lr, stream);
    if (hipError_t const e = hipGetLastError(); e) {
        return fail(MI_ERR_HIP, "guide adam: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

int32_t guide_train_records(GuideNet& net, float const* x, float const* dirs, float const* weights,
                            uint32_t const* num_records, uint32_t capacity, uint32_t steps,
                            uint32_t batch, float lr, unsigned long long* trained,
                            hipStream_t stream) {
    for (uint32_t k = 0; k < steps; ++k) {
        hipLaunchKernelGGL(set_window, dim3(1), dim3(1), 0, stream, num_records, capacity, 0u, k,
                           steps, batch, net.window, net.step_dev, trained);
        enqueue_gradients(net, x, dirs, weights, batch ? std::min(batch, capacity) : capacity, stream);
        enqueue_adam(net, lr, stream);
    }
    if (hipError_t const e = hipGetLastError(); e) {
        return fail(MI_ERR_HIP, "guide training: %s", hipGetErrorString(e));
    }
    return MI_OK;
}

}  // namespace mi
