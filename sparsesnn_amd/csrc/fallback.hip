// Unfused fallback path and spike (un)packing for gfx950.
//
// dense_conv_bn_kernel mirrors the reference's decomposed Conv+BN kernels
// conv2d_bn_t4_kernel / conv1x1_bn_t4_kernel (sengine/kernels/conv2d_bn_if_t4.py:551-673):
// one GEMM over all T*B images with the BN epilogue acc*scale + bias.  It differs in
// keeping the BN output in fp32 (the reference rounds it to fp16, which is what breaks
// its fp32 parity, sengine/scripts/verify_correctness.py:4-9).  Used for convs whose
// weights are not 2:4 (sengine/optimizer.py:845-853 routes them to a dense conv + a
// standalone neuron) and for shapes the sparse kernel does not take.
//
// multistep_neuron_kernel mirrors lif_neuron_kernel / if_neuron_kernel
// (sengine/csrc/kernels.cuh:18-54): one thread per spatial element walks the T
// timesteps in order, so there is no cross-thread membrane race.  The arithmetic is
// that of the PyTorch neurons (models/neurons.py:121-146,169-184), including soft reset
// and v_reset, which the reference's native kernels ignore.
#include "common.h"
#include "internal.h"

namespace sengine {

// 64-row x 64-channel units per CU from which a workgroup takes two of them (each weight fragment
// read from LDS then feeds two row tiles).  Smaller outputs run one stage's latency after another and
// want more workgroups.  3x3, 128 channels in, one unit / two, us: 192 units 8.7 / 10.4, 592 14.2 /
// 14.8, 800 16.8 / 15.4, 1,200 22.1 / 20.7, 3,136 46.4 / 39.8; two weight planes 592 21.2 / 21.4, 800
// 25.9 / 22.1; fp16 input 592 20.2 / 23.0, 800 25.6 / 23.9, 1,200 33.7 / 34.7, 2,000 50.6 / 47.3.  Four
// units measured slower at every size (fewer, longer workgroups in a round).
constexpr int64_t kDenseWideUnits = 3;

struct DenseParams {
  const uint8_t* in;
  const u32x4_t* wvals;
  const float* scale;
  const float* bias;
  float* out;
  int C, H, W, F, KW, SH, SW, PH, PW, DH, DW, OH, OW;
  int64_t rows;  // T*B*OH*OW: no neuron here, so the timesteps are just more images
  int nstage;    // taps * C / (32 * CW)
  float enc_scale;
};

// Implicit GEMM over all T*B images.  Bound by the matrix cores and, on shallow reductions, by
// the fp32 output (4 bytes per value against 1 bit in).  Workgroup = 4 waves = 64 output
// channels x 64*RT rows; wave w owns rows 16*RT*w .. +16*RT-1 and all 64 channels (4*RT
// accumulator tiles), so a 1 KB weight fragment read from LDS feeds RT matrix instructions and
// an expanded activation fragment (about 10 VALU) feeds 4.
//
// The reduction runs in stages of CW k-steps (32*CW channels of one tap): the stage's weights
// are copied through registers into one of two LDS buffers by the whole workgroup, the
// activations (CW words, or CW 16-byte pieces, of each of the lane's RT rows) go straight to
// registers in one load per row, and both are requested a stage ahead of their use; one barrier
// per stage.  128->256 28x28 k3, T = 4, B = 16, spike bits: 85.8 -> 45.8 us against one load
// per byte, tap and timestep with nothing in flight over the matrix instructions.
template <int IN_ENC, int PLANES, int RT, int CW>
__global__ __launch_bounds__(256) void dense_conv_bn_kernel(DenseParams p) {
  constexpr bool BITS = IN_ENC == SENGINE_ENC_BITS;
  constexpr int NA = CW * PLANES;   // 16-byte weight pieces per thread and stage
  constexpr int BW = BITS ? CW : 4 * CW;  // activation words per row and stage
  typedef uint32_t bword_t __attribute__((ext_vector_type(BW == 1 ? 2 : BW)));
  __shared__ u32x4_t sA[2][NA][256];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int g = lane >> 4;
  const int col = lane & 15;
  const int G = blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * (64 * RT) + wave * (16 * RT) + col;
  const int pixb = BITS ? p.C >> 3 : p.C * 2;  // bytes per input pixel

  const uint8_t* src[RT];  // tap (0, 0), channel 0 of each row's window (only read where inside)
  int ih0[RT], iw0[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int64_t row = row0 + 16 * r;
    const uint32_t m = (uint32_t)(row < p.rows ? row : 0);  // rows past the end: computed, not stored
    const uint32_t ohw = (uint32_t)(p.OH * p.OW);
    const uint32_t n = m / ohw, rem = m - n * ohw;
    const int oh = (int)(rem / (uint32_t)p.OW), ow = (int)(rem - (uint32_t)oh * (uint32_t)p.OW);
    ih0[r] = oh * p.SH - p.PH;
    iw0[r] = ow * p.SW - p.PW;
    src[r] = p.in + (((int64_t)n * p.H + ih0[r]) * p.W + iw0[r]) * pixb + (BITS ? 0 : 16 * g);
  }

  const u32x4_t* wv = p.wvals + (size_t)G * p.nstage * NA * 256 + tid;
  u32x4_t aw[NA];
  bword_t bn[RT];
  uint32_t inside[RT];  // all ones where the loaded row's tap lies inside the image
  // counters of the next stage to load (uniform): tap (kr, ks), channel c0
  int kr = 0, ks = 0, c0 = 0;
  auto load = [&]() {
#pragma unroll
    for (int i = 0; i < NA; ++i) aw[i] = wv[i * 256];
    wv += NA * 256;
    const int dh = kr * p.DH, dw = ks * p.DW;
    const int64_t toff = ((int64_t)dh * p.W + dw) * pixb + (BITS ? c0 >> 3 : c0 * 2);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const bool ok = (unsigned)(ih0[r] + dh) < (unsigned)p.H && (unsigned)(iw0[r] + dw) < (unsigned)p.W;
      const uint8_t* s = ok ? src[r] + toff : p.in;  // outside: any valid address, the value is masked at its use
      inside[r] = ok ? ~0u : 0u;
      if constexpr (BITS) {
        if constexpr (BW == 1) {
          bn[r][0] = *reinterpret_cast<const uint32_t*>(s);
        } else {
          typedef uint32_t w_t __attribute__((ext_vector_type(BW), aligned(4)));
          bn[r] = *reinterpret_cast<const w_t*>(s);
        }
      } else {
#pragma unroll
        for (int k = 0; k < CW; ++k) {
          const u32x4_t v = *reinterpret_cast<const u32x4_t*>(s + (ok ? 64 * k : 0));
#pragma unroll
          for (int u = 0; u < 4; ++u) bn[r][4 * k + u] = v[u];
        }
      }
    }
    c0 += 32 * CW;
    if (c0 == p.C) {
      c0 = 0;
      if (++ks == p.KW) {
        ks = 0;
        ++kr;
      }
    }
  };

  float4_t acc[RT][4];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int a = 0; a < 4; ++a) acc[r][a] = float4_t{0.f, 0.f, 0.f, 0.f};

  load();
#pragma unroll
  for (int i = 0; i < NA; ++i) sA[0][i][tid] = aw[i];
  __syncthreads();
  for (int st = 0; st < p.nstage; ++st) {
    const int buf = st & 1;
    bword_t bc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int k = 0; k < BW; ++k) bc[r][k] = bn[r][k] & inside[r];
    if (st + 1 < p.nstage) load();
#pragma unroll
    for (int k = 0; k < CW; ++k) {
      half8_t av[PLANES][4];
#pragma unroll
      for (int pl = 0; pl < PLANES; ++pl)
#pragma unroll
        for (int a = 0; a < 4; ++a)
          av[pl][a] = __builtin_bit_cast(half8_t, sA[buf][k * PLANES + pl][a * 64 + lane]);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        half8_t bf;
        if constexpr (BITS)
          bf = expand_bits8((bc[r][k] >> (8 * g)) & 0xffu);
        else
          bf = __builtin_bit_cast(half8_t, u32x4_t{bc[r][4 * k], bc[r][4 * k + 1], bc[r][4 * k + 2], bc[r][4 * k + 3]});
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int pl = 0; pl < PLANES; ++pl)
            acc[r][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[pl][a], bf, acc[r][a], 0, 0, 0);
      }
    }
    if (st + 1 < p.nstage) {
#pragma unroll
      for (int i = 0; i < NA; ++i) sA[buf ^ 1][i][tid] = aw[i];
    }
    __syncthreads();
  }

  const int cob = G * 64 + g * 16;
  float sc[16], bi[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    sc[j] = p.scale[cob + j] * p.enc_scale;
    bi[j] = p.bias[cob + j];
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int64_t row = row0 + 16 * r;
    if (row >= p.rows) continue;
    float4_t* dst = reinterpret_cast<float4_t*>(p.out + row * p.F + cob);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = __builtin_fmaf(acc[r][a][i], sc[4 * a + i], bi[4 * a + i]);
      dst[a] = o;
    }
  }
}

template <int IN_ENC, int PLANES, int RT, int CW>
static hipError_t launch_dense(DenseParams& p, int taps, hipStream_t s) {
  p.nstage = taps * (p.C / (32 * CW));
  const dim3 grid((unsigned)((p.rows + 64 * RT - 1) / (64 * RT)), (unsigned)(p.F / 64));
  hipLaunchKernelGGL((dense_conv_bn_kernel<IN_ENC, PLANES, RT, CW>), grid, dim3(256), 0, s, p);
  return hipGetLastError();
}

template <int IN_ENC, int PLANES, int CW>
static hipError_t launch_dense_rt(DenseParams& p, int taps, hipStream_t s) {
  const int64_t units = (p.rows + 63) / 64 * (p.F / 64);
  return units >= kDenseWideUnits * device_cus() ? launch_dense<IN_ENC, PLANES, 2, CW>(p, taps, s)
                                  : launch_dense<IN_ENC, PLANES, 1, CW>(p, taps, s);
}

// k-steps per stage: as many as divide the channels, bounded by the registers that hold a stage.
template <int IN_ENC, int PLANES>
static hipError_t launch_dense_cw(DenseParams& p, int taps, hipStream_t s) {
  if constexpr (IN_ENC == SENGINE_ENC_BITS && PLANES == 1)
    if (p.C % 128 == 0) return launch_dense_rt<IN_ENC, PLANES, 4>(p, taps, s);
  if (p.C % 64 == 0) return launch_dense_rt<IN_ENC, PLANES, 2>(p, taps, s);
  return launch_dense_rt<IN_ENC, PLANES, 1>(p, taps, s);
}

struct NeuronKernelParams {
  const float* x;
  float* state;
  uint8_t* out;
  float* h_trace;
  int64_t n;
  int T;
  NeuronParams np;
};

// One thread per element, any pointer alignment and length.
template <int OUT_ENC>
__global__ __launch_bounds__(256) void multistep_neuron_kernel(NeuronKernelParams p) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = s < p.n;
  const int lane = threadIdx.x & 63;
  float v = (valid && p.state) ? p.state[s] : 0.f;
  for (int t = 0; t < p.T; ++t) {
    const float x = valid ? p.x[(int64_t)t * p.n + s] : 0.f;
    float xf = x;
    if (p.np.neuron == SENGINE_NEURON_LIF && p.np.pow2) xf = x * p.np.rtau;  // exact
    const float h = neuron_charge(p.np, v, xf);
    const bool spike = valid && h >= p.np.vth;
    v = neuron_reset(p.np, h, spike);
    if (valid && p.h_trace) p.h_trace[(int64_t)t * p.n + s] = h;
    if (OUT_ENC == SENGINE_ENC_BITS) {
      const uint64_t mask = __ballot(spike);
      // n % 32 == 0, so a 32-lane half-wave maps to exactly one word when its first lane is valid
      if ((lane & 31) == 0 && valid)
        reinterpret_cast<uint32_t*>(p.out)[((int64_t)t * p.n + s) >> 5] = (uint32_t)(mask >> (lane & 32));
    } else if (valid) {
      reinterpret_cast<_Float16*>(p.out)[(int64_t)t * p.n + s] = spike ? (_Float16)1.0f : (_Float16)0.0f;
    }
  }
  if (valid && p.state) p.state[s] = v;
}

// Bits of one 32-element word, four per lane in a run of eight lanes: every lane of the run ends
// with the whole word (three butterfly steps on the DPP network, no LDS).
__device__ __forceinline__ uint32_t or_over_8_lanes(uint32_t x) {
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xb1, 0xf, 0xf, true);   // quad_perm [1,0,3,2]
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4e, 0xf, 0xf, true);   // quad_perm [2,3,0,1]
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xf, 0xf, true);  // row_half_mirror
  return x;
}

// Four elements per thread (16-byte accesses; the pointers and n allow them), the inputs of up to
// four timesteps in flight together.  Bound by HBM: one fp32 read per element and step.  The spike
// words of four steps are stored by four different lanes of each eight-lane run in one instruction.
// 3.2M elements x 4 steps (51 MB): 16.7 -> 11.7 us against the form above, 1.6M 6.7 -> 4.9.
template <int OUT_ENC>
__global__ __launch_bounds__(256) void multistep_neuron4_kernel(NeuronKernelParams p) {
  constexpr int TC = 4;
  const int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  const bool valid = s < p.n;
  const int64_t sc = valid ? s : 0;
  const int sub = threadIdx.x & 7;
  const bool lif_pow2 = p.np.neuron == SENGINE_NEURON_LIF && p.np.pow2;
  float4_t v = float4_t{0.f, 0.f, 0.f, 0.f};
  if (p.state) v = *reinterpret_cast<const float4_t*>(p.state + sc);
  for (int t0 = 0; t0 < p.T; t0 += TC) {
    float4_t x[TC];
#pragma unroll
    for (int k = 0; k < TC; ++k) {
      if (t0 + k >= p.T) break;
      x[k] = *reinterpret_cast<const float4_t*>(p.x + (int64_t)(t0 + k) * p.n + sc);
    }
    uint32_t mine = 0;
#pragma unroll
    for (int k = 0; k < TC; ++k) {
      if (t0 + k >= p.T) break;
      float4_t h;
      uint32_t nib = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h[i] = neuron_charge(p.np, v[i], lif_pow2 ? x[k][i] * p.np.rtau : x[k][i]);  // exact
        const bool spike = h[i] >= p.np.vth;
        v[i] = neuron_reset(p.np, h[i], spike);
        nib |= (uint32_t)spike << i;
      }
      if (valid && p.h_trace) *reinterpret_cast<float4_t*>(p.h_trace + (int64_t)(t0 + k) * p.n + s) = h;
      if (OUT_ENC == SENGINE_ENC_BITS) {
        const uint32_t word = or_over_8_lanes(nib << (4 * sub));
        mine = sub == k ? word : mine;
      } else if (valid) {
        const uint32_t lo = ((nib & 1) ? 0x3c00u : 0u) | ((nib & 2) ? 0x3c000000u : 0u);
        const uint32_t hi = ((nib & 4) ? 0x3c00u : 0u) | ((nib & 8) ? 0x3c000000u : 0u);
        *reinterpret_cast<uint2*>(p.out + ((int64_t)(t0 + k) * p.n + s) * 2) = uint2{lo, hi};
      }
    }
    // n % 32 == 0: a run of eight lanes is inside or outside as a whole
    if (OUT_ENC == SENGINE_ENC_BITS && valid && sub < TC && t0 + sub < p.T)
      reinterpret_cast<uint32_t*>(p.out)[((int64_t)(t0 + sub) * p.n + s) >> 5] = mine;
  }
  if (valid && p.state) *reinterpret_cast<float4_t*>(p.state + s) = v;
}

template <int X_ENC>
__global__ __launch_bounds__(256) void pack_spikes_kernel(const void* x, int64_t n, uint32_t* bits) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  bool on = false;
  if (e < n) {
    if (X_ENC == SENGINE_ENC_F16) on = (float)static_cast<const _Float16*>(x)[e] != 0.f;
    else on = static_cast<const float*>(x)[e] != 0.f;
  }
  const uint64_t mask = __ballot(on);
  if ((lane & 31) == 0 && e < n) bits[e >> 5] = (uint32_t)(mask >> (lane & 32));
}

template <int OUT_ENC>
__global__ __launch_bounds__(256) void unpack_spikes_kernel(const uint32_t* bits, int64_t n, void* out) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const bool on = (bits[e >> 5] >> (e & 31)) & 1u;
  if (OUT_ENC == SENGINE_ENC_F16) static_cast<_Float16*>(out)[e] = on ? (_Float16)1.0f : (_Float16)0.0f;
  else static_cast<float*>(out)[e] = on ? 1.0f : 0.0f;
}

// Eight elements per thread (16-byte accesses): one byte of spike bits each way.  Bound by HBM on
// the dense side.
template <int X_ENC>
__global__ __launch_bounds__(256) void pack_spikes8_kernel(const u32x4_t* x, int64_t n8, uint8_t* bits) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n8) return;
  uint32_t b = 0;
  if (X_ENC == SENGINE_ENC_F16) {
    const u32x4_t v = x[i];
#pragma unroll
    for (int k = 0; k < 4; ++k)  // nonzero: any bit but the sign
      b |= ((v[k] & 0x7fffu) ? 1u << (2 * k) : 0u) | ((v[k] & 0x7fff0000u) ? 2u << (2 * k) : 0u);
  } else {
    const u32x4_t lo = x[2 * i], hi = x[2 * i + 1];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      b |= ((lo[k] & 0x7fffffffu) ? 1u << k : 0u) | ((hi[k] & 0x7fffffffu) ? 16u << k : 0u);
  }
  bits[i] = (uint8_t)b;
}

template <int OUT_ENC>
__global__ __launch_bounds__(256) void unpack_spikes8_kernel(const uint8_t* bits, int64_t n, u32x4_t* out) {
  constexpr int PER = OUT_ENC == SENGINE_ENC_F16 ? 8 : 4;  // elements of one 16-byte store
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i * PER >= n) return;
  u32x4_t v;
  if (OUT_ENC == SENGINE_ENC_F16) {
    const uint32_t b = bits[i];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = ((b >> (2 * k) & 1u) ? 0x3c00u : 0u) | ((b >> (2 * k + 1) & 1u) ? 0x3c000000u : 0u);
  } else {
    const uint32_t b = (uint32_t)bits[i >> 1] >> (4 * (int)(i & 1));
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = (b >> k & 1u) ? 0x3f800000u : 0u;
  }
  out[i] = v;
}

inline bool aligned16(const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; }

}  // namespace sengine

using namespace sengine;

extern "C" int sengine_amd_dense_conv_bn(const sengine_conv_lif_desc* d, const void* data, const void* blob_values,
                                         const float* bn_scale, const float* bn_bias, float* out,
                                         hipStream_t stream) {
  Geometry geo;
  int rc = check_desc(d, &geo, false);
  if (rc) return rc;
  if (!data || !blob_values || !bn_scale || !bn_bias || !out) return set_error(-1, "dense_conv_bn: null pointer");
  if (d->T != 1 && d->T != 2 && d->T != 4 && d->T != 8) return set_error(-3, "dense_conv_bn: T must be 1, 2, 4 or 8");
  if (d->in_enc != SENGINE_ENC_BITS && d->in_enc != SENGINE_ENC_F16)
    return set_error(-2, "dense_conv_bn: in_enc must be BITS or F16");
  if (geo.M > (1ll << 30)) return set_error(-2, "dense_conv_bn: B*OH*OW too large");
  DenseParams p;
  p.in = static_cast<const uint8_t*>(data);
  p.wvals = static_cast<const u32x4_t*>(blob_values);
  p.scale = bn_scale;
  p.bias = bn_bias;
  p.out = out;
  p.C = d->C_in; p.H = d->H; p.W = d->W; p.F = d->C_out; p.KW = d->KW;
  p.SH = d->stride_h; p.SW = d->stride_w; p.PH = d->pad_h; p.PW = d->pad_w;
  p.DH = d->dil_h; p.DW = d->dil_w; p.OH = geo.OH; p.OW = geo.OW;
  p.rows = d->T * geo.M;
  // a row is indexed in 32 bits; that many rows of 64 fp32 outputs are 512 GiB
  if (p.rows > 0x7fffffffll) return set_error(-2, "dense_conv_bn: T*B*OH*OW too large");
  p.enc_scale = d->in_enc == SENGINE_ENC_BITS ? 1.0f / kBitSpikeValue : 1.0f;
  const int taps = d->KH * d->KW;
  if (d->in_enc == SENGINE_ENC_BITS)
    return (int)(d->weight_planes == 1 ? launch_dense_cw<SENGINE_ENC_BITS, 1>(p, taps, stream)
                                       : launch_dense_cw<SENGINE_ENC_BITS, 2>(p, taps, stream));
  return (int)(d->weight_planes == 1 ? launch_dense_cw<SENGINE_ENC_F16, 1>(p, taps, stream)
                                     : launch_dense_cw<SENGINE_ENC_F16, 2>(p, taps, stream));
}

extern "C" int sengine_amd_multistep_neuron(int32_t T, int64_t n, int32_t neuron, int32_t hard_reset, float tau,
                                            float v_threshold, float v_reset, const float* x, float* state,
                                            int32_t out_enc, void* spikes, float* h_trace, hipStream_t stream) {
  if (T < 1 || n < 1) return set_error(-2, "multistep_neuron: T and n must be >= 1");
  if (!x || !spikes) return set_error(-1, "multistep_neuron: null pointer");
  if (const char* why = neuron_invalid(neuron, tau)) return set_error(-2, why);
  if (out_enc == SENGINE_ENC_BITS && n % 32 != 0) return set_error(-2, "multistep_neuron: bit output needs n % 32 == 0");
  if (out_enc != SENGINE_ENC_BITS && out_enc != SENGINE_ENC_F16)
    return set_error(-2, "multistep_neuron: out_enc must be BITS or F16");
  NeuronKernelParams p{x, state, static_cast<uint8_t*>(spikes), h_trace, n, T,
                       make_neuron_params(neuron, hard_reset, tau, v_threshold, v_reset)};
  // Four elements per thread once one each is more threads than the chip holds (2,048 per CU) and
  // would take a second round; below, four neurons in one thread are only a longer chain.  T = 4, bits,
  // one element / four, us: 32,768 elements 2.6 / 3.4, 393,216 3.1 / 3.7, 524,288 3.4 / 3.8, 655,360
  // 4.2 / 4.0, 1,605,632 6.7 / 4.9.  Needs 16-byte rows: every timestep's row and every buffer on a
  // 16-byte boundary (fp16 spikes: 8).
  if (n > 2048ll * device_cus() && n % 4 == 0 && aligned16(x) && aligned16(state) && aligned16(h_trace) &&
      (out_enc == SENGINE_ENC_BITS || reinterpret_cast<uintptr_t>(spikes) % 8 == 0)) {
    const dim3 grid4((unsigned)((n / 4 + 255) / 256));
    if (out_enc == SENGINE_ENC_BITS)
      hipLaunchKernelGGL(multistep_neuron4_kernel<SENGINE_ENC_BITS>, grid4, dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL(multistep_neuron4_kernel<SENGINE_ENC_F16>, grid4, dim3(256), 0, stream, p);
    return (int)hipGetLastError();
  }
  dim3 grid((unsigned)((n + 255) / 256));
  if (out_enc == SENGINE_ENC_BITS)
    hipLaunchKernelGGL(multistep_neuron_kernel<SENGINE_ENC_BITS>, grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(multistep_neuron_kernel<SENGINE_ENC_F16>, grid, dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

extern "C" int sengine_amd_pack_spikes(const void* x, int32_t x_enc, int64_t n_pos, int32_t C, uint32_t* bits,
                                       hipStream_t stream) {
  if (!x || !bits) return set_error(-1, "pack_spikes: null pointer");
  if (n_pos < 0 || C < 1 || C % 32 != 0) return set_error(-2, "pack_spikes: need C % 32 == 0");
  const int64_t n = n_pos * C;
  if (n == 0) return 0;
  if (aligned16(x) && (x_enc == SENGINE_ENC_F16 || x_enc == SENGINE_ENC_F32)) {
    const dim3 grid8((unsigned)((n / 8 + 255) / 256));
    const u32x4_t* x16 = static_cast<const u32x4_t*>(x);
    uint8_t* b8 = reinterpret_cast<uint8_t*>(bits);
    if (x_enc == SENGINE_ENC_F16)
      hipLaunchKernelGGL(pack_spikes8_kernel<SENGINE_ENC_F16>, grid8, dim3(256), 0, stream, x16, n / 8, b8);
    else
      hipLaunchKernelGGL(pack_spikes8_kernel<SENGINE_ENC_F32>, grid8, dim3(256), 0, stream, x16, n / 8, b8);
    return (int)hipGetLastError();
  }
  dim3 grid((unsigned)((n + 255) / 256));
  if (x_enc == SENGINE_ENC_F16)
    hipLaunchKernelGGL(pack_spikes_kernel<SENGINE_ENC_F16>, grid, dim3(256), 0, stream, x, n, bits);
  else if (x_enc == SENGINE_ENC_F32)
    hipLaunchKernelGGL(pack_spikes_kernel<SENGINE_ENC_F32>, grid, dim3(256), 0, stream, x, n, bits);
  else
    return set_error(-2, "pack_spikes: x_enc must be F16 or F32");
  return (int)hipGetLastError();
}

extern "C" int sengine_amd_unpack_spikes(const uint32_t* bits, int64_t n_pos, int32_t C, void* out, int32_t out_enc,
                                         hipStream_t stream) {
  if (!bits || !out) return set_error(-1, "unpack_spikes: null pointer");
  if (n_pos < 0 || C < 1 || C % 32 != 0) return set_error(-2, "unpack_spikes: need C % 32 == 0");
  const int64_t n = n_pos * C;
  if (n == 0) return 0;
  if (aligned16(out) && (out_enc == SENGINE_ENC_F16 || out_enc == SENGINE_ENC_F32)) {
    const int64_t stores = n / (out_enc == SENGINE_ENC_F16 ? 8 : 4);
    const dim3 grid16((unsigned)((stores + 255) / 256));
    const uint8_t* b8 = reinterpret_cast<const uint8_t*>(bits);
    u32x4_t* o16 = static_cast<u32x4_t*>(out);
    if (out_enc == SENGINE_ENC_F16)
      hipLaunchKernelGGL(unpack_spikes8_kernel<SENGINE_ENC_F16>, grid16, dim3(256), 0, stream, b8, n, o16);
    else
      hipLaunchKernelGGL(unpack_spikes8_kernel<SENGINE_ENC_F32>, grid16, dim3(256), 0, stream, b8, n, o16);
    return (int)hipGetLastError();
  }
  dim3 grid((unsigned)((n + 255) / 256));
  if (out_enc == SENGINE_ENC_F16)
    hipLaunchKernelGGL(unpack_spikes_kernel<SENGINE_ENC_F16>, grid, dim3(256), 0, stream, bits, n, out);
  else if (out_enc == SENGINE_ENC_F32)
    hipLaunchKernelGGL(unpack_spikes_kernel<SENGINE_ENC_F32>, grid, dim3(256), 0, stream, bits, n, out);
  else
    return set_error(-2, "unpack_spikes: out_enc must be F16 or F32");
  return (int)hipGetLastError();
}
