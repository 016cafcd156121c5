// denoise.hip — kernels of the learned denoiser for gfx950.
//
// The network is a convolutional encoder-decoder over NHWC bf16 tensors.
// Every 3x3 convolution is an implicit GEMM on the matrix cores:
//   forward      M = pixels, N = Cout, K = 9 * Cin   (v_mfma_f32_16x16x32_bf16)
//   data grad    M = pixels, N = Cin,  K = 9 * Cout  (taps mirrored; same kernel)
//   weight grad  M = Cout,   N = Cin,  K = pixels    (v_mfma_f32_16x16x32_bf16, all 9 taps per pass)
// Operand lanes: lane l holds A[l % 16][8 (l / 16) + j] and
// B[8 (l / 16) + j][l % 16] for j < 8, and D[4 (l / 16) + r][l % 16] for
// r < 4. Channel counts are multiples of 16, so every fragment is one
// aligned 16-byte load.
// Accumulation is fp32; weight gradients are summed per split and reduced
// in a fixed order, so training steps are deterministic.
#include "denoise.h"
#include "rows_plan.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace gdn {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even; NaN stays NaN
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}


// ---- convolution, forward and data gradient --------------------------------
// A block owns a tile of kTR image rows x kTC columns of one image and NT*16
// output channels; wave w computes row w of the tile: 4 pixel fragments of
// 16 columns x NT channel fragments. The input channels run in chunks of
// kCK: per chunk the block stages the tile's input halo ((kTR+2) x (kTC+2)
// pixels, read once for all 9 taps) and the chunk's weights in LDS, then
// every wave runs K = 9 * chunk through v_mfma_f32_16x16x32_bf16. One K=32
// step covers two 16-channel sub-slices (tap, channel group) in tap-major
// order: lanes 0-31 take the first, lanes 32-63 the second (zero past the
// end). DGRAD reads the input at p - off_t (the transposed convolution) and
// masks it by the ReLU of the forward output while staging.
constexpr int kTR = 4;               // tile rows, one per wave
constexpr int kTC = 64;              // tile columns, 4 fragments of 16
constexpr int kHR = kTR + 2, kHC = kTC + 2;
constexpr int kCK = 32;              // input channels per staged chunk
constexpr int kLS = kCK;             // LDS row (pixel or weight row) in bf16: 64 B, pieces swizzled by swz

// A 16-byte LDS read (ds_read_b128) is served 16 lanes at a time: lanes
// 0-31 and 32-63 are separate halves, and within a half the quads (4 lanes)
// whose index l >> 2 has an even number of set bits go in one pass, the others
// in the next. Two lanes of a pass conflict when their addresses differ but
// agree in bits 4-7 (the same four of the 64 banks). An MFMA operand read
// takes pixels P .. P + 15 (lane & 15) of piece q = (lane >> 4) & 1 and, in
// lanes 32-63, the next sub-slice. In 64-byte rows piece q of pixel p goes to
// slot q ^ swz(p), and the weight rows the same way by row: every pass then
// covers the 16 bank groups once. The layout was checked conflict free against
// SQ_LDS_BANK_CONFLICT for every read of a chunk, mirrored taps and 16-channel
// chunks included.
__device__ __forceinline__ int swz(int p) { return (p >> 1) & 3; }

template <int NT>
constexpr int conv_out_stride() {  // fp32 row stride of the output staging: the 4 lane groups' rows land in distinct banks
  return NT * 16 + 4;
}
template <int NT>
constexpr size_t conv_lds_bytes() {  // the halo and weights of a chunk, or the output staging
  return std::max(size_t(kHR * kHC + 9 * NT * 16) * kLS * sizeof(uint16_t),
                  size_t(4 * 64 * conv_out_stride<NT>()) * sizeof(float));
}

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v4f mfma32(uint4 a, uint4 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0,
                                                 0);
}


// Zeroes the bf16 elements of a whose mask element is not positive.
__device__ __forceinline__ uint4 mask8(uint4 a, uint4 m) {
  uint32_t av[4] = {a.x, a.y, a.z, a.w}, mv[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t lo = bf2f(uint16_t(mv[k])) > 0.f ? 0x0000ffffu : 0u;
    const uint32_t hi = bf2f(uint16_t(mv[k] >> 16)) > 0.f ? 0xffff0000u : 0u;
    av[k] &= lo | hi;
  }
  return make_uint4(av[0], av[1], av[2], av[3]);
}

// The MFMA steps of one staged chunk of G 16-channel groups.
template <int NT, bool DGRAD, int G>
__device__ __forceinline__ void conv_chunk(const uint16_t* halo, const uint16_t* wts, int lane, int wave,
                                           v4f (&acc)[4][NT]) {
  const int half = (lane >> 4) & 1;
  const int col = lane & 15;
#pragma unroll
  for (int i = 0; i < (9 * G + 1) / 2; ++i) {
    const int sub = 2 * i + (lane >> 5);
    const bool valid = sub < 9 * G;
    const int tap = valid ? sub / G : 0;
    const int q = (sub % G) * 2 + half;  // 16-byte piece of the pixel or weight row
    int dy = tap / 3 - 1, dx = tap % 3 - 1;
    if (DGRAD) dy = -dy, dx = -dx;
    uint4 b[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int r = tap * NT * 16 + j * 16 + col;
      b[j] = valid ? *reinterpret_cast<const uint4*>(wts + r * kLS + 8 * (q ^ swz(r))) : make_uint4(0, 0, 0, 0);
    }
    const int p0 = (wave + 1 + dy) * kHC + col + 1 + dx;  // pixels p0 + 16 f share the swizzle of p0
    const uint16_t* arow = halo + p0 * kLS + 8 * (q ^ swz(p0));
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const uint4 a = valid ? *reinterpret_cast<const uint4*>(arow + f * 16 * kLS) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[f][j] = mfma32(a, b[j], acc[f][j]);
    }
  }
}

// Stages one chunk (G 16-channel groups from channel c0) of the tile's input
// halo and of the weights into LDS. Each batch of loads is issued before
// its LDS stores, halo first, then weights, so a block waits for memory twice
// per chunk rather than once per piece. When xa is
// set the input is the decoder's concatenation [up2(xa) (ca channels), x]:
// channels below ca come from xa at half resolution (nearest), the rest from x.
template <int NT, bool DGRAD, int G>
__device__ __forceinline__ void conv_stage(uint16_t* halo, uint16_t* wts, const uint16_t* __restrict__ x,
                                           const uint16_t* __restrict__ mask, int cin,
                                           const uint16_t* __restrict__ xa, int ca,
                                           const uint16_t* __restrict__ wgt, int co0, int c0, int n, int h0,
                                           int w0, int H, int W, int tid) {
  constexpr int QP = 2 * G;  // 16-byte pieces per pixel or weight row
  constexpr int HP = kHR * kHC * QP, HI = (HP + 255) / 256;
  constexpr int WP = 9 * NT * 16 * QP, WI = (WP + 255) / 256;
  const int cx = xa ? cin - ca : cin, cs = xa ? ca : 0;  // channels of x, first channel from x
  {
    uint4 hv[HI];
#pragma unroll
    for (int k = 0; k < HI; ++k) {
      const int i = tid + 256 * k;
      hv[k] = make_uint4(0, 0, 0, 0);
      if (i < HP) {
        const int px = i / QP, c = c0 + 8 * (i % QP);
        const int hh = h0 - 1 + px / kHC, ww = w0 - 1 + px % kHC;
        if (hh >= 0 && hh < H && ww >= 0 && ww < W) {
          if (c < cs) {
            hv[k] = *reinterpret_cast<const uint4*>(
                xa + ((size_t(n) * (H / 2) + hh / 2) * (W / 2) + ww / 2) * ca + c);
          } else {
            const size_t off = ((size_t(n) * H + hh) * W + ww) * cx + (c - cs);
            hv[k] = *reinterpret_cast<const uint4*>(x + off);
            if (DGRAD && mask) hv[k] = mask8(hv[k], *reinterpret_cast<const uint4*>(mask + off));
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < HI; ++k) {
      const int i = tid + 256 * k;
      if (i < HP) *reinterpret_cast<uint4*>(halo + (i / QP) * kLS + 8 * ((i % QP) ^ swz(i / QP))) = hv[k];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the two batches apart: fewer live registers
  {
    uint4 wv[WI];
#pragma unroll
    for (int k = 0; k < WI; ++k) {
      const int i = tid + 256 * k;
      wv[k] = make_uint4(0, 0, 0, 0);
      if (i < WP) {
        const int r = i / QP, co = r % (NT * 16), tap = r / (NT * 16);
        wv[k] = *reinterpret_cast<const uint4*>(wgt + (size_t(co0 + co) * 9 + tap) * cin + c0 + 8 * (i % QP));
      }
    }
#pragma unroll
    for (int k = 0; k < WI; ++k) {
      const int i = tid + 256 * k;
      if (i < WP) *reinterpret_cast<uint4*>(wts + (i / QP) * kLS + 8 * ((i % QP) ^ swz(i / QP))) = wv[k];
    }
  }
}

template <int NT, bool DGRAD, bool OUT_F32>
__global__ __launch_bounds__(256) void k_conv(const uint16_t* __restrict__ x, const uint16_t* __restrict__ mask,
                                              int cin, const uint16_t* __restrict__ xa, int ca,
                                              const uint16_t* __restrict__ wgt, const float* __restrict__ bias,
                                              void* __restrict__ y, uint16_t* __restrict__ pooled, int cout,
                                              int co_first, int H, int W, int nrt, int nct, int relu,
                                              const uint16_t* __restrict__ omask) {
  extern __shared__ uint4 lds4[];
  uint16_t* halo = reinterpret_cast<uint16_t*>(lds4);
  uint16_t* wts = halo + kHR * kHC * kLS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ct = blockIdx.x % nct, rt = (blockIdx.x / nct) % nrt, n = blockIdx.x / (nct * nrt);
  const int h0 = rt * kTR, w0 = ct * kTC;
  const int co0 = co_first + blockIdx.y * NT * 16;
  v4f acc[4][NT];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[f][j] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < cin; c0 += kCK) {
    __syncthreads();  // the previous chunk's reads are done
    if (cin - c0 >= kCK) {
      conv_stage<NT, DGRAD, 2>(halo, wts, x, mask, cin, xa, ca, wgt, co0, c0, n, h0, w0, H, W, tid);
      __syncthreads();
      conv_chunk<NT, DGRAD, 2>(halo, wts, lane, wave, acc);
    } else {
      conv_stage<NT, DGRAD, 1>(halo, wts, x, mask, cin, xa, ca, wgt, co0, c0, n, h0, w0, H, W, tid);
      __syncthreads();
      conv_chunk<NT, DGRAD, 1>(halo, wts, lane, wave, acc);
    }
  }
  // Epilogue through LDS: each wave writes its 64 pixels x NT*16 channels
  // (bias and ReLU applied) as fp32 rows, then stores whole 16-byte pieces of
  // consecutive channels, instead of 2-byte values scattered over 4 pixels.
  constexpr int OS = conv_out_stride<NT>();
  __syncthreads();  // every wave is done with the staged halo and weights
  float* stage = reinterpret_cast<float*>(lds4) + wave * 64 * OS;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int cl = j * 16 + (lane & 15);
    const float b = (!DGRAD && bias) ? bias[co0 + cl] : 0.f;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[f][j][r] + b;
        if (relu) v = fmaxf(v, 0.f);
        stage[(f * 16 + (lane >> 4) * 4 + r) * OS + cl] = v;
      }
  }
  __syncthreads();
  if (!OUT_F32 && pooled) {  // also the 2x2 max pool of the tile: 2 rows of 32 pixels
    // rounding to bf16 is monotonic, so the max of the rounded values is the rounded max
    const int H2 = H / 2, W2 = W / 2;
    constexpr int G = NT * 2;  // 8-channel pieces per pixel
    for (int i = tid; i < 2 * 32 * G; i += 256) {
      const int g = i % G, pc = (i / G) % 32, pr = i / (G * 32);
      const int h2 = h0 / 2 + pr, w2 = w0 / 2 + pc;
      if (h2 >= H2 || w2 >= W2) continue;
      const float* a = reinterpret_cast<const float*>(lds4) + (2 * pr) * 64 * OS + (2 * pc) * OS + 8 * g;
      uint32_t o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float m[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int c = 2 * k + e;
          m[e] = fmaxf(fmaxf(a[c], a[OS + c]), fmaxf(a[64 * OS + c], a[64 * OS + OS + c]));
        }
        o[k] = uint32_t(f2bf(m[0])) | (uint32_t(f2bf(m[1])) << 16);
      }
      *reinterpret_cast<uint4*>(pooled + ((size_t(n) * H2 + h2) * W2 + w2) * cout + co0 + 8 * g) =
          make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
  const int row = h0 + wave;
  if (row >= H) return;
  const size_t pix0 = (size_t(n) * H + row) * W;
  if (OUT_F32) {
    constexpr int G = NT * 4;  // 4-channel pieces per pixel
    for (int i = lane; i < 64 * G; i += 64) {
      const int p = i / G, g = i % G;
      if (w0 + p >= W) continue;
      const float4 v = *reinterpret_cast<const float4*>(stage + p * OS + 4 * g);
      *reinterpret_cast<float4*>(static_cast<float*>(y) + (pix0 + w0 + p) * cout + co0 + 4 * g) = v;
    }
  } else {
    constexpr int G = NT * 2;  // 8-channel pieces per pixel
    for (int i = lane; i < 64 * G; i += 64) {
      const int p = i / G, g = i % G;
      if (w0 + p >= W) continue;
      const float4 a = *reinterpret_cast<const float4*>(stage + p * OS + 8 * g);
      const float4 b = *reinterpret_cast<const float4*>(stage + p * OS + 8 * g + 4);
      const uint4 o = make_uint4(uint32_t(f2bf(a.x)) | (uint32_t(f2bf(a.y)) << 16),
                                 uint32_t(f2bf(a.z)) | (uint32_t(f2bf(a.w)) << 16),
                                 uint32_t(f2bf(b.x)) | (uint32_t(f2bf(b.y)) << 16),
                                 uint32_t(f2bf(b.z)) | (uint32_t(f2bf(b.w)) << 16));
      const size_t off = (pix0 + w0 + p) * cout + co0 + 8 * g;
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(y) + off) =
          omask ? mask8(o, *reinterpret_cast<const uint4*>(omask + off)) : o;
    }
  }
}

typedef __attribute__((address_space(3))) void lds_void;
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kOutOfRange = 0x80000000u;  // a buffer offset past every tensor
constexpr int kWaitVm0 = 0x0F70;    // s_waitcnt vmcnt(0)
constexpr int kWaitLgkm0 = 0xC07F;  // s_waitcnt lgkmcnt(0)

// A workgroup barrier for LDS data only: this wave's LDS reads and writes are
// complete, then the waves meet. Unlike __syncthreads it does not also wait
// for the LDS copies in flight; those are waited for per buffer.
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A raw buffer resource over [base, base + bytes): reads past the end return
// zeros.
__device__ __forceinline__ i32x4 buffer_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(int32_t(uint32_t(a)));
  r.y = __builtin_amdgcn_readfirstlane(int32_t(uint32_t(a >> 32) & 0xffffu));  // stride 0
  r.z = __builtin_amdgcn_readfirstlane(int32_t(bytes));
  r.w = 0x00020000;
  return r;
}

// Copies 16 bytes per lane from byte offset off of the buffer src to LDS:
// lane l writes dst + 16 l, dst being the same LDS address in every lane (it
// goes to M0). Written in assembly so that the compiler does not take the
// copy in flight for a write to every LDS array and wait for it before the
// reads of the other buffer; the kernel waits for it itself (vmcnt) before it
// reads the buffer. The copy writes no register. The compiler keeps nothing in
// M0 across these blocks in this kernel (no LDS-copy builtins, message sends
// or relative register moves), so clobbering it is safe here.
__device__ __forceinline__ void lds_copy16(const uint4* dst, i32x4 src, uint32_t off) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(uint32_t(reinterpret_cast<uintptr_t>((const lds_void*)dst)));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(m0), "v"(off), "s"(src)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// ---- convolution by rows: weights in registers, pixels straight from global memory --
// Forward and data gradient for the layer shapes of launch_rows. A wave owns a
// strip of 16 pixel columns and NT * 16 output channels and walks down the rows
// of a segment. The roles of the MFMA operands are swapped against k_conv:
// A holds weights (M = output channels), B pixels (N = 16 columns), so that
//   - the layer's weights stay in registers for the wave's whole life;
//   - a pixel fragment, read once, serves the three output rows it touches;
//   - a lane ends with 4 NT consecutive channels of one pixel (fragment j's row
//     4 g + r is channel 4 NT g + 4 j + r), which it stores as they are: no
//     staging in LDS, no barrier anywhere.
// A fragment is one 16-byte buffer load per lane (16 pixels); columns and rows
// outside the image are read past the buffer's range and arrive as zeros. Every
// load and store is such a buffer access, so a row's body has no branch and the
// waits for the loads in flight are exact; the loads run PF rows ahead.
//
// Sums are made in a fixed order: by groups of input channels, tap by tap within one. Forward that is
// the order of the kernels this one replaced, k_conv's or (PAIRS) the persistent LDS kernel's, bit for bit. A data
// gradient takes the pixel taps in that order, so its weight taps come last to first, where k_conv takes the weight taps
// in order and mirrors the pixels: the same terms, rounded otherwise here and there (gradients of a small batch differ by
// a relative 7e-5; their error against 64 bits is the same). A group of 32 channels takes one K = 32 MFMA step per tap.
// A group of 16 pairs taps (0,1), (2,3), (4,5), (6,7), (8,-) in the two halves of K. A part's odd 16 channels are such a group;
// with PAIRS all are. Its fragments, of row i, are the column taps F = (-1 | 0), G = (+1 | -1) and H = (0 | +1), and
// output row r takes F(r-1), G(r-1) with the upper half of G(r), H(r), F(r+1), G(r+1) with zeros. Two groups side by
// side are loaded as one of 32 channels, three contiguous loads a row, and their fragments made by exchanging register
// halves: loading them as they are takes six loads of 32-byte pieces, and 32->32 took 72 us for 60 at 1920x1080.
//
// What bounds it, on one MI355X at 1920x1080: the full-resolution layers of 16 and 32 channels move 3.7 to 4.9 TB/s,
// near what a copy reaches; the wide ones run one wave per SIMD, whose instruction stream (MFMA steps, exchanges,
// packing) then bounds them. With the pixels through LDS, as in k_conv, 64 pixels x 32 channels x 32 outputs cost 6 LDS
// reads per 8 MFMA steps, more than the LDS delivers. Without the empty asm statements below, weights are copied from
// accumulation registers on each use and row offsets become branches around the loads: 48+32->32 took 152 us, not 117.
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {  // round to nearest even
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{lo, hi}, v2bf));
}
__device__ __forceinline__ float relu_of(float v) { return __builtin_amdgcn_fmed3f(v, 0.f, __builtin_huge_valf()); }

constexpr int kRowsBytes = 0x40000000;  // a segment's rows of any tensor take less
struct RowsJob {  // a launch's tensors and shape
  const uint16_t* x;    // the full-resolution part, CB channels
  const uint16_t* xa;   // the half-resolution part, CA channels (CA > 0)
  const uint16_t* wgt;  // [cout][9][CA + CB]
  const float* bias;
  void* y;              // bf16 [n][h][w][cout]; ROWS_F32 fp32; ROWS_RADIANCE fp32 [n][rh][rw][3]
  uint16_t* pooled;     // ROWS_POOL: 2x2 max pool of y
  const uint16_t* omask;  // ROWS_GRAD_MASK
  int rh, rw;
  int cout, co_first;
  int N, H, W;
  int nseg, nstrip, seg_rows, groups;  // row segments and strips of an image; output groups of NT * 16 channels
};
// Forward (bias, ReLU), the same with the pooled copy, data gradient (taps mirrored), the same masked by the ReLU
// of the tensor it belongs to, network output z, network output as radiance expm1(max(z, 0)) of channels 0..2.
enum RowsMode { ROWS_FWD, ROWS_POOL, ROWS_GRAD, ROWS_GRAD_MASK, ROWS_F32, ROWS_RADIANCE };

// The units of an input of CA + CB channels, in order: 32 channels each, then a part's odd 16.
template <int CA, int CB, bool PAIRS>
struct RowsPlan {
  static constexpr int WA = CA / 32, OA = CA / 16 % 2, WB = CB / 32, OB = CB / 16 % 2;
  static constexpr int NC = WA + OA + WB + OB;
  static constexpr int WIDE = PAIRS ? 10 : 9, ODD = 5;  // MFMA steps of a unit, per output row and fragment
  static constexpr int STEPS = WIDE * (WA + WB) + ODD * (OA + OB);
  static constexpr bool in_a(int c) { return c < WA + OA; }
  static constexpr int local(int c) { return in_a(c) ? c : c - WA - OA; }  // within its part
  static constexpr bool odd(int c) { return local(c) >= (in_a(c) ? WA : WB); }
  static constexpr int first(int c) { return 32 * local(c); }  // first channel within its part
  static constexpr int steps(int c) { return odd(c) ? ODD : WIDE; }
  static constexpr int step0(int c) {  // the unit's first MFMA step
    int s = 0;
    for (int k = 0; k < c; ++k) s += steps(k);
    return s;
  }
};

template <int CA, int CB, bool PAIRS, int NT, RowsMode MODE, int WAVES, int PF, int LDSA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_conv_rows(RowsJob q) {
  using P = RowsPlan<CA, CB, PAIRS>;
  constexpr int CIN = CA + CB, NC = P::NC, BW = 3 + PF;  // BW: rows of a fragment ring
  constexpr bool F32 = MODE == ROWS_F32 || MODE == ROWS_RADIANCE;
  constexpr bool MIRROR = MODE == ROWS_GRAD || MODE == ROWS_GRAD_MASK;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  // blocks are dealt round-robin to the 8 XCDs; an XCD's blocks share one contiguous eighth of the
  // tiles, four of a block at a time (one a wave), and a block keeps its output channels
  const int ntile = q.N * q.nseg * q.nstrip, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int t0 = int(int64_t(ntile) * xcd / 8) + wave, t1 = int(int64_t(ntile) * (xcd + 1) / 8);
  const int per = (gridDim.x >> 3) / q.groups;  // blocks of an XCD with the same channels
  const int co0 = q.co_first + slot % q.groups * (NT * 16);
  const int cl = co0 + 4 * NT * g;              // this lane's first output channel

  // the weights, step by step: this lane's piece of each fragment; the last LDSA steps' in LDS
  constexpr int AREG = P::STEPS - LDSA;
  u32x4 A[AREG][NT];
  __shared__ u32x4 Al[LDSA ? LDSA : 1][NT][64];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const bool pair = P::odd(c) || PAIRS;
    const int c0 = (P::in_a(c) ? 0 : CA) + P::first(c);
#pragma unroll
    for (int i = 0; i < P::steps(c); ++i) {
      const int tap = pair ? 2 * (i % 5) + (g >> 1) : i, ch = c0 + (pair ? 16 * (i / 5) + 8 * (g & 1) : 8 * g);
      const bool live = tap < 9;
      const int t = live ? (MIRROR ? 8 - tap : tap) : 0;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int co = co0 + 4 * NT * (col >> 2) + 4 * j + (col & 3);
        u32x4 v = *reinterpret_cast<const u32x4*>(q.wgt + (size_t(co) * 9 + t) * CIN + ch);
        if (!live) v = u32x4{0u, 0u, 0u, 0u};
        const int step = P::step0(c) + i;
        if (step < AREG) A[step < AREG ? step : 0][j] = v;
        else if (wave == 0) Al[step - AREG][j][lane] = v;
      }
    }
  }
  // matrix operands only: kept in accumulation registers, which leaves the others to the pixels
#pragma unroll
  for (int i = 0; i < AREG; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(A[i][j]));
  v4f bj[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) bj[j] = MIRROR ? v4f{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const v4f*>(q.bias + cl + 4 * j);

  if (LDSA) __syncthreads();

  for (int tile = t0 + slot / q.groups * 4; tile < t1; tile += per * 4) {
    const int strip = tile % q.nstrip, sg = (tile / q.nstrip) % q.nseg, n = tile / (q.nstrip * q.nseg);
    const int r0 = sg * q.seg_rows, r1 = min(r0 + q.seg_rows, q.H), w = strip * 16 + col;
    const int i0 = max(r0 - 1, 0), i1 = min(r1 + 1, q.H);  // input rows read
    // buffers over the rows this job reads and writes, so that offsets stay small for tensors of any size
    constexpr int kRaw = 0x00020000;
    const int pb = q.W * CB * 2, Wa = q.W >> 1, pa = Wa * CA * 2, a0 = i0 >> 1;
    const auto rb = __builtin_amdgcn_make_buffer_rsrc((void*)(q.x + (size_t(n) * q.H + i0) * q.W * CB), 0, (i1 - i0) * pb, kRaw);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc((void*)(CA ? q.xa + (size_t(n) * (q.H >> 1) + a0) * Wa * CA : q.x), 0,
                                                      CA ? (((i1 + 1) >> 1) - a0) * pa : 0, kRaw);
    const int py = MODE == ROWS_RADIANCE ? q.rw * 12 : q.W * q.cout * (F32 ? 4 : 2);  // output bytes per row
    const int yrows = MODE == ROWS_RADIANCE ? max(min(r1, q.rh) - r0, 0) : r1 - r0;
    const size_t ybase = MODE == ROWS_RADIANCE ? (size_t(n) * q.rh + r0) * q.rw * 12 : (size_t(n) * q.H + r0) * py;
    const auto ry = __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(q.y) + ybase, 0, yrows * py, kRaw);
    const int yoff = MODE == ROWS_RADIANCE ? (g == 0 && w < q.rw ? w * 12 : int(kOutOfRange))
                                           : (w < q.W ? (w * q.cout + cl) * (F32 ? 4 : 2) : int(kOutOfRange));
    const auto rm = __builtin_amdgcn_make_buffer_rsrc(
        MODE == ROWS_GRAD_MASK ? (void*)(reinterpret_cast<const char*>(q.omask) + ybase) : q.y, 0,
        MODE == ROWS_GRAD_MASK ? yrows * py : 0, kRaw);
    const int pp = (q.W >> 1) * q.cout * 2;
    const auto rp = __builtin_amdgcn_make_buffer_rsrc(
        MODE == ROWS_POOL ? (void*)(reinterpret_cast<char*>(q.pooled) + (size_t(n) * (q.H >> 1) + (r0 >> 1)) * pp) : q.y, 0,
        MODE == ROWS_POOL ? ((r1 - r0) >> 1) * pp : 0, kRaw);
    const int poff = (col & 1) == 0 && w < q.W ? ((w >> 1) * q.cout + cl) * 2 : int(kOutOfRange);
    // this lane's byte offset in a row of a part at column tap dx, or past every buffer
    auto offset = [&](bool a, int dx, int ch) {
      const int ww = w + dx;
      return dx < 2 && ww >= 0 && ww < q.W ? ((a ? ww >> 1 : ww) * (a ? CA : CB) + ch) * 2 : int(kOutOfRange);
    };
    const int hi = g >> 1, c8 = 8 * g, p8 = 8 * (g & 1);
    int of[2][2][3];  // [part][odd unit][fragment]
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int k = 0; k < 3; ++k) of[a][0][k] = offset(a == 0, k - 1, c8);
      of[a][1][0] = offset(a == 0, hi ? 0 : -1, p8);
      of[a][1][1] = offset(a == 0, hi ? -1 : 1, p8);
      of[a][1][2] = offset(a == 0, hi ? 1 : 0, p8);
    }
    // a row outside the image; less than kOutOfRange, so that the two can be added
    constexpr int kRowOut = kRowsBytes;
    const int rows = r1 - r0;
    u32x4 B[NC][3][BW];  // fragment ring: row r0 - 1 + m in slot m % BW
    u32x2 M[NT][BW];     // ROWS_GRAD_MASK: the output mask of row r0 + m in slot m % BW
    // Byte offsets of input row r0 - 1 + m in both parts, past the buffer outside the image. Read back as
    // uniform values, they stay selects, where a branch around each load would serialise the loads.
    struct RowAt { int a, b; };
    auto row_of = [&](int m) {
      const int i = r0 - 1 + m;
      const bool in = uint32_t(i - i0) < uint32_t(i1 - i0);
      const int a = __builtin_amdgcn_readfirstlane(((i >> 1) - a0) * pa), b = __builtin_amdgcn_readfirstlane((i - i0) * pb);
      return RowAt{__builtin_amdgcn_readfirstlane(in ? a : kRowOut), __builtin_amdgcn_readfirstlane(in ? b : kRowOut)};
    };
    // Fragment k of the units of 32 channels or of the odd ones, row r0 - 1 + m.
    auto load = [&](auto S, bool odd, int k, RowAt r) {
      constexpr int slot_ = decltype(S)::value;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (P::odd(c) != odd) continue;
        const bool a = P::in_a(c);
        B[c][k][slot_] = __builtin_amdgcn_raw_buffer_load_b128(a ? ra : rb, of[a ? 0 : 1][odd][k] + (a ? r.a : r.b) + 2 * P::first(c), 0, 0);
      }
    };
    auto load_mask = [&](auto S, int m) {
      constexpr int slot_ = decltype(S)::value;
      if constexpr (MODE == ROWS_GRAD_MASK) {
        const int sm = yoff + (m < rows ? m * py : kRowOut);
#pragma unroll
        for (int j = 0; j + 1 < NT; j += 2) {
          const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rm, sm + 8 * j, 0, 0);
          M[j][slot_] = u32x2{v[0], v[1]};
          M[j + 1][slot_] = u32x2{v[2], v[3]};
        }
        if constexpr (NT & 1) M[NT - 1][slot_] = __builtin_amdgcn_raw_buffer_load_b64(rm, sm + 8 * (NT - 1), 0, 0);
      }
    };
    u32x4 F[NC][2][BW];  // PAIRS: the column taps (-1 | 0) of a unit's two 16-channel halves
    // The lower and the upper halves of two fragments, side by side: of the same pixels' 32 channels at two taps, the
    // pair fragments of channels 0..15 and of 16..31.
    auto halves = [](u32x4 p, u32x4 q2, u32x4& lower, u32x4& upper) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto v = __builtin_amdgcn_permlane32_swap(p[e], q2[e], false, false);
        lower[e] = v[0];
        upper[e] = v[1];
      }
    };
    v4f acc[NT];
    u32x2 prev[NT];  // ROWS_POOL: the row above
#pragma unroll
    for (int j = 0; j < NT; ++j) prev[j] = u32x2{0u, 0u};
    // Output row r0 + m from its sums.
    auto finish = [&](auto S, int m) {
      constexpr int slot_ = decltype(S)::value;
      v4f v[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[j][r] = MIRROR ? acc[j][r] : acc[j][r] + bj[j][r];
      const int so = yoff + m * py;
      if constexpr (MODE == ROWS_RADIANCE) {
        typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
        u32x3 o;
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = __float_as_uint(expm1f(fmaxf(v[0][c], 0.f)));
        __builtin_amdgcn_raw_buffer_store_b96(o, ry, so, 0, 0);
      } else if constexpr (MODE == ROWS_F32) {
#pragma unroll
        for (int j = 0; j < NT; ++j) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[j]), ry, so + 16 * j, 0, 0);
      } else {
        u32x2 p[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if (!MIRROR) p[j] = u32x2{pack_bf16(relu_of(v[j][0]), relu_of(v[j][1])), pack_bf16(relu_of(v[j][2]), relu_of(v[j][3]))};
          else p[j] = u32x2{pack_bf16(v[j][0], v[j][1]), pack_bf16(v[j][2], v[j][3])};
          if (MODE == ROWS_GRAD_MASK)  // zero where the mask is not positive
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const uint32_t k = M[j][slot_][e];
              p[j][e] &= (bf2f(uint16_t(k)) > 0.f ? 0x0000ffffu : 0u) | (__uint_as_float(k & 0xffff0000u) > 0.f ? 0xffff0000u : 0u);
            }
        }
        auto put = [&](auto rsrc, const u32x2(&d)[NT], int o) {
#pragma unroll
          for (int j = 0; j + 1 < NT; j += 2)
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{d[j][0], d[j][1], d[j + 1][0], d[j + 1][1]}, rsrc, o + 8 * j, 0, 0);
          if constexpr (NT & 1) __builtin_amdgcn_raw_buffer_store_b64(d[NT - 1], rsrc, o + 8 * (NT - 1), 0, 0);
        };
        put(ry, p, so);
        if constexpr (MODE == ROWS_POOL) {  // the stored values are already bf16: the max of them is the pooled value
          u32x2 d[NT];
#pragma unroll
          for (int j = 0; j < NT; ++j) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              float lo = fmaxf(bf2f(uint16_t(prev[j][e])), bf2f(uint16_t(p[j][e])));
              float up = fmaxf(__uint_as_float(prev[j][e] & 0xffff0000u), __uint_as_float(p[j][e] & 0xffff0000u));
              lo = fmaxf(lo, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(lo), 0xB1, 0xf, 0xf, true)));
              up = fmaxf(up, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(up), 0xB1, 0xf, 0xf, true)));
              d[j][e] = (__float_as_uint(lo) >> 16) | (__float_as_uint(up) & 0xffff0000u);
            }
            prev[j] = p[j];
          }
          put(rp, d, poff + (m & 1 ? (m >> 1) * pp : kRowOut));  // segments start on even rows
        }
      }
    };
    // Step t makes output row r0 + t and reads what step t + PF needs new.
    auto row = [&](auto T, int t) {
      constexpr int k = decltype(T)::value;  // t % BW
      auto at = [](auto i) { return std::integral_constant<int, decltype(i)::value % BW>{}; };
#define GT_AT(d) at(std::integral_constant<int, k + (d)>{})
      const RowAt ahead = row_of(t + 2 + PF);
#pragma unroll
      for (int f = 0; f < 3; ++f) load(GT_AT(2 + PF), false, f, ahead);
      if constexpr (P::OA || P::OB) {
        load(GT_AT(2 + PF), true, 0, ahead);
        load(GT_AT(2 + PF), true, 1, ahead);
        load(GT_AT(1 + PF), true, 2, row_of(t + 1 + PF));
      }
      load_mask(GT_AT(PF), t + PF);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        constexpr int up = k, mid = (k + 1) % BW, down = (k + 2) % BW;  // slots of the three rows
        u32x4 b[10];
        if (P::odd(c)) {
          b[0] = B[c][0][up];
          b[2] = B[c][2][mid];
          b[3] = B[c][0][down];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            b[1][e] = hi ? B[c][1][mid][e] : B[c][1][up][e];
            b[4][e] = hi ? 0u : B[c][1][down][e];
          }
        } else if (PAIRS) {
          halves(B[c][0][down], B[c][1][down], F[c][0][down], F[c][1][down]);
          b[0] = F[c][0][up];
          b[5] = F[c][1][up];
          halves(B[c][2][up], B[c][0][mid], b[1], b[6]);
          halves(B[c][1][mid], B[c][2][mid], b[2], b[7]);
          b[3] = F[c][0][down];
          b[8] = F[c][1][down];
          halves(B[c][2][down], u32x4{0u, 0u, 0u, 0u}, b[4], b[9]);
        } else {
#pragma unroll
          for (int i = 0; i < 9; ++i) b[i] = B[c][i % 3][(k + i / 3) % BW];
        }
#pragma unroll
        for (int i = 0; i < P::steps(c); ++i) {
          const int step = P::step0(c) + i;
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[j] = mfma32(__builtin_bit_cast(uint4, step < AREG ? A[step < AREG ? step : 0][j]
                                                                     : Al[step < AREG ? 0 : step - AREG][j][lane]),
                               __builtin_bit_cast(uint4, b[i]), acc[j]);
        }
      }
      finish(T, t);
    };
    // the rows the first PF steps would have asked for
    auto warm = [&](auto Mv) {
      constexpr int m = decltype(Mv)::value;
      if constexpr (m < 2 + PF) {
        const RowAt r = row_of(m);
#pragma unroll
        for (int f = 0; f < 3; ++f) load(Mv, false, f, r);
        load(Mv, true, 0, r);
        load(Mv, true, 1, r);
        if constexpr (m >= 1 && m < 1 + PF) load(Mv, true, 2, r);
        if constexpr (m < PF) load_mask(Mv, m);
      }
    };
    warm(std::integral_constant<int, 0>{});
    warm(std::integral_constant<int, 1>{});
    warm(std::integral_constant<int, 2>{});
    warm(std::integral_constant<int, 3>{});
    warm(std::integral_constant<int, 4>{});
    if constexpr (PAIRS) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (!P::odd(c))
#pragma unroll
          for (int m = 0; m < 2; ++m) halves(B[c][0][m], B[c][1][m], F[c][0][m], F[c][1][m]);
    }
#define GT_ROW(K)                                    \
  if constexpr (K < BW) {                            \
    row(std::integral_constant<int, K % BW>{}, t);   \
    if (++t == rows) break;                          \
  }
    for (int t = 0;;) {
      GT_ROW(0)
      GT_ROW(1)
      GT_ROW(2)
      GT_ROW(3)
      GT_ROW(4)
      GT_ROW(5)
    }
#undef GT_ROW
#undef GT_AT
  }
}

// ---- convolution, weight gradient -----------------------------------------
// dW[co][tap][ci] = sum over pixels p of dPre[p][co] * x[p + off(tap)][ci],
// with dPre the output gradient (masked by the ReLU of the forward output by
// the kernel that made it). A block owns kWBands bands of kWR image rows of
// one image (its split) and NCO x NCI 16-channel fragments of (co, ci); wave w
// takes row w of each band. The four waves' sums are added in wave order
// through LDS, and the blocks of the first ci group also sum dPre against
// ones (the bias).
constexpr int kWR = 4;
constexpr size_t kWRed = 4 * 36 * 64 * sizeof(float);  // the four waves' sums of one (a, b) pair
// Bands of kWR rows per block: a block's sums cover kWBands bands (its split),
// which halves the partial sums written and reduced against one band per block.
constexpr int kWBands = 2;

// The end of a weight-gradient block: the waves exchange their sums through
// LDS (red, kWRed bytes), one (a, b) pair at a time; each adds a quarter of
// them in wave order and writes it to the block's row of partial sums (out:
// weights, then the bias at nw). The caller has synchronised the block after
// its last LDS read. With wave 0 adding all of them, the weight gradients
// of a 2x119x140 batch took 13 to 20 us each; so, 11 to 18.
template <int NCO, int NCI>
__device__ __forceinline__ void wgrad_finish(float* red, v4f (&acc)[9][NCO][NCI], v4f (&bacc)[NCO], bool bias,
                                             float* __restrict__ out, size_t nw, int cin, int co0, int ci0, int wave,
                                             int lane) {
#pragma unroll
  for (int a = 0; a < NCO; ++a)
#pragma unroll
    for (int b = 0; b < NCI; ++b) {
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * 36 + t * 4 + r) * 64 + lane] = acc[t][a][b][r];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        const int i = wave * 9 + k, t = i >> 2, r = i & 3;
        float v = red[i * 64 + lane];
        v += red[(36 + i) * 64 + lane];
        v += red[(72 + i) * 64 + lane];
        v += red[(108 + i) * 64 + lane];
        const int co = co0 + a * 16 + (lane >> 4) * 4 + r;
        const int ci = ci0 + b * 16 + (lane & 15);
        out[uint32_t((co * 9 + t) * cin + ci)] = v;
      }
    }
  if (bias) {
    __syncthreads();
    if (wave > 0) {
#pragma unroll
      for (int a = 0; a < NCO; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[((wave - 1) * 4 * NCO + a * 4 + r) * 64 + lane] = bacc[a][r];
    }
    __syncthreads();
    if (wave == 0 && (lane & 15) == 0) {  // column 0 of the all-ones product
#pragma unroll
      for (int a = 0; a < NCO; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = bacc[a][r];
          v += red[((0 * NCO + a) * 4 + r) * 64 + lane];
          v += red[((1 * NCO + a) * 4 + r) * 64 + lane];
          v += red[((2 * NCO + a) * 4 + r) * 64 + lane];
          out[nw + co0 + a * 16 + (lane >> 4) * 4 + r] = v;
        }
    }
  }
}

// The kernel walks its bands in tiles of TC columns. dPre (kWR rows x TC
// columns) and x (kWR + 2 rows x TC + 2 columns: one beyond the tile on each
// side) lie in LDS as they lie in HBM, one 32-byte row of 16 channels per
// pixel, in one region per 16-channel fragment, copied straight from global
// memory by buffer loads that write LDS (each region from its own tensor, so
// a block's channels may straddle the decoder concatenation); the next tile's
// copy runs while the waves work on this one. The MFMA
// operands come from ds_read_b64_tr_b16: over 16 lanes, lane l names 4
// channels of pixel row (l >> 2) & 3 of a 4 x 16 block and receives channel
// l's 4 pixels, so two reads give a lane its 8 K values (pixels) and a column
// tap is an offset of the pixel index. Slots are swizzled by bit 3 of the
// pixel, which puts the two 16-lane groups of a read pass (pixels 8 apart) in
// different banks. The buffer resources start at the first row the block's
// bands read, so offsets stay small for tensors of any size (kWBands * kWR + 2
// rows of the widest tensor must stay below 2 GB).
template <int TC>  // tile columns
constexpr int wgt_dslots() {  // 16-byte slots of one dPre fragment region
  return (kWR * TC * 2 + 63) / 64 * 64;
}
template <int TC>
constexpr int wgt_xslots() {  // ... of one x fragment region (TC + 2 columns)
  return ((kWR + 2) * (TC + 2) * 2 + 63) / 64 * 64;
}

__device__ __forceinline__ int wgt_slot(int p, int k) {  // piece k (0, 1) of pixel p
  return (2 * p + k) ^ (((p >> 3) & 1) << 3);
}
__device__ __forceinline__ int wgt_pixel(int slot) {  // the pixel of a slot (wgt_slot is its own inverse on bit 3)
  const int q = slot >> 1;
  return q ^ (((q >> 3) & 1) << 2);
}

template <int NCO, int NCI, int TC>
constexpr size_t wgrad_tr_lds_bytes() {  // two buffers
  return std::max(size_t(2) * (NCO * wgt_dslots<TC>() + NCI * wgt_xslots<TC>()) * 16, kWRed);
}

typedef short v4s __attribute__((ext_vector_type(4)));

// The 8 K values of this lane for a 16 x 32 operand whose K runs over the
// pixels p0 + 0 .. 31 of a fragment region (byte address base).
__device__ __forceinline__ uint4 wgt_operand(const char* base, int p0, int lane) {
  const int g = lane >> 4, r = (lane >> 2) & 3, c = lane & 3;
  u32x2 v[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int p = p0 + 8 * g + 4 * h + r;
    const char* a = base + wgt_slot(p, c >> 1) * 16 + (c & 1) * 8;
    v[h] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (__attribute__((address_space(3))) v4s*)((const lds_void*)a)));
  }
  return make_uint4(v[0].x, v[0].y, v[1].x, v[1].y);
}

template <int NCO, int NCI, int TC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_wgrad_tr(
    const uint16_t* __restrict__ x, int cin, const uint16_t* __restrict__ xa, int ca, const uint16_t* __restrict__ dy,
    int cout, int N, int H, int W, int nsplit, int ncog, int ci_first, float* __restrict__ partial) {
  constexpr int kWDS = wgt_dslots<TC>(), kWXS = wgt_xslots<TC>(), kWXC = TC + 2;
  constexpr int BUF = NCO * kWDS + NCI * kWXS;  // slots of one buffer: dPre regions, then x regions
  extern __shared__ uint4 wlds4[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.x / nsplit, band0 = (blockIdx.x % nsplit) * kWBands;
  const int co0 = (blockIdx.y % ncog) * NCO * 16, ci0 = ci_first + (blockIdx.y / ncog) * NCI * 16;
  const bool bias = ci0 == 0;  // uniform over the block
  const int cx = cin - ca;
  // rows [hb, he) hold everything the block reads (x's halo row above and below included)
  const int hb = max(band0 * kWR - 1, 0), he = min((band0 + kWBands) * kWR + 1, H);
  const i32x4 rd = buffer_rsrc(dy + (size_t(n) * H + hb) * W * cout, uint32_t(size_t(he - hb) * W * cout * 2));
  const i32x4 rx = buffer_rsrc(x + (size_t(n) * H + hb) * W * cx, uint32_t(size_t(he - hb) * W * cx * 2));
  const int hb2 = hb / 2, he2 = (he + 1) / 2;  // the same rows of the half-resolution part
  const i32x4 ra = xa ? buffer_rsrc(xa + (size_t(n) * (H / 2) + hb2) * (W / 2) * ca,
                                    uint32_t(size_t(he2 - hb2) * (W / 2) * ca * 2))
                      : buffer_rsrc(x, 0u);
  v4f acc[9][NCO][NCI], bacc[NCO];
#pragma unroll
  for (int a = 0; a < NCO; ++a) {
    bacc[a] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int b = 0; b < NCI; ++b) acc[t][a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  // the copies of the tile at rows r0.., column c0 into buffer buf: wave w issues slots
  // [64 i, 64 i + 64) of each region for i = w, w + 4, ...
  auto copy = [&](uint4* buf, int r0, int c0) {
#pragma unroll
    for (int a = 0; a < NCO; ++a) {
#pragma unroll
      for (int i0 = 0; i0 < kWDS / 64; i0 += 4) {
        const int i = i0 + wave, sl = i * 64 + lane, p = wgt_pixel(sl);
        const int h = r0 + p / TC, w = c0 + p % TC;
        uint32_t off = kOutOfRange;
        if (p < kWR * TC && h < H && w < W)
          off = uint32_t((((size_t(h) - hb) * W + w) * cout + co0 + 16 * a + 8 * (sl & 1)) * 2);
        lds_copy16(buf + a * kWDS + i * 64, rd, off);
      }
    }
#pragma unroll
    for (int b = 0; b < NCI; ++b) {
      const int c = ci0 + 16 * b;  // the fragment's first channel: below ca it comes from xa at half resolution
      const bool half_res = c < ca;
#pragma unroll
      for (int i0 = 0; i0 < kWXS / 64; i0 += 4) {
        const int i = i0 + wave;
        if (i < kWXS / 64) {
          const int sl = i * 64 + lane, p = wgt_pixel(sl);
          const int h = r0 - 1 + p / kWXC, w = c0 - 1 + p % kWXC;
          uint32_t off = kOutOfRange;
          if (p < (kWR + 2) * kWXC && h >= 0 && h < H && w >= 0 && w < W)
            off = half_res ? uint32_t((((size_t(h) / 2 - hb2) * (W / 2) + w / 2) * ca + c + 8 * (sl & 1)) * 2)
                           : uint32_t((((size_t(h) - hb) * W + w) * cx + c - ca + 8 * (sl & 1)) * 2);
          lds_copy16(buf + NCO * kWDS + b * kWXS + i * 64, half_res ? ra : rx, off);
        }
      }
    }
  };
  const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);  // bf16 1.0 x 8
  // steps: the tiles of band band0, then of band0 + 1, ...
  const int ntiles = (W + TC - 1) / TC;
  const int nb = min(kWBands, (H + kWR - 1) / kWR - band0), S = nb * ntiles;
  copy(wlds4, band0 * kWR, 0);
  for (int t = 0; t < S; ++t) {
    uint4* cur = wlds4 + (t & 1) * BUF;
    __builtin_amdgcn_s_waitcnt(kWaitVm0);  // this wave's copies of step t are done
    lds_barrier();                        // ... and every wave's; the other buffer's reads are done
    if (t + 1 < S) copy(wlds4 + ((t + 1) & 1) * BUF, (band0 + (t + 1) / ntiles) * kWR, (t + 1) % ntiles * TC);
    if ((band0 + t / ntiles) * kWR + wave >= H) continue;  // this wave's row is past the image: its dPre is zero
    const char* dT = reinterpret_cast<const char*>(cur);
    const char* xT = reinterpret_cast<const char*>(cur + NCO * kWDS);
#pragma unroll
    for (int kc = 0; kc < TC / 32; ++kc) {
      uint4 A[NCO];
#pragma unroll
      for (int a = 0; a < NCO; ++a) A[a] = wgt_operand(dT + a * kWDS * 16, wave * TC + 32 * kc, lane);
#pragma unroll
      for (int b = 0; b < NCI; ++b) {
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
          const int dr = tap / 3, dx = tap % 3 - 1;
          const uint4 B = wgt_operand(xT + b * kWXS * 16, (wave + dr) * kWXC + 32 * kc + 1 + dx, lane);
#pragma unroll
          for (int a = 0; a < NCO; ++a) acc[tap][a][b] = mfma32(A[a], B, acc[tap][a][b]);
        }
      }
      if (bias) {
#pragma unroll
        for (int a = 0; a < NCO; ++a) bacc[a] = mfma32(A[a], ones, bacc[a]);
      }
    }
  }
  __syncthreads();  // every wave is done with the tiles
  const size_t nw = size_t(cout) * 9 * cin;
  wgrad_finish<NCO, NCI>(reinterpret_cast<float*>(wlds4), acc, bacc, bias,
                         partial + size_t(blockIdx.x) * (nw + cout), nw, cin, co0, ci0, wave, lane);
}

// out[i] = sum over s < splits of partial[s * stride + i], i < n. A block of 256 threads
// owns 32 consecutive outputs; its 8 thread groups sum the splits congruent
// to their group index mod 8, in increasing order, and group sums are added
// in group order: a fixed order, so results are deterministic.
__global__ __launch_bounds__(256) void k_reduce(const float* __restrict__ partial, int splits, size_t n,
                                                size_t stride, float* __restrict__ out) {
  __shared__ float part[8][33];
  const int o = threadIdx.x & 31, g = threadIdx.x >> 5;
  const size_t i = blockIdx.x * size_t(32) + o;
  float acc = 0.f;
  if (i < n) {
    int k = g;
    for (; k + 24 < splits; k += 32) {  // four independent loads in flight
      const float a = partial[size_t(k) * stride + i], b = partial[size_t(k + 8) * stride + i];
      const float c = partial[size_t(k + 16) * stride + i], d = partial[size_t(k + 24) * stride + i];
      acc += a;
      acc += b;
      acc += c;
      acc += d;
    }
    for (; k < splits; k += 8) acc += partial[size_t(k) * stride + i];
  }
  part[g][o] = acc;
  __syncthreads();
  if (g == 0 && i < n) {
    float t = part[0][o];
#pragma unroll
    for (int j = 1; j < 8; ++j) t += part[j][o];
    out[i] = t;
  }
}

// ---- pooling, upsampling, concatenation -----------------------------------

// Pieces of 8 channels (16 bytes): every channel count and offset here is a
// multiple of 16.
__device__ __forceinline__ void unpack8(uint4 v, float (&f)[8]) {
  const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = bf2f(uint16_t(u[k]));
    f[2 * k + 1] = bf2f(uint16_t(u[k] >> 16));
  }
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  uint32_t u[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) u[k] = uint32_t(f2bf(f[2 * k])) | (uint32_t(f2bf(f[2 * k + 1])) << 16);
  return make_uint4(u[0], u[1], u[2], u[3]);
}

__global__ void k_pool_bwd(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy,
                           const uint16_t* __restrict__ add, int add_c, int add_off, uint16_t* __restrict__ dx, int c,
                           int H, int W, size_t n8, int relu_mask) {
  // one 2x2 window and 8 channels per thread: n8 = windows * c / 8
  const int H2 = H / 2, W2 = W / 2, c8 = c / 8;
  for (size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x; i < n8; i += size_t(gridDim.x) * blockDim.x) {
    const int ch = int(i % c8) * 8;
    const size_t q = i / c8;
    const int w2 = int(q % W2);
    const size_t t = q / W2;
    const int h2 = int(t % H2);
    const size_t b = t / H2;
    const size_t p0 = (b * H + 2 * h2) * W + 2 * w2;
    const size_t px[4] = {p0, p0 + 1, p0 + W, p0 + W + 1};  // scan order
    float xv[4][8];
#pragma unroll
    for (int k = 0; k < 4; ++k) unpack8(*reinterpret_cast<const uint4*>(x + px[k] * c + ch), xv[k]);
    // per channel, the window's first maximum in scan order takes the gradient
    int arg[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float m = xv[0][e];
      arg[e] = 0;
#pragma unroll
      for (int k = 1; k < 4; ++k)
        if (xv[k][e] > m) { m = xv[k][e]; arg[e] = k; }
    }
    float up[8];
    unpack8(*reinterpret_cast<const uint4*>(dy + q * c + ch), up);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float g[8], ad[8];
      if (add) unpack8(*reinterpret_cast<const uint4*>(add + px[k] * add_c + add_off + ch), ad);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        g[e] = k == arg[e] ? up[e] : 0.f;
        if (add) g[e] += ad[e];
        if (relu_mask && !(xv[k][e] > 0.f)) g[e] = 0.f;  // x is the ReLU output
      }
      *reinterpret_cast<uint4*>(dx + px[k] * c + ch) = pack8(g);
    }
  }
}

__global__ void k_upcat_bwd(const uint16_t* __restrict__ dout, int ca, int cb, uint16_t* __restrict__ da,
                            const uint16_t* __restrict__ da_mask, int H, int W, size_t n8) {
  // 8 channels of one half-resolution pixel per thread: n8 = pixels * ca / 8
  const int c = ca + cb, H2 = H / 2, W2 = W / 2, ca8 = ca / 8;
  for (size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x; i < n8; i += size_t(gridDim.x) * blockDim.x) {
    const int ch = int(i % ca8) * 8;
    size_t q = i / ca8;
    const int w2 = int(q % W2);
    q /= W2;
    const int h2 = int(q % H2);
    const size_t b = q / H2;
    const size_t base = ((b * H + 2 * h2) * W + 2 * w2) * c + ch;
    float v0[8], v1[8], v2[8], v3[8], o[8];
    unpack8(*reinterpret_cast<const uint4*>(dout + base), v0);
    unpack8(*reinterpret_cast<const uint4*>(dout + base + c), v1);
    unpack8(*reinterpret_cast<const uint4*>(dout + base + size_t(W) * c), v2);
    unpack8(*reinterpret_cast<const uint4*>(dout + base + size_t(W) * c + c), v3);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float s = v0[e] + v1[e];
      s += v2[e] + v3[e];
      o[e] = s;
    }
    const size_t off = (i / ca8) * ca + ch;
    uint4 r = pack8(o);
    if (da_mask) r = mask8(r, *reinterpret_cast<const uint4*>(da_mask + off));
    *reinterpret_cast<uint4*>(da + off) = r;
  }
}

// ---- input, loss, output ---------------------------------------------------
constexpr float kHalvesClip = 2.f;  // bound of the halves' log difference (channels 9-11)

__global__ void k_pack(const float* __restrict__ beauty, const float* __restrict__ beauty_b,
                       const float* __restrict__ albedo, const float* __restrict__ normal, int h, int w,
                       uint16_t* __restrict__ x, int Hp, int Wp, size_t npx) {
  for (size_t p = blockIdx.x * size_t(blockDim.x) + threadIdx.x; p < npx; p += size_t(gridDim.x) * blockDim.x) {
    const int xx = int(p % Wp);
    const size_t t = p / Wp;
    const int yy = int(t % Hp);
    const size_t b = t / Hp;
    const size_t s = ((b * h + min(yy, h - 1)) * w + min(xx, w - 1)) * 3;
    uint16_t v[16];
#pragma unroll
    for (int c = 9; c < 16; ++c) v[c] = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float a = beauty[s + c];
      if (beauty_b) {
        const float b2 = beauty_b[s + c];
        v[c] = f2bf(log1pf(fmaxf(0.5f * (a + b2), 0.f)));
        // clipped: a firefly's log ratio (up to ~10) would take the network far outside
        // what it was trained on, while a ratio of e^2 already marks one half as an outlier
        v[9 + c] = f2bf(fminf(fmaxf(log1pf(fmaxf(a, 0.f)) - log1pf(fmaxf(b2, 0.f)), -kHalvesClip), kHalvesClip));
      } else {
        v[c] = f2bf(log1pf(fmaxf(a, 0.f)));
      }
      v[3 + c] = f2bf(albedo[s + c]);
      v[6 + c] = f2bf(normal[s + c]);
    }
    uint32_t u[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k] = uint32_t(v[2 * k]) | (uint32_t(v[2 * k + 1]) << 16);
    uint4* o = reinterpret_cast<uint4*>(x + p * 16);  // the pixel's 32 bytes in two 16-byte stores
    o[0] = make_uint4(u[0], u[1], u[2], u[3]);
    o[1] = make_uint4(u[4], u[5], u[6], u[7]);
  }
}

__device__ __forceinline__ float tone(float z) { return z >= 0.f ? 1.f - expf(-z) : z; }
__device__ __forceinline__ float dtone(float z) { return z >= 0.f ? expf(-z) : 1.f; }
constexpr float kRelL2Eps = 0.01f;

// One element's loss and d loss / d z.
template <int KIND>
__device__ __forceinline__ float loss_elem(float zc, float tc, float* dl) {
  if (KIND == GT_DENOISE_LOSS_REL_L2) {
    const float y = zc >= 0.f ? expm1f(zc) : zc;
    const float dy = zc >= 0.f ? expf(zc) : 1.f;
    const float yc = fmaxf(y, 0.f);
    const float inv = 1.f / (yc * yc + kRelL2Eps);  // held constant: the gradient's root is the mean target
    const float d = y - tc;
    *dl = 2.f * d * inv * dy;
    return d * d * inv;
  }
  const float d = tone(zc) - tc / (1.f + tc);
  *dl = (d > 0.f ? 1.f : (d < 0.f ? -1.f : 0.f)) * dtone(zc);
  return fabsf(d);
}

template <int KIND>
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ z, const float* __restrict__ target, int h,
                                              int w, uint16_t* __restrict__ dz, float* __restrict__ partial, int Hp,
                                              int Wp, size_t npx, float inv_count) {
  __shared__ float red[256];
  float acc = 0.f;
  for (size_t p = blockIdx.x * size_t(blockDim.x) + threadIdx.x; p < npx; p += size_t(gridDim.x) * blockDim.x) {
    const int xx = int(p % Wp);
    const size_t t = p / Wp;
    const int yy = int(t % Hp);
    const size_t b = t / Hp;
    uint4* g = reinterpret_cast<uint4*>(dz + p * 16);  // channels 0-7, 8-15; only 0-2 carry a gradient
    g[1] = make_uint4(0, 0, 0, 0);
    if (yy >= h || xx >= w) {
      g[0] = make_uint4(0, 0, 0, 0);
      continue;
    }
    const float* tg = target + ((b * h + yy) * w + xx) * 3;
    const float4 zp = *reinterpret_cast<const float4*>(z + p * 16);
    const float zc[3] = {zp.x, zp.y, zp.z};
    uint16_t gc[3];
    for (int c = 0; c < 3; ++c) {
      float dl;
      acc += loss_elem<KIND>(zc[c], fmaxf(tg[c], 0.f), &dl);
      gc[c] = f2bf(dl * inv_count);
    }
    g[0] = make_uint4(uint32_t(gc[0]) | (uint32_t(gc[1]) << 16), uint32_t(gc[2]), 0, 0);
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_unpack(const float* __restrict__ z, float* __restrict__ out, int h, int w, int Hp, int Wp,
                         size_t n) {
  for (size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    const int c = int(i % 3);
    const size_t p = i / 3;
    const int xx = int(p % w);
    const size_t t = p / w;
    const int yy = int(t % h);
    const size_t b = t / h;
    out[i] = expm1f(fmaxf(z[((b * Hp + yy) * Wp + xx) * 16 + c], 0.f));
  }
}

// ---- optimiser ---------------------------------------------------------------
__global__ void k_adam_all(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                           float* __restrict__ v, size_t n, float lr, float b1, float b2, float eps, float c1, float c2,
                           const AdamSeg* __restrict__ segs, int nseg) {
  for (size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    for (int k = 0; k < nseg; ++k) {  // the segment holding i, if any (biases have no copies)
      const AdamSeg sg = segs[k];
      const size_t cin = size_t(sg.cin), cout = size_t(sg.cout);
      if (i < sg.w_off || i - sg.w_off >= cout * 9 * cin) continue;
      const size_t j = i - sg.w_off;
      const uint16_t b = f2bf(pi);
      sg.w16[j] = b;
      const size_t ci = j % cin, t = (j / cin) % 9, co = j / (cin * 9);
      sg.wt16[(ci * 9 + t) * cout + co] = b;
      break;
    }
  }
}

__global__ void k_to_bf16(const float* __restrict__ p, uint16_t* __restrict__ w16, uint16_t* __restrict__ wt16,
                          int cin, int cout, size_t n) {
  for (size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    const uint16_t b = f2bf(p[i]);
    w16[i] = b;
    const size_t ci = i % cin, t = (i / cin) % 9, co = i / (size_t(cin) * 9);
    wt16[(ci * 9 + t) * cout + co] = b;
  }
}

unsigned grid_for(size_t n, unsigned block = 256) {
  size_t g = (n + block - 1) / block;
  return unsigned(g < 65535u * 8 ? (g ? g : 1) : 65535u * 8);
}

template <bool DGRAD, bool F32, int NT>
void launch_nt(hipStream_t s, const uint16_t* x, const uint16_t* mask, int cin, const uint16_t* xa, int ca,
               const uint16_t* w, const float* bias, void* y, uint16_t* pooled, int cout, int co_first, int groups,
               Dims d, int relu, const uint16_t* omask) {
  const int nrt = (d.h + kTR - 1) / kTR, nct = (d.w + kTC - 1) / kTC;
  constexpr size_t lds = conv_lds_bytes<NT>();
  static const hipError_t attr =  // once per instantiation: allow more than 64 KiB of LDS
      hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conv<NT, DGRAD, F32>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
  (void)attr;
  hipLaunchKernelGGL((k_conv<NT, DGRAD, F32>), dim3(d.n * nrt * nct, groups), dim3(256), lds, s, x, mask, cin, xa,
                     ca, w, bias, y, pooled, cout, co_first, d.h, d.w, nrt, nct, relu, omask);
}

// Output channels in groups of 64 (NT = 4), then one launch for the rest.
int device_cus() {
  static std::atomic<int> cus{0};
  int n = cus.load(std::memory_order_relaxed);
  if (!n) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cus.store(n, std::memory_order_relaxed);
  }
  return n;
}

// How an instance is built: waves per SIMD (512 registers per lane, shared), rows read ahead (1 to 3), and steps
// whose weights stay in LDS.
template <int WAVES_, int PF_, int LDSA_ = 0>
struct RowsCfg {
  static constexpr int WAVES = WAVES_, PF = PF_, LDSA = LDSA_;
};

template <int CA, int CB, bool PAIRS, int NT, RowsMode MODE, class CFG>
bool launch_rows_nt(hipStream_t s, RowsJob q) {
  const RowsSplit p = rows_split(q.N, q.H, q.W, q.groups, device_cus() * 4 * CFG::WAVES);
  const size_t widest = std::max({CA * 2, CB * 2, q.cout * (MODE == ROWS_F32 ? 4 : 2), 12});
  if (size_t(p.rows + 2) * q.W * widest >= kRowsBytes) return false;
  q.seg_rows = p.rows;
  q.nseg = p.segs;
  q.nstrip = p.strips;
  hipLaunchKernelGGL((k_conv_rows<CA, CB, PAIRS, NT, MODE, CFG::WAVES, CFG::PF, CFG::LDSA>), dim3(8 * p.blocks), dim3(256), 0, s, q);
  return true;
}

template <int CA, int CB, bool PAIRS, int NT, class CFG>
bool launch_rows_mode(hipStream_t s, const RowsJob& q, RowsMode mode) {
  switch (mode) {
    case ROWS_FWD: return launch_rows_nt<CA, CB, PAIRS, NT, ROWS_FWD, CFG>(s, q);
    case ROWS_POOL: if constexpr (CA == 0) return launch_rows_nt<CA, CB, PAIRS, NT, ROWS_POOL, CFG>(s, q); else return false;
    case ROWS_GRAD: if constexpr (CA == 0) return launch_rows_nt<CA, CB, false, NT, ROWS_GRAD, CFG>(s, q); else return false;
    case ROWS_GRAD_MASK: if constexpr (CA == 0) return launch_rows_nt<CA, CB, false, NT, ROWS_GRAD_MASK, CFG>(s, q); else return false;
    default: return false;
  }
}

// The output channels in groups of two fragments; an odd one in a launch of its own.
template <int CA, int CB, bool PAIRS, int NT, class CFG, class CFG1 = CFG>
bool launch_rows_all(hipStream_t s, RowsJob q, RowsMode mode) {
  const int frags = q.cout / 16, full = frags / NT, rest = frags % NT;
  q.groups = full;
  q.co_first = 0;
  if (full && !launch_rows_mode<CA, CB, PAIRS, NT, CFG>(s, q, mode)) return false;
  q.groups = 1;
  q.co_first = full * NT * 16;
  return rest == 0 || launch_rows_mode<CA, CB, PAIRS, 1, CFG1>(s, q, mode);
}

// ... of a layer whose output channels are whole groups.
template <int CA, int CB, bool PAIRS, int NT, class CFG>
bool launch_rows_fit(hipStream_t s, RowsJob q, RowsMode mode) {
  q.groups = q.cout / 16 / NT;
  q.co_first = 0;
  return launch_rows_mode<CA, CB, PAIRS, NT, CFG>(s, q, mode);
}

// The layers that take the row kernel (rows_frags); false for the others, which take k_conv. Measured on one MI355X (us;
// k_conv or the persistent LDS kernel that stood here before, then this one) on a 1920x1080 frame: 16->32 58 and 54,
// 32->32 76 and 54, 32->48 39 and 29, 48->48 47 and 32, 48->64 32 and 13, 64->64 34 and 22, 64->96 18 and 15, 96->96 22
// and 15, 48+32->32 171 and 117, 64+48->48 87 and 53, 96+64->64 62 and 45, the output 52 and 45, 80->32 179 and 107 (228
// with k_conv). 128 channels in a part lost and have no instance (128->128: 14 and 20; a wave's weights fill its registers
// for a few rows' work). Parts of 80 and 112 channels (but for 80->32) and the other concatenations have none either: no
// one has been built or measured. An instance takes as many output channels per wave as its registers hold, which divides
// the fragment loads by them; the widest keep weights in LDS, and one wave per SIMD beat two that spill.
//
// PAIRS follows the layer, in the forward direction, so that its images stay the bits of the kernel that made it before:
// taps pair over 16 channels in the shapes of the default network's full-resolution level and of level 1's 32->48 and
// 48->48 (the persistent kernel's), 32 channels to a tap elsewhere (k_conv's). Data gradients never pair.
bool launch_rows(hipStream_t s, const RowsJob& q, int ca, int cb, RowsMode mode) {
  if (mode == ROWS_F32 || mode == ROWS_RADIANCE) {
    if (ca || cb != 32 || q.cout != 16) return false;
    RowsJob r = q;
    r.groups = 1;
    r.co_first = 0;
    return mode == ROWS_F32 ? launch_rows_nt<0, 32, true, 1, ROWS_F32, RowsCfg<2, 2>>(s, r)
                            : launch_rows_nt<0, 32, true, 1, ROWS_RADIANCE, RowsCfg<2, 2>>(s, r);
  }
  const int64_t tiles = int64_t(q.N) * ((q.H + kTR - 1) / kTR) * ((q.W + kTC - 1) / kTC);
  const int nt = rows_frags(ca, cb, q.cout, mode == ROWS_GRAD || mode == ROWS_GRAD_MASK, tiles);
  if (nt == 0) return false;
  switch (ca * 1000 + cb) {
    case 16:
      if (nt == 3) return launch_rows_fit<0, 16, true, 3, RowsCfg<2, 2>>(s, q, mode);
      return launch_rows_all<0, 16, true, 2, RowsCfg<4, 1>>(s, q, mode);
    case 32:
      if (nt == 3) return launch_rows_fit<0, 32, true, 3, RowsCfg<2, 2>>(s, q, mode);
      if (q.cout == 32) return launch_rows_fit<0, 32, true, 2, RowsCfg<2, 2>>(s, q, mode);
      // five fragments a wave where they divide: 32->80 in one launch, 66 us at 16x256x256; 61 + 51 in launches of 2 and 1
      if (nt == 5) return launch_rows_fit<0, 32, false, 5, RowsCfg<1, 2>>(s, q, mode);
      return launch_rows_all<0, 32, false, 2, RowsCfg<2, 2>>(s, q, mode);
    case 48:
      if (nt == 3) return launch_rows_fit<0, 48, true, 3, RowsCfg<1, 2>>(s, q, mode);
      return launch_rows_all<0, 48, false, 2, RowsCfg<1, 2>, RowsCfg<2, 1>>(s, q, mode);
    case 64:
      if (nt == 3) return launch_rows_fit<0, 64, false, 3, RowsCfg<1, 1>>(s, q, mode);
      return launch_rows_all<0, 64, false, 2, RowsCfg<1, 1>, RowsCfg<2, 1>>(s, q, mode);
    case 80: {  // an encoder level's first layer
      if (mode != ROWS_FWD) return false;
      RowsJob r = q;
      r.groups = 1;
      r.co_first = 0;
      return launch_rows_nt<0, 80, false, 2, ROWS_FWD, RowsCfg<1, 1>>(s, r);
    }
    case 96:
      if (nt == 3) return launch_rows_fit<0, 96, false, 3, RowsCfg<1, 1, 6>>(s, q, mode);
      return launch_rows_all<0, 96, false, 2, RowsCfg<1, 1>>(s, q, mode);
    case 48032: return launch_rows_fit<48, 32, true, 2, RowsCfg<1, 1>>(s, q, mode);
    case 64032: return launch_rows_fit<64, 32, false, 2, RowsCfg<1, 1>>(s, q, mode);
    case 64048: return launch_rows_fit<64, 48, false, 3, RowsCfg<1, 1, 12>>(s, q, mode);
    case 96064: return launch_rows_fit<96, 64, false, 2, RowsCfg<1, 1, 26>>(s, q, mode);
    default: return false;
  }
}

template <bool DGRAD, bool F32>
void launch_groups(hipStream_t s, int nt, int first_frag, int groups, const uint16_t* x, const uint16_t* mask, int cin,
                   const uint16_t* xa, int ca, const uint16_t* w, const float* bias, void* y, int cout, Dims d,
                   int relu, uint16_t* pooled, const uint16_t* omask) {
  const int c0 = first_frag * 16;
  switch (nt) {
    case 1: launch_nt<DGRAD, F32, 1>(s, x, mask, cin, xa, ca, w, bias, y, pooled, cout, c0, groups, d, relu, omask); break;
    case 2: launch_nt<DGRAD, F32, 2>(s, x, mask, cin, xa, ca, w, bias, y, pooled, cout, c0, groups, d, relu, omask); break;
    case 3: launch_nt<DGRAD, F32, 3>(s, x, mask, cin, xa, ca, w, bias, y, pooled, cout, c0, groups, d, relu, omask); break;
    default: launch_nt<DGRAD, F32, 4>(s, x, mask, cin, xa, ca, w, bias, y, pooled, cout, c0, groups, d, relu, omask); break;
  }
}

// The row kernel for the layers it takes. Otherwise output channels in groups
// of NT 16-channel fragments (conv_frags), then one launch for the rest.
template <bool DGRAD, bool F32>
void launch_conv(hipStream_t s, const uint16_t* x, const uint16_t* mask, int cin, const uint16_t* xa, int ca,
                 const uint16_t* w, const float* bias, void* y, int cout, Dims d, int relu,
                 uint16_t* pooled = nullptr, const uint16_t* omask = nullptr) {
  if (!mask) {
    RowsJob q{};
    q.x = x; q.xa = xa; q.wgt = w; q.bias = bias; q.y = y; q.pooled = pooled; q.omask = omask;
    q.cout = cout; q.N = d.n; q.H = d.h; q.W = d.w;
    const RowsMode mode = F32 ? ROWS_F32 : DGRAD ? (omask ? ROWS_GRAD_MASK : ROWS_GRAD) : pooled ? ROWS_POOL : ROWS_FWD;
    const bool like = F32 ? !relu : DGRAD || (relu && !omask);  // a bias with ReLU, or neither, as the modes have them
    if (like && launch_rows(s, q, xa ? ca : 0, xa ? cin - ca : cin, mode)) return;
  }
  const int tiles = d.n * ((d.h + kTR - 1) / kTR) * ((d.w + kTC - 1) / kTC);
  const int nt = conv_frags(tiles);
  const int frags = cout / 16, full = frags / nt, rest = frags % nt;
  if (full) launch_groups<DGRAD, F32>(s, nt, 0, full, x, mask, cin, xa, ca, w, bias, y, cout, d, relu, pooled, omask);
  if (rest)
    launch_groups<DGRAD, F32>(s, rest, full * nt, 1, x, mask, cin, xa, ca, w, bias, y, cout, d, relu, pooled, omask);
}

// Weight-gradient splits: one per kWBands bands of kWR rows of one image.
int wgrad_splits(Dims d) { return d.n * (((d.h + kWR - 1) / kWR + kWBands - 1) / kWBands); }

template <int NCO, int NCI, int TC>
void launch_wgrad_tr(hipStream_t s, const uint16_t* x, int cin, const uint16_t* xa, int ca, const uint16_t* dy,
                     int cout, Dims d, float* partial, int ci_first, int ncig) {
  constexpr size_t lds = wgrad_tr_lds_bytes<NCO, NCI, TC>();
  static const hipError_t attr =  // once per instantiation: allow more than 64 KiB of LDS
      hipFuncSetAttribute(reinterpret_cast<const void*>(&k_wgrad_tr<NCO, NCI, TC>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
  (void)attr;
  const int ncog = cout / (NCO * 16);
  const int nsplit = wgrad_splits(d) / d.n;
  hipLaunchKernelGGL((k_wgrad_tr<NCO, NCI, TC>), dim3(d.n * nsplit, ncog * ncig), dim3(256), lds, s, x, cin, xa, ca,
                     dy, cout, d.n, d.h, d.w, nsplit, ncog, ci_first, partial);
}


}  // namespace

void conv_fwd(hipStream_t s, const uint16_t* x, int cin, const uint16_t* w, const float* bias, void* y, int cout,
              Dims d, bool relu, bool out_f32, uint16_t* pooled) {
  if (out_f32) launch_conv<false, true>(s, x, nullptr, cin, nullptr, 0, w, bias, y, cout, d, relu ? 1 : 0);
  else launch_conv<false, false>(s, x, nullptr, cin, nullptr, 0, w, bias, y, cout, d, relu ? 1 : 0, pooled);
}

bool conv_fwd_radiance(hipStream_t s, const uint16_t* x, int cin, const uint16_t* w, const float* bias, float* out,
                       int h, int w_img, Dims d) {
  if (cin != 32) return false;
  RowsJob q{};
  q.x = x; q.wgt = w; q.bias = bias; q.y = out; q.rh = h; q.rw = w_img; q.cout = 16; q.N = d.n; q.H = d.h; q.W = d.w;
  return launch_rows(s, q, 0, 32, ROWS_RADIANCE);
}

void conv_fwd_upcat(hipStream_t s, const uint16_t* a, int ca, const uint16_t* b, int cb, const uint16_t* w,
                    const float* bias, uint16_t* y, int cout, Dims d, bool relu) {
  launch_conv<false, false>(s, b, nullptr, ca + cb, a, ca, w, bias, y, cout, d, relu ? 1 : 0);
}

void conv_dgrad(hipStream_t s, const uint16_t* dy, const uint16_t* y, int cout, const uint16_t* wt, uint16_t* dx,
                int cin, Dims d, const uint16_t* dx_mask) {
  // the transposed problem: input dy (cout channels), output dx (cin channels)
  launch_conv<true, false>(s, dy, y, cout, nullptr, 0, wt, nullptr, dx, cin, d, 0, nullptr, dx_mask);
}

size_t wgrad_scratch_floats(int cin, int cout, Dims d) {
  const size_t splits = size_t(wgrad_splits(d));
  return splits * (size_t(cout) * 9 * cin + cout);
}

void conv_wgrad(hipStream_t s, const uint16_t* x, int cin, const uint16_t* dy, int cout, Dims d, float* dw, float* db,
                float* scratch, size_t scratch_floats, const uint16_t* xa, int ca) {
  const int splits = wgrad_splits(d);
  const size_t nw = size_t(cout) * 9 * cin;
  if (scratch_floats < size_t(splits) * (nw + cout)) return;  // sized by wgrad_scratch_floats
  // a block's buffer resources span kWBands * kWR + 2 rows of the widest tensor (the network's
  // widths and 256 channels at most keep this far below 2 GB)
  if (size_t(kWBands * kWR + 2) * d.w * std::max(cin, cout) * 2 >= kOutOfRange) return;
  // Two output- and two input-channel fragments per block where the layer has them, so that
  // fewer blocks stage the same dPre and x tiles; an odd last input fragment takes a launch of its
  // own (it writes its own columns of the same partial rows).
  const int pairs = cin / 32, odd = (cin / 16) % 2;
  // Double-buffered tiles of 32 columns (two blocks of 2 x 2 fragments fit a CU with both buffers
  // only at that size; 1 x 2 and 1 x 1 also measured faster) or 64 (2 x 1).
  if ((cout / 16) % 2 == 0) {
    if (pairs) launch_wgrad_tr<2, 2, 32>(s, x, cin, xa, ca, dy, cout, d, scratch, 0, pairs);
    if (odd) launch_wgrad_tr<2, 1, 64>(s, x, cin, xa, ca, dy, cout, d, scratch, 32 * pairs, 1);
  } else {
    if (pairs) launch_wgrad_tr<1, 2, 32>(s, x, cin, xa, ca, dy, cout, d, scratch, 0, pairs);
    if (odd) launch_wgrad_tr<1, 1, 32>(s, x, cin, xa, ca, dy, cout, d, scratch, 32 * pairs, 1);
  }
  const size_t row = nw + cout;  // a split's partial sums: weights, then bias
  if (db == dw + nw) {  // the usual parameter layout: one reduction for both
    hipLaunchKernelGGL(k_reduce, dim3(unsigned((row + 31) / 32)), dim3(256), 0, s, scratch, splits, row, row, dw);
  } else {
    hipLaunchKernelGGL(k_reduce, dim3(unsigned((nw + 31) / 32)), dim3(256), 0, s, scratch, splits, nw, row, dw);
    hipLaunchKernelGGL(k_reduce, dim3(unsigned((size_t(cout) + 31) / 32)), dim3(256), 0, s, scratch + nw, splits,
                       size_t(cout), row, db);
  }
}

void pool_bwd(hipStream_t s, const uint16_t* x, const uint16_t* dy, const uint16_t* add, int add_c, int add_off,
              uint16_t* dx, int c, Dims d, bool relu_mask) {
  const size_t n8 = size_t(d.n) * (d.h / 2) * (d.w / 2) * (c / 8);  // windows x 8-channel pieces
  hipLaunchKernelGGL(k_pool_bwd, dim3(grid_for(n8)), dim3(256), 0, s, x, dy, add, add_c, add_off, dx, c, d.h, d.w,
                     n8, relu_mask ? 1 : 0);
}

void upcat_bwd(hipStream_t s, const uint16_t* dout, int ca, int cb, uint16_t* da, Dims d, const uint16_t* da_mask) {
  const size_t n8 = size_t(d.n) * (d.h / 2) * (d.w / 2) * (ca / 8);
  hipLaunchKernelGGL(k_upcat_bwd, dim3(grid_for(n8)), dim3(256), 0, s, dout, ca, cb, da, da_mask, d.h, d.w, n8);
}

void pack_input(hipStream_t s, const float* beauty, const float* beauty_b, const float* albedo, const float* normal,
                int h, int w, uint16_t* x, Dims dp) {
  const size_t n = size_t(dp.pixels());
  hipLaunchKernelGGL(k_pack, dim3(grid_for(n)), dim3(256), 0, s, beauty, beauty_b, albedo, normal, h, w, x, dp.h,
                     dp.w, n);
}

int loss_blocks(Dims dp) {
  const size_t n = size_t(dp.pixels());
  return int(std::min<size_t>((n + 255) / 256, 1024));
}

void loss(hipStream_t s, int kind, const float* z, const float* target, int h, int w, uint16_t* dz, float* partial,
          Dims dp) {
  const size_t n = size_t(dp.pixels());
  const float inv = 1.0f / float(size_t(dp.n) * h * w * 3);
  if (kind == GT_DENOISE_LOSS_REL_L2)
    hipLaunchKernelGGL(k_loss<GT_DENOISE_LOSS_REL_L2>, dim3(loss_blocks(dp)), dim3(256), 0, s, z, target, h, w, dz,
                       partial, dp.h, dp.w, n, inv);
  else
    hipLaunchKernelGGL(k_loss<GT_DENOISE_LOSS_L1_TONEMAP>, dim3(loss_blocks(dp)), dim3(256), 0, s, z, target, h, w,
                       dz, partial, dp.h, dp.w, n, inv);
}

void unpack_output(hipStream_t s, const float* z, float* out, int h, int w, Dims dp) {
  const size_t n = size_t(dp.n) * h * w * 3;
  hipLaunchKernelGGL(k_unpack, dim3(grid_for(n)), dim3(256), 0, s, z, out, h, w, dp.h, dp.w, n);
}

void adam_all(hipStream_t s, float* p, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2,
              float eps, float c1, float c2, const AdamSeg* segs, int nseg) {
  hipLaunchKernelGGL(k_adam_all, dim3(grid_for(n)), dim3(256), 0, s, p, g, m, v, n, lr, b1, b2, eps, c1, c2, segs,
                     nseg);
}

void to_bf16(hipStream_t s, const float* p, uint16_t* w16, uint16_t* wt16, int cin, int cout) {
  const size_t n = size_t(cout) * 9 * cin;
  hipLaunchKernelGGL(k_to_bf16, dim3(grid_for(n)), dim3(256), 0, s, p, w16, wt16, cin, cout, n);
}

}  // namespace gdn
