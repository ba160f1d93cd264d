// The dense pieces of a transformer block around the attention call, for serving a stack of blocks without leaving the
// library between two attention calls: linear layers with their bias, activation or residual in the same launch, and
// layer norm.  16-bit operands, fp32 sums; values are rounded where a layer hands its result to the next.
#include <algorithm>

#include "../../include/moda_hip.h"
#include "block.h"
#include "geometry.h"
#include "tile.h"
#include "tile16.h"
#include "tuning.h"

namespace moda {

struct LinearPart {
  const uint16_t *w, *bias;
  uint16_t* y;
  int64_t ldy;
  int n, tile_end;  // output features; feature tiles of this part and of those before it
};
struct LinearArgs {
  const uint16_t *x, *residual;
  int64_t ldx, ld_res;
  int rows, K, m_tiles, n_tiles, n_parts;
  LinearPart part[3];
};

enum Epilogue { kBias, kGelu, kResidual };

// y = x W^T: both operands have the summation index innermost, so a k step is a 64-element-wide tile of each, staged
// like the attention kernels' 64-wide tiles.  Four waves share a BM (rows) x BN (features) output tile, two by two.
// The features sit on the matrix instruction's A side: a lane then holds four consecutive features of one row.
//
// Sized for a vision model's linears (12 608 rows, K 256 .. 1024), where a launch is 8 to 20 us and the k loop 4 to 16
// steps: what counts is enough workgroups in flight to cover each one's start and end, not a large tile.
template <typename T, int BM, int BN, int NST, Epilogue EPI>
__global__ __launch_bounds__(256, 2) void linear_kernel(const LinearArgs a) {
  constexpr int DIST = NST - 1, MB = BN / 32, NB = BM / 32, STAGE = (BM + BN) * 64;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  lds_ptr smem = (lds_ptr)smem_raw;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wf = wave & 1;
  const int mt = linear_row_tile(blockIdx.x, a.n_tiles);
  int nt = linear_feature_tile(blockIdx.x, a.n_tiles);
  if (mt >= a.m_tiles) return;
  int pi = 0;
  if (a.n_parts > 1 && nt >= a.part[0].tile_end) pi = (a.n_parts > 2 && nt >= a.part[1].tile_end) ? 2 : 1;
  const LinearPart p = a.part[pi];
  if (pi > 0) nt -= a.part[pi - 1].tile_end;
  const int r0 = mt * BM, f0 = nt * BN, nk = a.K / 64;

  typedef AsyncTileLoader<64, BM, 256> LoadX;
  typedef AsyncTileLoader<64, BN, 256> LoadW;
  LoadX lx;
  LoadW lw;
  lx.init(tid);
  lw.init(tid);
  int ld_st = 0;
  auto issue = [&](int it) {
    lds_ptr xs = smem + ld_st * STAGE;
    lx.load(xs, a.x + it * 64, a.ldx, r0, a.rows, 64);
    lw.load(xs + BM * 64, p.w + it * 64, a.K, f0, p.n, 64);
    ld_st = (ld_st + 1 == NST) ? 0 : ld_st + 1;
  };
  auto wait_tile = [&](int next) {
    if (DIST == 2 && next + 1 < nk)
      LoadX::template wait_but<LoadX::N + LoadW::N>();
    else
      LoadX::wait_all();
  };
  Operand16<64> oa;
  oa.init(lane);
  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < DIST; j++)
    if (j < nk) issue(j);
  wait_tile(0);
  __syncthreads();
  int st = 0;
  for (int it = 0; it < nk; it++) {
    if (it + DIST < nk) issue(it + DIST);
    lds_cptr xs = smem + st * STAGE + wm * (BM / 2) * 64, ws = smem + st * STAGE + (BM + wf * (BN / 2)) * 64;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      i32x4 wo[MB], xo[NB];
#pragma unroll
      for (int mb = 0; mb < MB; mb++) wo[mb] = oa.row_operand(ws, 16 * mb, ks);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) xo[nb] = oa.row_operand(xs, 16 * nb, ks);
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[mb][nb] = mfma16<T>(wo[mb], xo[nb], acc[mb][nb]);
    }
    st = (st + 1 == NST) ? 0 : st + 1;
    wait_tile(it + 1);
    __syncthreads();
  }

  auto four = [](const uint16_t* src, float (&f)[4]) {
    const i32x2 w = *reinterpret_cast<const i32x2*>(src);
    unpack2<T>(w[0], f[0], f[1]);
    unpack2<T>(w[1], f[2], f[3]);
  };
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int f = f0 + wf * (BN / 2) + 16 * mb + slot_base(q4);
    if (f >= p.n) continue;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias) four(p.bias + f, bias);
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const int r = r0 + wm * (BM / 2) + 16 * nb + slot_base(n >> 2) + (n & 3);
      if (r >= a.rows) continue;
      float x[4], res[4] = {0.f, 0.f, 0.f, 0.f};
      if (EPI == kResidual) four(a.residual + (int64_t)r * a.ld_res + f, res);
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = acc[mb][nb][i] + bias[i];
      if (EPI != kBias) {  // the linear layer's own result is a 16-bit value, as it is when the layers run one by one
        unpack2<T>(pack2<T>(x[0], x[1]), x[0], x[1]);
        unpack2<T>(pack2<T>(x[2], x[3]), x[2], x[3]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (EPI == kGelu) x[i] = gelu(x[i]);
        if (EPI == kResidual) x[i] += res[i];
      }
      i32x2 w;
      w[0] = pack2<T>(x[0], x[1]);
      w[1] = pack2<T>(x[2], x[3]);
      *reinterpret_cast<i32x2*>(p.y + (int64_t)r * p.ldy + f) = w;
    }
  }
}

// Layer norm: LPR lanes share a row, CH 16-byte pieces each; mean, then the sum of squared deviations, from registers.
template <typename T, int LPR, int CH>
__global__ __launch_bounds__(256) void layer_norm_kernel(const uint16_t* x, const uint16_t* weight, const uint16_t* bias, float eps,
                                                         uint16_t* y, int rows, int dim) {
  layer_norm_rows<T, LPR, CH>(blockIdx.x, x, weight, bias, eps, y, rows, dim);
}

namespace {

template <typename T, int BM, int BN, int NST, Epilogue EPI>
hipError_t launch_linear_t(LinearArgs a, hipStream_t stream) {
  constexpr size_t smem = (size_t)NST * (BM + BN) * 64 * sizeof(uint16_t);
  static LdsAttrState attr;
  const hipError_t e = allow_dynamic_lds(attr, reinterpret_cast<const void*>(&linear_kernel<T, BM, BN, NST, EPI>), smem);
  if (e != hipSuccess) return e;
  a.m_tiles = (a.rows + BM - 1) / BM;
  a.n_tiles = 0;
  for (int i = 0; i < a.n_parts; i++) a.part[i].tile_end = a.n_tiles += (a.part[i].n + BN - 1) / BN;
  const int64_t nblk = linear_blocks(a.m_tiles, a.n_tiles);
  if (nblk >= (1ll << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((linear_kernel<T, BM, BN, NST, EPI>), dim3((unsigned)nblk), dim3(256), smem, stream, a);
  return hipGetLastError();
}

template <typename T, Epilogue EPI>
hipError_t launch_linear_e(const LinearArgs& a, int cus, hipStream_t stream) {
  int features[3];
  for (int i = 0; i < a.n_parts; i++) features[i] = a.part[i].n;
  switch (pick_linear_tile(a.rows, a.K, features, a.n_parts, cus)) {
    case LinearTile::k128x128: return launch_linear_t<T, 128, 128, 2, EPI>(a, stream);
    case LinearTile::k128x64: return launch_linear_t<T, 128, 64, 2, EPI>(a, stream);
    case LinearTile::k128x64ThreeStages: return launch_linear_t<T, 128, 64, 3, EPI>(a, stream);
    default: return launch_linear_t<T, 64, 64, 2, EPI>(a, stream);
  }
}

template <typename T>
hipError_t launch_layer_norm_t(int rows, int dim, const uint16_t* x, const uint16_t* w, const uint16_t* b, float eps, uint16_t* y,
                               hipStream_t stream) {
  auto go = [&](auto lpr, auto ch) {
    constexpr int LPR = decltype(lpr)::value, CH = decltype(ch)::value;
    hipLaunchKernelGGL((layer_norm_kernel<T, LPR, CH>), dim3((unsigned)((rows + 256 / LPR - 1) / (256 / LPR))), dim3(256), 0, stream, x, w, b,
                       eps, y, rows, dim);
    return hipGetLastError();
  };
  using std::integral_constant;
  const integral_constant<int, 1> one{};
  const integral_constant<int, 64> wave{};
  if (dim <= 128) return go(integral_constant<int, 16>{}, one);
  if (dim <= 256) return go(integral_constant<int, 32>{}, one);
  if (dim <= 512) return go(wave, one);
  if (dim <= 1024) return go(wave, integral_constant<int, 2>{});
  if (dim <= 2048) return go(wave, integral_constant<int, 4>{});
  return go(wave, integral_constant<int, 8>{});
}

}  // namespace

hipError_t launch_linear(int dtype, int64_t rows, int64_t K, const void* x, int64_t ldx, const moda_hip_linear_part* parts, int n_parts,
                         const void* residual, int64_t ld_res, bool gelu, int compute_units, hipStream_t stream) {
  LinearArgs a = {};
  a.x = (const uint16_t*)x;
  a.residual = (const uint16_t*)residual;
  a.ldx = ldx;
  a.ld_res = ld_res;
  a.rows = (int)rows;
  a.K = (int)K;
  a.n_parts = n_parts;
  for (int i = 0; i < n_parts; i++)
    a.part[i] = LinearPart{(const uint16_t*)parts[i].w, (const uint16_t*)parts[i].bias, (uint16_t*)parts[i].y, parts[i].ldy, (int)parts[i].n, 0};
  auto run = [&](auto type) {
    typedef decltype(type) T;
    if (residual) return gelu ? hipErrorInvalidValue : launch_linear_e<T, kResidual>(a, compute_units, stream);
    return gelu ? launch_linear_e<T, kGelu>(a, compute_units, stream) : launch_linear_e<T, kBias>(a, compute_units, stream);
  };
  return dtype == 0 ? run(BF16{}) : run(FP16{});
}

hipError_t launch_layer_norm(int dtype, int64_t rows, int64_t dim, const void* x, const void* weight, const void* bias, float eps, void* y,
                             hipStream_t stream) {
  const uint16_t *xp = (const uint16_t*)x, *w = (const uint16_t*)weight, *b = (const uint16_t*)bias;
  return dtype == 0 ? launch_layer_norm_t<BF16>((int)rows, (int)dim, xp, w, b, eps, (uint16_t*)y, stream)
                    : launch_layer_norm_t<FP16>((int)rows, (int)dim, xp, w, b, eps, (uint16_t*)y, stream);
}

}  // namespace moda
