// A2V bridge output projection with the per-token residual norm fused into
// its epilogue (gfx950, bf16 MFMA).
//
// Reference: the a2v bridge residual is ConditionalCrossAttention's output
// projection, delta_h = self.o(x) = x W^T + b (nn.Linear(dim, dim),
// hymm/models/modules/interactionv2.py:225, :348), stored as
// a2v_bridge_residual (hymm/models/modules/mova.py:127-137), whose per-token
// L2 norms drive the audio terms of the shape choice
// (hymm/models/modules/wan_video_dit.py:742-752: residual.norm(dim=-1)).  The
// reference runs the projection and then reads the [S, C] residual again for
// the norms; here the norm is formed while the projection's output tiles are
// still in registers.
//
// Kernels:
//   linear_rownorm_kernel  y[M,N] = x[M,K] W[N,K]^T + b (bf16 out, fp32
//                          accumulate) and, per row m and 256-column tile t,
//                          partial[m][t] = sum over the tile's columns of
//                          bf16(y)^2 (the squares of the stored values)
//   rownorm_finish_kernel  norms[m] = sqrt(sum_t partial[m][t]), t ascending
//
// MI355X design: persistent workgroups of four waves (one per SIMD), one 256 x
// 256 output tile at a time (fewer tiles than CUs, or a nearly empty last
// round: 128 or 64 rows), each wave 128 x 128 = 8 x 8 blocks of
// v_mfma_f32_16x16x32_bf16 (256 accumulator AGPRs; the tile computes C^T = W
// x^T, so each lane owns one output row and four consecutive columns per
// block).  Stages of 64 columns of K: a ring of five 32 KB slots (all of the
// 160 KB) takes x and W tiles in turn by global_load_lds_dwordx4, three tiles
// ahead of the stage being read.  A stage is two steps of 64 MFMAs; each step
// reads the next one's fragments (two ds_read_b128 per eight MFMAs) and issues
// one copy per eight MFMAs; the one barrier of a stage stands between its
// steps, when all of the stage's fragments are in registers, so the MFMAs go on
// right behind it.  The stages run on over the end of an output tile: its
// epilogue works while the next tile's first 96 KB land, turning the
// accumulators through the one free slot so that y is stored in rows of 256
// bytes.  LDS rows are 128 bytes, unpadded, with the 16-byte chunks of row r
// XOR-swizzled by (r >> 1) & 7, so the row-operand reads (16 consecutive rows,
// one chunk each, per 16 lanes) hit distinct bank groups.  Tiles are ordered so
// that each XCD (own L2) works on about 8 x 4 neighbouring output tiles at a
// time, which share their k-slices of x and W in its L2.  Deterministic (no
// atomics).
//
// Measured at M = 75,600, N = K = 5,120 (3.96 TFLOP): 3.93 -> 2.89 ms, 1,009 ->
// 1,369 TFLOP/s, against 2.80 ms of torch's F.linear (hipBLASLt) without the
// norms.  What the time was: an epilogue of 24 us per tile (16-byte pieces of y
// and a branch per rounded element; K = 64, 5,120 tiles: 475 -> 199 us, now the
// write of y), the copies' latency at each stage's end, and 32 x 32 x 16 MFMAs
// with bursts of fragment reads (as few cycles, but a lower clock: 2.68 against
// 2.39 ms at M = 65,536).
// Stages of 32 columns with four in flight were slower (3.81 ms): rows of 64
// bytes double the L2 requests.  Now bound by the matrix cores at the clock
// that their power leaves (about 1.7 GHz; with x = 0, M = 65,536 takes 2.03
// instead of 2.39 ms) and by the last round of tiles (24 for 23.1).
#include "common.h"
#include "mfma.h"
#include "tile_dma.h"

namespace {

constexpr int kBN = 256, kBK = 64;
constexpr int kSlots = 5;                          // ring of x and W tiles in turn (160 KB)
constexpr int kRowBytes = kBK * 2;                 // 128
constexpr int kTileBytes = kBN * kRowBytes;        // 32 KB: the W tile of a stage (the x tile: at most that)
constexpr int kOprojThreads = 256;                 // 4 waves
constexpr int kCopies = kTileBytes / 1024 / 4;     // 8 KB-instructions per wave and W tile
constexpr int kGroupM = 4;                         // output-tile rows per group of the launch order

struct OprojArgs {
  const uint16_t* x;     // [M, K]
  const uint16_t* w;     // [N, K]
  const uint16_t* bias;  // [N] or null
  int64_t M;
  int N, K;
  int mtiles, ntiles;    // ceil(M / (32 R)), N / 256
  int total;             // output tiles
  uint16_t* y;           // [M, N]
  float* partial;        // [M, ntiles]
};

// byte offset of logical 16-byte chunk c (0..7) of tile row r: chunks XOR-
// swizzled by (r >> 1) & 7, so that the 16 rows one 16-lane group reads
// (one chunk each) fall in 16 distinct 16-byte bank groups (two rows per
// 256-byte bank line: (r & 1, (r >> 1) & 7) differ for 16 consecutive rows)
__device__ __forceinline__ uint32_t swz(int r, int c) { return (uint32_t)(r * kRowBytes + 16 * (c ^ ((r >> 1) & 7))); }

// an accumulator element, moved out of its AGPR here (left to the compiler, all
// 256 are moved at once and the copies' offsets spill)
__device__ __forceinline__ float acc_read(float a) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}

// R: blocks of 16 rows per wave (output tiles of 32 R rows)
template <int R>
__global__ __launch_bounds__(kOprojThreads, 1) void linear_rownorm_kernel(OprojArgs a) {
  static_assert(R == 8 || R == 4 || R == 2, "R copies of x per wave and stage");
  constexpr int kBM = 32 * R;
  __shared__ __align__(1024) uint8_t smem[kSlots * kTileBytes];

  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, l16 = lane & 15;
  const int w = (int)uniform_u32((uint32_t)tid >> 6);
  const int mh = w & 1, nh = w >> 1;

  // Launch order.  Hardware id b runs on XCD b & 7: each XCD takes a
  // contiguous range of logical ids; logical ids walk groups of kGroupM
  // output-tile rows column by column, so the ~32 workgroups an XCD runs at
  // once cover about 4 x 8 tiles and share each k-slice of x (8 ways) and W
  // (4 ways) in that XCD's L2 (4-row groups measured 4% faster than 8-row
  // groups; plain row order was within 1%).
  const int nwg = (int)gridDim.x, per = a.total / 8;
  auto tile_of = [&](int b, int& mt, int& nt) {
    const int lid = b < per * 8 ? (b & 7) * per + (b >> 3) : b;
    const int gsize = kGroupM * a.ntiles;
    const int grp = lid / gsize, first_m = grp * kGroupM;
    const int gm = a.mtiles - first_m < kGroupM ? a.mtiles - first_m : kGroupM;
    const int inner = lid - grp * gsize;
    mt = first_m + inner % gm;
    nt = inner / gm;
  };

  // DMA plan: KB-instruction i of a tile covers its bytes [1024 i, 1024 i + 1024);
  // lane L writes 16 bytes at 16 L: row 8 i + L / 8, stored chunk L % 8, logical
  // chunk (L % 8) ^ ((row >> 1) & 7).  Wave w issues i = w + 4 c.
  uint32_t xoff[R], woff[kCopies];  // byte offsets of this lane's 16 bytes at k = 0
  const uint32_t last = (uint32_t)a.M - 1, ld = (uint32_t)a.K * 2;  // M < 2^25 (x below 4 GiB)
  auto x_tile = [&](int v) {
    int mt, nt;
    tile_of(v, mt, nt);
    const int t = opaque_thread_id(), row = 8 * w + (t & 63) / 8;  // (not kept across the tile)
    const uint32_t chunk = 16u * ((t % 8) ^ ((row >> 1) & 7));  // the same for rows 32 apart
#pragma unroll
    for (int c = 0; c < R; ++c) {
      const uint32_t m = (uint32_t)(mt * kBM + row + 32 * c);
      xoff[c] = (m < last ? m : last) * ld + chunk;  // rows past M re-read the last row (never stored)
    }
  };
  auto w_tile = [&](int v) {
    int mt, nt;
    tile_of(v, mt, nt);
    const int t = opaque_thread_id(), row = 8 * w + (t & 63) / 8;
    const uint32_t chunk = 16u * ((t % 8) ^ ((row >> 1) & 7));
#pragma unroll
    for (int c = 0; c < kCopies; ++c) woff[c] = (uint32_t)(nt * kBN + row + 32 * c) * ld + chunk;
  };
  const int nsteps = a.K / kBK;
  const uint32_t lds0 = lds_addr(smem) + 1024u * (uint32_t)w;
  const uint8_t* const xb = (const uint8_t*)uniform_ptr(a.x);
  const uint8_t* const wb = (const uint8_t*)uniform_ptr(a.w);
  // the tiles to copy next: output tile, k offset, slot.  The copies run on
  // into the workgroup's next output tile (after its last one, into that one
  // again: slots that nothing reads any more, so every stage issues and waits
  // alike)
  const uint32_t kend = (uint32_t)nsteps * kRowBytes;
  uint32_t kx = 0, kw = 0, put = 0;
  int vx = (int)blockIdx.x, vw = vx;
  auto next_slot = [&](uint32_t s) { return s + kTileBytes == kSlots * kTileBytes ? 0u : s + kTileBytes; };
  auto copy_x = [&](int c) { dma_b128(xoff[c], xb + kx, lds0 + put + 4096u * (uint32_t)c); };
  auto copy_w = [&](int c) { dma_b128(woff[c], wb + kw, lds0 + put + 4096u * (uint32_t)c); };
  auto copied_x = [&] {
    kx += kRowBytes;
    put = next_slot(put);
    if (kx == kend) {
      kx = 0;
      if (vx + nwg < a.total) x_tile(vx += nwg);
    }
  };
  auto copied_w = [&] {
    kw += kRowBytes;
    put = next_slot(put);
    if (kw == kend) {
      kw = 0;
      if (vw + nwg < a.total) w_tile(vw += nwg);
    }
  };
  x_tile(vx);
  w_tile(vw);

  f32x4 acc[8][R];

  // operand fragments of k-step s (32 wide): A = W rows 128 nh + 16 i + l16, B =
  // x rows 16 R mh + 16 j + l16, logical chunk 4 s + g: the offset of chunk g
  // XOR 64 s (4 s only touches the top bit of the chunk), rows 16 i an immediate
  const uint32_t offA = swz(nh * 128 + l16, g), offB = swz(mh * 16 * R + l16, g);
  bf16x8 av[2][8], bv[2][R];
  uint32_t get = 0;  // slot of the stage's x tile; its W tile is in the next one
  uint32_t pA = 0, pB = 0;
  auto stage_at = [&] {
    pB = get + offB;
    get = next_slot(get);
    pA = get + offA;
    get = next_slot(get);
  };
  auto load = [&](int s, int i) {
    if (i < R) bv[s][i] = *reinterpret_cast<const bf16x8*>(smem + (pB ^ (64u * s)) + 16 * kRowBytes * i);
    av[s][i] = *reinterpret_cast<const bf16x8*>(smem + (pA ^ (64u * s)) + 16 * kRowBytes * i);
  };
  auto mul = [&](int s, int i) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < R; ++j)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(av[s][i]), "v"(bv[s][j]));
    __builtin_amdgcn_sched_barrier(0);
  };
  // both tiles of the next stage have landed (the x tile after them may still
  // be in flight) and every wave has its fragments of this one
  auto landed = [&] {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(R));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };

#pragma unroll
  for (int c = 0; c < R; ++c) copy_x(c);
  copied_x();
#pragma unroll
  for (int c = 0; c < kCopies; ++c) copy_w(c);
  copied_w();
#pragma unroll
  for (int c = 0; c < R; ++c) copy_x(c);
  copied_x();
  landed();
  stage_at();
#pragma unroll
  for (int i = 0; i < 8; ++i) load(0, i);
#pragma unroll
  for (int c = 0; c < kCopies; ++c) copy_w(c);
  copied_w();
  for (int v = (int)blockIdx.x; v < a.total; v += nwg) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    asm volatile("s_nop 7");  // before inline assembly reads them
    for (int ks = 0; ks < nsteps; ++ks) {
      // 64 MFMAs of step 0 while step 1's fragments are read and an x tile is copied
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        load(1, i);
        mul(0, i);
        if (i < R) copy_x(i);
      }
      copied_x();
      landed();
      stage_at();
      // step 1, with the next stage's first fragments and a W tile
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        load(0, i);
        mul(1, i);
        copy_w(i);
      }
      copied_w();
    }

    // epilogue, while the next output tile's first copies land: acc[i][j]
    // element e holds C^T[n][m] with n = n0 + 16 i + 4 g + e, m = m0 + 16 j +
    // l16.  The wave turns 32 rows of 128 columns at a time through 8 KB of the
    // slot that the next x tile is copied to after the last barrier, chunk c of
    // row r at c ^ (r & 15), and stores rows of 256 bytes.
    int mt, nt;
    tile_of(v, mt, nt);
    const int m0 = mt * kBM + 16 * R * mh, n0 = nt * kBN + 128 * nh, M = (int)a.M;
    const int lane = opaque_thread_id() & 63, g = lane >> 4, l16 = lane & 15;
    uint8_t* const stage = smem + put + 8192u * (uint32_t)w;
    asm volatile("s_nop 15\n\ts_nop 15");  // the last MFMAs' results, read by inline assembly below
    uint2 bias[8];  // of columns 16 i + 4 g .. + 3
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bias[i] = a.bias ? *reinterpret_cast<const uint2*>(a.bias + n0 + 16 * i + 4 * g) : uint2{0u, 0u};
    float ss[R];  // squares of the stored values of this lane's row, per m block
#pragma unroll
    for (int j = 0; j < R; ++j) {
      ss[j] = 0.0f;
      const int row = 16 * (j & 1) + l16;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint2 u = bias[i];
        asm volatile("" : "+v"(u.x), "+v"(u.y));  // (unpacked here, not kept as floats for all j)
        const float bb[4] = {__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
                             __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
        uint2 o;  // (v_cvt_pk_bf16_f32: round to nearest even, as the scalar helper without its branch)
        o.x = pack_bf16(acc_read(acc[i][j][0]) + bb[0], acc_read(acc[i][j][1]) + bb[1]);
        o.y = pack_bf16(acc_read(acc[i][j][2]) + bb[2], acc_read(acc[i][j][3]) + bb[3]);
        const float t[4] = {__uint_as_float(o.x << 16), __uint_as_float(o.x & 0xffff0000u),
                            __uint_as_float(o.y << 16), __uint_as_float(o.y & 0xffff0000u)};
#pragma unroll
        for (int e = 0; e < 4; ++e) ss[j] = __builtin_fmaf(t[e], t[e], ss[j]);
        *reinterpret_cast<uint2*>(stage + 256 * row + 16 * ((2 * i + (g >> 1)) ^ l16) + 8 * (g & 1)) = o;
        if (i & 1) __builtin_amdgcn_sched_barrier(0);
      }
      if (j & 1) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int row = 4 * r + (lane >> 4);
          const uint4 o = *reinterpret_cast<const uint4*>(stage + 256 * row + 16 * ((lane & 15) ^ (row & 15)));
          const int m = m0 + 16 * (j - 1) + row;
          if (m < M) *reinterpret_cast<uint4*>(a.y + (int64_t)m * a.N + n0 + 8 * (lane & 15)) = o;
        }
      }
    }
    // row partial of this wave (its 128 columns): the four lane groups hold
    // different columns of the same row; then the two waves of a row
    float* const part = reinterpret_cast<float*>(stage);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float t = xor32_add(ss[j] + __shfl_xor(ss[j], 16));
      if (g == 0) part[16 * j + l16] = t;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    if (nh == 0) {
#pragma unroll
      for (int h = 0; h < (R + 3) / 4; ++h) {
        const int m = m0 + 64 * h + lane;
        if (m < M && 64 * h + lane < 16 * R)
          a.partial[(int64_t)m * a.ntiles + nt] = part[64 * h + lane] + part[2 * 2048 + 64 * h + lane];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();  // the x tile copied there next stays off what other waves read
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
  dma_wait_all();
}

template <typename TO>
__global__ __launch_bounds__(256) void rownorm_finish_kernel(const float* __restrict__ partial, int64_t M, int nt,
                                                              TO* __restrict__ norms) {
  const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (m >= M) return;
  float s = 0.0f;
  for (int t = 0; t < nt; ++t) s = s + partial[m * nt + t];
  const float r = sqrtf(s);
  if (sizeof(TO) == 2) reinterpret_cast<uint16_t*>(norms)[m] = f2bf(r);
  else reinterpret_cast<float*>(norms)[m] = r;
}

template <int R>
void launch_rows(OprojArgs a, int cus, hipStream_t stream) {
  a.mtiles = (int)((a.M + 32 * R - 1) / (32 * R));
  a.total = a.mtiles * a.ntiles;
  linear_rownorm_kernel<R><<<(unsigned)(a.total < cus ? a.total : cus), kOprojThreads, 0, stream>>>(a);
}

// Rows per output tile: the height whose rounds of tiles cost least.  A round of
// 256, 128 and 64 rows takes 118, 67 and 59 us at K = 5,120 (the lower tiles
// wait for the copies of W, not for the matrix cores), in much the same ratios
// at other K.  Measured, 256 against 128 against 64 rows (N = K): 200 x 5,120 98
// / 64 / 60 us; 700 x 1,536 39 / 24 / 18; 1,000 x 5,120 103 / 68 / 119; 4,000 x
// 5,120 213 / 207 / 301; 6,528 x 5,120 323 / 291 / 469; 8,000 x 1,536 45 / 54 /
// 60; 12,000 x 5,120 483 / 544 / 852.  Within 3% of the best height at 200 to
// 20,000 rows and N x K of 5,120 x 512, 5,120 x 1,024, 1,536^2, 2,048^2, 3,072^2,
// 5,120 x 2,560, 5,120^2 and 1,280 x 8,192.
void launch_rownorm(const OprojArgs& a, hipStream_t stream) {
  const int cus = resident_workgroups<linear_rownorm_kernel<8>>(kOprojThreads);
  auto cost = [&](int rows, int64_t us) {
    const int64_t tiles = (a.M + rows - 1) / rows * a.ntiles;
    return (tiles + cus - 1) / cus * us;
  };
  const int64_t c8 = cost(256, 118), c4 = cost(128, 67), c2 = cost(64, 59);
  if (c8 <= c4 && c8 <= c2) launch_rows<8>(a, cus, stream);
  else if (c4 <= c2) launch_rows<4>(a, cus, stream);
  else launch_rows<2>(a, cus, stream);
}

}  // namespace

extern "C" {

int prism_linear_rownorm(const void* x, const void* w, const void* bias, int64_t M, int N, int K, void* y, void* norms,
                         int norms_dtype, float* partial, hipStream_t stream) {
  PRISM_REQUIRE(x && w && y && norms && partial, "prism_linear_rownorm: null pointer");
  PRISM_REQUIRE(M >= 1, "prism_linear_rownorm: M must be >= 1");
  PRISM_REQUIRE(N >= kBN && N % kBN == 0, "prism_linear_rownorm: N=%d must be a positive multiple of %d", N, kBN);
  PRISM_REQUIRE(K >= 64 && K % 64 == 0, "prism_linear_rownorm: K=%d must be a positive multiple of 64", K);
  PRISM_REQUIRE(norms_dtype == PRISM_F32 || norms_dtype == PRISM_BF16, "prism_linear_rownorm: bad norms dtype");
  // per-lane source offsets are 32-bit byte offsets from the tensors' bases
  PRISM_REQUIRE(M * (int64_t)K * 2 < (1ll << 32) && (int64_t)N * K * 2 < (1ll << 32),
                "prism_linear_rownorm: x and W must each be smaller than 4 GiB");
  const int ntiles = N / kBN;
  PRISM_REQUIRE((M + 63) / 64 * ntiles < (1ll << 31), "prism_linear_rownorm: grid too large");
  OprojArgs a;
  a.x = (const uint16_t*)x; a.w = (const uint16_t*)w; a.bias = (const uint16_t*)bias;
  a.M = M; a.N = N; a.K = K; a.ntiles = ntiles; a.y = (uint16_t*)y; a.partial = partial;
  launch_rownorm(a, stream);
  const unsigned fb = (unsigned)((M + 255) / 256);
  if (norms_dtype == PRISM_BF16) rownorm_finish_kernel<uint16_t><<<fb, 256, 0, stream>>>(partial, M, ntiles, (uint16_t*)norms);
  else rownorm_finish_kernel<float><<<fb, 256, 0, stream>>>(partial, M, ntiles, (float*)norms);
  PRISM_LAUNCH_CHECK("prism_linear_rownorm");
  return PRISM_OK;
}

}  // extern "C"
