// k_net.hip -- kernels of the learned pressure preconditioner (the U-Net in
// net.hpp): MFMA implicit-GEMM 3x3x3 convolutions (forward and input
// gradient), MFMA weight gradients, and the VALU glue (first layer, head,
// pooling, relu masks, loss, Adam).
//
// MFMA v_mfma_f32_16x16x32_bf16 lane layout (64 lanes, j = lane / 16,
// c = lane % 16):  A[16 x 32]: lane holds A[c][8j .. 8j+7];
// B[32 x 16]: lane holds B[8j .. 8j+7][c];  D[16 x 16]: lane holds
// D[4j .. 4j+3][c].  (Checked on the device by the probe kernel below.)
#include "common.hpp"
#include "net.hpp"

namespace pyro {

namespace {
__device__ __forceinline__ f32x4 mfma16x16x32(const bf16x8 &a, const bf16x8 &b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float bf(bf16 v) { return (float)v; }
__device__ __forceinline__ bf16 tobf(float f) { return (bf16)f; }
inline unsigned nblk(uint64_t n, int nt = 256) { return (unsigned)((n + nt - 1) / nt); }
}  // namespace

// ------------------------------------------------------------ probe
__global__ __launch_bounds__(64) void k_mfma_probe(const bf16 *a, const bf16 *b, float *d) {
  const int l = threadIdx.x;
  const bf16x8 av = *reinterpret_cast<const bf16x8 *>(a + 8 * l);
  const bf16x8 bv = *reinterpret_cast<const bf16x8 *>(b + 8 * l);
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  acc = mfma16x16x32(av, bv, acc);
  for (int i = 0; i < 4; i++) d[4 * l + i] = acc[i];
}
void launch_mfma_probe(const bf16 *a, const bf16 *b, float *d, hipStream_t s) { k_mfma_probe<<<1, 64, 0, s>>>(a, b, d); }

// ------------------------------------------------------------ packing
// The upsampled input of a layer with one 16-row output block (cout = 16) is
// staged in 16-channel chunks (smaller LDS footprint, higher occupancy);
// otherwise in 32-channel chunks.
int conv_a_chunk(int cout) { return cout == 16 ? 16 : 32; }
int conv_groups(int ca, int cb, int cout) {
  const int cca = conv_a_chunk(cout);
  return (ca / cca) * (cca == 32 ? 27 : 14) + (cb == 16 ? 14 : (cb / 32) * 27);
}

// element e of the packed weights of one conv (see net.hpp)
__device__ __forceinline__ bf16 packed_weight(const float *__restrict__ W, int cout, int cin, int ca_e, int cb_e,
                                              int cout_e, bool transposed, uint32_t e) {
  const int kk = (int)(e % 32u);
  const int co_e = (int)((e / 32u) % (uint32_t)cout_e);
  int grp = (int)(e / (32u * (uint32_t)cout_e));
  const int cca = cout_e == 16 ? 16 : 32, ga = cca == 32 ? 27 : 14;
  const int nA = ca_e / cca;
  int tap, ci_e;
  if (grp < nA * ga) {
    if (cca == 32) {
      tap = grp % 27;
      ci_e = 32 * (grp / 27) + kk;
    } else {
      tap = 2 * (grp % 14) + kk / 16;
      ci_e = 16 * (grp / 14) + (kk % 16);
    }
  } else {
    grp -= nA * ga;
    if (cb_e == 16) {
      tap = 2 * grp + kk / 16;
      ci_e = ca_e + (kk % 16);
    } else {
      tap = grp % 27;
      ci_e = ca_e + 32 * (grp / 27) + kk;
    }
  }
  float v = 0.0f;
  if (tap < 27) {
    if (!transposed)
      v = W[((size_t)co_e * cin + ci_e) * 27 + tap];
    else  // adjoint: input channel = original output channel, taps mirrored
      v = W[((size_t)ci_e * cin + co_e) * 27 + (26 - tap)];
  }
  return tobf(v);
}
// All packed copies of one parameter vector in one launch: a training step
// repacks every layer in both directions, and fourteen launches of a few
// thousand elements took 4.5 us each.
struct PackEntry {
  const __attribute__((address_space(1))) float *W;
  __attribute__((address_space(1))) bf16 *wp;
  int cout, cin, ca_e, cb_e, cout_e, transposed;
  uint32_t total, block0;  // elements, first block
};
struct PackArgs {
  int n;
  PackEntry e[PACK_MAX];
};
__global__ __launch_bounds__(256) void k_pack_conv(PackArgs) {
  // indexed by block where the arguments lie (a copy would be indexed in scratch memory)
  const PackArgs &a = *(const PackArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  int k = 0;
  while (k + 1 < a.n && blockIdx.x >= a.e[k + 1].block0) k++;
  const PackEntry &p = a.e[k];
  const uint32_t e = (blockIdx.x - p.block0) * 256u + threadIdx.x;
  if (e >= p.total) return;
  p.wp[e] = packed_weight((const float *)p.W, p.cout, p.cin, p.ca_e, p.cb_e, p.cout_e, p.transposed != 0, e);
}
void launch_pack_jobs(const PackJob *jobs, int n, hipStream_t s) {
  PackArgs a;
  uint32_t blocks = 0;
  a.n = n;
  for (int k = 0; k < a.n; k++) {
    const ConvSpec &c = jobs[k].c;
    PackEntry &p = a.e[k];
    p.W = (const __attribute__((address_space(1))) float *)jobs[k].W;
    p.wp = (__attribute__((address_space(1))) bf16 *)jobs[k].wp;
    p.cout = c.cout;
    p.cin = c.cin();
    p.ca_e = jobs[k].transposed ? 0 : c.ca;
    p.cb_e = jobs[k].transposed ? c.cout : c.cb;
    p.cout_e = jobs[k].transposed ? c.cin() : c.cout;
    p.transposed = jobs[k].transposed ? 1 : 0;
    p.total = (uint32_t)conv_groups(p.ca_e, p.cb_e, p.cout_e) * (uint32_t)p.cout_e * 32u;
    p.block0 = blocks;
    blocks += nblk(p.total);
  }
  k_pack_conv<<<blocks, 256, 0, s>>>(a);
}
void launch_pack_conv(const float *W, const ConvSpec &c, bool transposed, bf16 *wp, hipStream_t s) {
  const PackJob j[1] = {{W, wp, c, transposed}};
  launch_pack_convs(j, s);
}
__global__ __launch_bounds__(256) void k_pack_bf16(const float *__restrict__ w, uint32_t n, bf16 *__restrict__ o) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) o[i] = tobf(w[i]);
}
void launch_pack_bf16(const float *w, uint32_t n, bf16 *out, hipStream_t s) {
  k_pack_bf16<<<nblk(n), 256, 0, s>>>(w, n, out);
}

// ------------------------------------------------------------ conv (MFMA)
// Output tile 16 (x) x 4 (y) x 4 (z) voxels per 256-thread block: wave w
// takes row y0 + w, its four 16-voxel column blocks are z0 .. z0+3, lane c
// is x0 + c.  The input footprint (18 x 6 x 6 voxels) of one channel chunk
// (32 channels, or 16 for a 16-channel source) is staged in LDS, then every
// K32 group issues (cout/16) x 4 MFMAs with A = packed weights (global, L1
// resident) and B = 8 channels of one footprint voxel per lane.
constexpr int CV_TX = 16, CV_TY = 4, CV_TZ = 4;
constexpr int CV_FX = CV_TX + 2, CV_FY = CV_TY + 2, CV_FZ = CV_TZ + 2;
constexpr int CV_FN = CV_FX * CV_FY * CV_FZ;

struct ConvArgs {
  int nx, ny, nz;
  int anx, any;  // half-resolution grid of `a`
  const bf16 *a, *b, *wp;
  const float *bias;
  const bf16 *act;  // without RELU, if not null: the result is 0 where act is not positive
  bf16 *out;
  // out: the first `split` channels of all voxels, then the others.  A concat's
  // gradient has two readers, and each took every line of the joint rows (the
  // skip's 16.8 us a launch, now 12.6; the upsampled half's 13.9, now 10.9).
  int split;
};
// act at a voxel's four channels from co on, positive if there is no act (a
// pass of its own over the gradient and act took 25 us a training step at
// 80x160x80, the reads here 4).  A
// voxel outside the grid reads one inside: no branch, all loads in flight.
template <int COUT>
__device__ __forceinline__ bf16x4 act_at(const ConvArgs &p, int x, int y, int z, int co) {
  bf16x4 m = {tobf(1.0f), tobf(1.0f), tobf(1.0f), tobf(1.0f)};
  if (p.act) {
    x = x < p.nx ? x : p.nx - 1;
    y = y < p.ny ? y : p.ny - 1;
    z = z < p.nz ? z : p.nz - 1;
    m = *reinterpret_cast<const bf16x4 *>(
        p.act + ((size_t)x + (size_t)p.nx * ((size_t)y + (size_t)p.ny * (size_t)z)) * COUT + co);
  }
  return m;
}

// footprint offset (in voxels) of tap t relative to footprint voxel (col, w, nb)
__device__ __forceinline__ constexpr int tap_off(int t) {
  return (t / 9) * (CV_FX * CV_FY) + ((t / 3) % 3) * CV_FX + (t % 3);
}

// Stage one channel chunk (CC channels from `a` through nearest upsampling
// when FROMA, else from `b`) of the 18 x 6 x 6 footprint into LDS.  Every
// piece is loaded, from the nearest voxel inside the grid, and zeroed
// afterwards where it lies outside: without branches a thread's loads are in
// flight together instead of one after the other (forward pass at 24x40x24
// 126 -> 110 us, at 160x320x160 1256 -> 1208).
template <int CC, int CSRC, bool FROMA>
__device__ __forceinline__ void conv_stage(const ConvArgs &p, int c0, int x0, int y0, int z0, bf16 *lds) {
  constexpr int PIECES = CC / 8, STRIDE = CC + 8, N = CV_FN * PIECES, NPT = (N + 255) / 256;
  const bf16 *src = (FROMA ? p.a : p.b) + c0;
  uint4 val[NPT];
#pragma unroll
  for (int k = 0; k < NPT; k++) {
    const int s = min((int)threadIdx.x + 256 * k, N - 1);
    const int vox = s / PIECES, pc = s % PIECES;
    const int fx = vox % CV_FX, r2 = vox / CV_FX, fy = r2 % CV_FY, fz = r2 / CV_FY;
    const int gx = min(max(x0 + fx - 1, 0), p.nx - 1), gy = min(max(y0 + fy - 1, 0), p.ny - 1);
    const int gz = min(max(z0 + fz - 1, 0), p.nz - 1);
    size_t v;
    if (FROMA)
      v = (size_t)(gx >> 1) + (size_t)p.anx * ((size_t)(gy >> 1) + (size_t)p.any * (size_t)(gz >> 1));
    else
      v = (size_t)gx + (size_t)p.nx * ((size_t)gy + (size_t)p.ny * (size_t)gz);
    val[k] = *reinterpret_cast<const uint4 *>(src + v * CSRC + 8 * pc);
  }
#pragma unroll
  for (int k = 0; k < NPT; k++) {
    const int s = (int)threadIdx.x + 256 * k;
    const int vox = s / PIECES, pc = s % PIECES;
    const int fx = vox % CV_FX, r2 = vox / CV_FX, fy = r2 % CV_FY, fz = r2 / CV_FY;
    const int gx = x0 + fx - 1, gy = y0 + fy - 1, gz = z0 + fz - 1;
    const bool in = gx >= 0 && gx < p.nx && gy >= 0 && gy < p.ny && gz >= 0 && gz < p.nz;
    if (s < N) *reinterpret_cast<uint4 *>(lds + vox * STRIDE + 8 * pc) = in ? val[k] : make_uint4(0u, 0u, 0u, 0u);
  }
}

// MFMAs of one staged chunk: NG K32 groups (27 taps of 32 channels, or 14
// tap pairs of 16 channels).
template <int CC, int MB, int COUT>
__device__ __forceinline__ void conv_chunk(const bf16 *__restrict__ wp, const bf16 *lds, f32x4 (&acc)[MB][4], int w,
                                           int j, int col) {
  constexpr int NG = CC == 32 ? 27 : 14, STRIDE = CC + 8;
  // output voxel (col, w, nb) sits at footprint (col+1, w+1, nb+1); tap t reads
  // footprint (col+kx, w+ky, nb+kz) = base + nb*FX*FY + tap_off(t)
  const int base = w * CV_FX + col;
  auto group = [&](int g, const bf16x8 (&A)[MB]) {
    int off, ch;
    if (CC == 32) {
      off = tap_off(g);
      ch = 8 * j;
    } else {
      int t = 2 * g + (j >> 1);
      t = t > 26 ? 26 : t;  // the 28th tap has zero weights
      off = tap_off(t);
      ch = 8 * (j & 1);
    }
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      const bf16x8 B = *reinterpret_cast<const bf16x8 *>(lds + (base + nb * (CV_FX * CV_FY) + off) * STRIDE + ch);
#pragma unroll
      for (int m = 0; m < MB; m++) acc[m][nb] = mfma16x16x32(A[m], B, acc[m][nb]);
    }
  };
  if constexpr (MB == 1) {
    // batches of BS groups, the next batch's weight fragments loaded while
    // the current batch computes.  Short batches: with nine and seven the
    // forward pass at 24x40x24 took 87 us, now 78 (64x64x64 109, 102.5).
    constexpr int BS = CC == 32 ? 3 : 2, NBATCH = NG / BS;
    static_assert(NBATCH * BS == NG, "group batches");
    bf16x8 Acur[BS][1], Anext[BS][1];
#pragma unroll
    for (int g = 0; g < BS; g++)
      Acur[g][0] = *reinterpret_cast<const bf16x8 *>(wp + ((size_t)g * COUT + col) * 32 + 8 * j);
#pragma unroll 1
    for (int bt = 0; bt < NBATCH; bt++) {
      if (bt + 1 < NBATCH) {
#pragma unroll
        for (int g = 0; g < BS; g++)
          Anext[g][0] =
              *reinterpret_cast<const bf16x8 *>(wp + ((size_t)((bt + 1) * BS + g) * COUT + col) * 32 + 8 * j);
      }
#pragma unroll
      for (int g = 0; g < BS; g++) group(bt * BS + g, Acur[g]);
      if (bt + 1 < NBATCH) {
#pragma unroll
        for (int g = 0; g < BS; g++) Acur[g][0] = Anext[g][0];
      }
    }
  } else {
#pragma unroll 3
    for (int g = 0; g < NG; g++) {
      bf16x8 A[MB];
#pragma unroll
      for (int m = 0; m < MB; m++)
        A[m] = *reinterpret_cast<const bf16x8 *>(wp + ((size_t)g * COUT + m * 16 + col) * 32 + 8 * j);
      group(g, A);
    }
  }
}

// MS: blocks (blockIdx.y) that share a tile's output channels.
template <int CA, int CB, int COUT, bool RELU, int MS>
__global__ __launch_bounds__(256, 3) void k_conv3(ConvArgs p) {
  constexpr int MB = COUT / 16 / MS;
  constexpr int CCA = COUT == 16 ? 16 : 32;  // conv_a_chunk
  constexpr int NCA = CA / CCA;
  constexpr int NCB = CB == 16 ? 1 : CB / 32;
  constexpr int CCB = CB == 16 ? 16 : 32;
  constexpr int CCMAX = ((NCA > 0 && CCA == 32) || CCB == 32) ? 32 : 16;
  __shared__ __align__(16) bf16 lds[CV_FN * (CCMAX + 8)];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = lane >> 4, col = lane & 15;
  const int ntx = (p.nx + CV_TX - 1) / CV_TX, nty = (p.ny + CV_TY - 1) / CV_TY;
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0 = tx * CV_TX, y0 = ty * CV_TY, z0 = tz * CV_TZ;
  f32x4 acc[MB][4];
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int nb = 0; nb < 4; nb++) acc[m][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int c0 = MS > 1 ? (int)blockIdx.y * MB * 16 : 0;  // the block's first output channel
  const bf16 *wp = p.wp + c0 * 32;
#pragma unroll 1
  for (int q = 0; q < NCA; q++) {
    __syncthreads();
    conv_stage<CCA, CA, true>(p, CCA * q, x0, y0, z0, lds);
    __syncthreads();
    conv_chunk<CCA, MB, COUT>(wp, lds, acc, w, j, col);
    wp += (size_t)(CCA == 32 ? 27 : 14) * COUT * 32;
  }
#pragma unroll 1
  for (int q = 0; q < NCB; q++) {
    __syncthreads();
    conv_stage<CCB, CB, false>(p, 32 * q, x0, y0, z0, lds);
    __syncthreads();
    conv_chunk<CCB, MB, COUT>(wp, lds, acc, w, j, col);
    wp += (size_t)(CCB == 32 ? 27 : 14) * COUT * 32;
  }
  const int gx = x0 + col, gy = y0 + w;
  bf16x4 act[4][MB];
  if (!RELU) {
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
      for (int m = 0; m < MB; m++) act[nb][m] = act_at<COUT>(p, gx, gy, z0 + nb, c0 + m * 16 + 4 * j);
  }
  if (gx >= p.nx || gy >= p.ny) return;
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
    const int gz = z0 + nb;
    if (gz >= p.nz) continue;
    const size_t v = (size_t)gx + (size_t)p.nx * ((size_t)gy + (size_t)p.ny * (size_t)gz);
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const int cm = c0 + m * 16, co = cm + 4 * j;
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float t = acc[m][nb][i] + (p.bias ? p.bias[co + i] : 0.0f);
        if (RELU ? !(t > 0.0f) : !(bf(act[nb][m][i]) > 0.0f)) t = 0.0f;
        o[i] = tobf(t);
      }
      bf16 *to = cm < p.split ? p.out + v * p.split + co
                              : p.out + (size_t)p.nx * p.ny * p.nz * p.split + v * (COUT - p.split) + (co - p.split);
      *reinterpret_cast<bf16x4 *>(to) = o;
    }
  }
}

// 16 output channels from 16-channel chunks (CA/16 of the upsampled `a`, then
// `b`).  With one 16-row output block an MFMA of k_conv3 uses its B fragment
// once, and the LDS (128 B a clock, 8 clocks a fragment) feeds four matrix
// cores at half their rate.  Here a wave computes 16 x 4 x 4 voxels and keeps
// a plane's fragments in registers: a group's two taps are an x pair of one
// row (P: kx 0, 1; R: kx 1, 2), kx 2 with the next row's kx 0 (Q), the step
// to the next plane (X) or the 27th tap (L), so on one plane the rows' P, Q
// and R serve all nine (ky, kz) offsets: 26 reads for 56 products instead of
// 56.  The planes ascend and each voxel's groups stay in order, so every sum
// is k_conv3's.  Block: 16 x 8 x 8 voxels, footprint 18 x 10 x 10.
// Every piece of the footprint is loaded without a branch, so that a thread's
// fifteen are in flight together; with a branch around each the compiler
// waits for one before the next (160x320x160, forward pass: 1526 us, now 1256).
// Launches at 160x320x160 with k_conv3 and with this: 48 -> 16 channels 736 us
// and 363, 16 -> 16 332 and 188; at 80x160x80 95 and 46, 39 and 26.
constexpr int CS_Y = 8, CS_Z = 8, CS_FY = CS_Y + 2, CS_FZ = CS_Z + 2, CS_FN = CV_FX * CS_FY * CS_FZ;
template <int CA, bool RELU>
__global__ __launch_bounds__(256, 2) void k_conv3_16(ConvArgs p) {
  constexpr int NCH = CA / 16 + 1;
  constexpr int ROW = CV_FX * 16, PLANE = CS_FY * ROW;  // elements
  __shared__ __align__(16) bf16 lds[CS_FN * 16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = lane >> 4, col = lane & 15, up = j >> 1;
  const int ntx = (p.nx + CV_TX - 1) / CV_TX, nty = (p.ny + CS_Y - 1) / CS_Y;
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0 = tx * CV_TX, y0 = ty * CS_Y, z0 = tz * CS_Z;
  f32x4 acc[4][4];  // [z][y]
#pragma unroll
  for (int z = 0; z < 4; z++)
#pragma unroll
    for (int y = 0; y < 4; y++) acc[z][y] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int wy = 4 * (w & 1), wz = 4 * (w >> 1);
  // a lane's eight channels of footprint voxel fx of a row: the two halves of
  // a voxel change places where bit 3 of fx is set, so that sixteen voxels
  // (32 bytes apart) touch every bank once
  auto at = [&](int fx) __attribute__((always_inline)) {
    return lds + wz * PLANE + wy * ROW + fx * 16 + ((j ^ (fx >> 3)) & 1) * 8;
  };
  const bf16 *bP = at(col + up), *bR = at(col + 1 + up), *bL = at(col + 2) + 2 * ROW;
  const bf16 *bQ = at(up ? col : col + 2) + (up ? ROW : 0), *bX = at(up ? col : col + 2) + (up ? PLANE : 2 * ROW);
  // staging: a thread loads one 16-byte half of voxel sx of the rows sr + 7 k
  constexpr int PIECES = 2 * CV_FX, SROWS = 256 / PIECES, NROWS = CS_FY * CS_FZ;
  constexpr int NPT = (NROWS + SROWS - 1) / SROWS;
  const int sp = threadIdx.x % PIECES, sr = threadIdx.x / PIECES, sx = sp >> 1;
  const int sgx = x0 + sx - 1;
  const int cgx = min(max(sgx, 0), p.nx - 1);
  bf16 *sdst = lds + sx * 16 + ((sp ^ (sx >> 3)) & 1) * 8;
#pragma unroll 1
  for (int q = 0; q < NCH; q++) {
    const bool from_a = q < NCH - 1;
    const int sh = from_a ? 1 : 0;
    const size_t snx = (size_t)(from_a ? p.anx : p.nx), sny = (size_t)(from_a ? p.any : p.ny), sc = from_a ? CA : 16;
    const bf16 *src = (from_a ? p.a + 16 * q : p.b) + 8 * (sp & 1);
    const bf16 *wp = p.wp + (size_t)q * 14 * 16 * 32 + col * 32 + 8 * j;
    __syncthreads();
    bf16x8 A[14];
#pragma unroll
    for (int g = 0; g < 14; g++) A[g] = *reinterpret_cast<const bf16x8 *>(wp + (size_t)g * 16 * 32);
    {
      // every piece is loaded, from the nearest voxel inside the grid, and
      // zeroed afterwards where it lies outside: no branches, so that all of
      // a thread's loads are in flight together
      uint4 val[NPT];
#pragma unroll
      for (int k = 0; k < NPT; k++) {
        const int row = min(sr + SROWS * k, NROWS - 1);
        const int gy = min(max(y0 + row % CS_FY - 1, 0), p.ny - 1), gz = min(max(z0 + row / CS_FY - 1, 0), p.nz - 1);
        const size_t v = (size_t)(cgx >> sh) + snx * ((size_t)(gy >> sh) + sny * (size_t)(gz >> sh));
        val[k] = *reinterpret_cast<const uint4 *>(src + v * sc);
      }
#pragma unroll
      for (int k = 0; k < NPT; k++) {
        const int row = sr + SROWS * k, fy = row % CS_FY, fz = row / CS_FY;
        const int gy = y0 + fy - 1, gz = z0 + fz - 1;
        const bool in = sgx == cgx && gy >= 0 && gy < p.ny && gz >= 0 && gz < p.nz;
        if (sr < SROWS && row < NROWS)
          *reinterpret_cast<uint4 *>(sdst + row * ROW) = in ? val[k] : make_uint4(0u, 0u, 0u, 0u);
      }
    }
    __syncthreads();
    auto rd = [&](const bf16 *b, int plane, int row) __attribute__((always_inline)) {
      return *reinterpret_cast<const bf16x8 *>(b + plane * PLANE + row * ROW);
    };
#pragma unroll
    for (int pl = 0; pl < 6; pl++) {
      bf16x8 P[6], R[6], Q[5];
#pragma unroll
      for (int r = 0; r < 6; r++) {
        P[r] = rd(bP, pl, r);
        R[r] = rd(bR, pl, r);
        if (r < 5) Q[r] = rd(bQ, pl, r);
      }
      bf16x8 X[4], L[4];
#pragma unroll
      for (int y = 0; y < 4; y++) {
        if (pl >= 1 && pl <= 4) X[y] = rd(bX, pl - 1, y);
        if (pl >= 2) L[y] = rd(bL, pl, y);
      }
      // one product of every (plane offset, row) in turn: twelve sums in flight
#pragma unroll
      for (int st = 0; st < 5; st++) {
#pragma unroll
        for (int y = 0; y < 4; y++) {
          if (pl <= 3 && st < 4) {  // kz = 0: groups 0..3
            const bf16x8 &B = st == 0 ? P[y] : st == 1 ? Q[y] : st == 2 ? R[y + 1] : P[y + 2];
            acc[pl < 4 ? pl : 0][y] = mfma16x16x32(A[st], B, acc[pl < 4 ? pl : 0][y]);
          }
          if (pl >= 1 && pl <= 4) {  // the step to kz = 1, then groups 5..8
            const bf16x8 &B = st == 0 ? X[y] : st == 1 ? R[y] : st == 2 ? P[y + 1] : st == 3 ? Q[y + 1] : R[y + 2];
            const int z = pl >= 1 && pl <= 4 ? pl - 1 : 0;
            acc[z][y] = mfma16x16x32(A[4 + st], B, acc[z][y]);
          }
          if (pl >= 2) {  // kz = 2: groups 9..13
            const bf16x8 &B = st == 0 ? P[y] : st == 1 ? Q[y] : st == 2 ? R[y + 1] : st == 3 ? P[y + 2] : L[y];
            const int z = pl >= 2 ? pl - 2 : 0;
            acc[z][y] = mfma16x16x32(A[9 + st], B, acc[z][y]);
          }
        }
      }
    }
  }
  const int gx = x0 + col;
  bf16x4 act[4][4];
  if (!RELU) {
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++) act[z][y] = act_at<16>(p, gx, y0 + wy + y, z0 + wz + z, 4 * j);
  }
  if (gx >= p.nx) return;
  float bias[4];
#pragma unroll
  for (int i = 0; i < 4; i++) bias[i] = p.bias ? p.bias[4 * j + i] : 0.0f;
#pragma unroll
  for (int z = 0; z < 4; z++) {
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const int gy = y0 + wy + y, gz = z0 + wz + z;
      if (gy >= p.ny || gz >= p.nz) continue;
      const size_t v = (size_t)gx + (size_t)p.nx * ((size_t)gy + (size_t)p.ny * (size_t)gz);
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float t = acc[z][y][i] + bias[i];
        if (RELU ? !(t > 0.0f) : !(bf(act[z][y][i]) > 0.0f)) t = 0.0f;
        o[i] = tobf(t);
      }
      *reinterpret_cast<bf16x4 *>(p.out + v * 16 + 4 * j) = o;
    }
  }
}

bool launch_conv3(const G3 &g, const bf16 *a, const G3 &ga, int ca, const bf16 *b, int cb, const bf16 *wp,
                  const float *bias, int cout, bool relu, bf16 *out, hipStream_t s, const bf16 *act, int split) {
  ConvArgs p;
  p.nx = g.nx; p.ny = g.ny; p.nz = g.nz;
  p.anx = ga.nx; p.any = ga.ny;
  p.a = a; p.b = b; p.wp = wp; p.bias = bias; p.act = act; p.out = out; p.split = split ? split : cout;
  const unsigned nb = (unsigned)(((g.nx + CV_TX - 1) / CV_TX) * ((g.ny + CV_TY - 1) / CV_TY) *
                                 ((g.nz + CV_TZ - 1) / CV_TZ));
  const unsigned nb16 = (unsigned)(((g.nx + CV_TX - 1) / CV_TX) * ((g.ny + CS_Y - 1) / CS_Y) *
                                   ((g.nz + CS_Z - 1) / CS_Z));
  // A layer on a coarse grid has fewer tiles than the chip has compute units.
  // Its output channels are then split over MS blocks a tile, as far as all
  // blocks are resident at once (three to a compute unit, 768).  In us, one
  // block a tile and split: 64 -> 64 at 6 tiles 23 and 12, at 100 32 and 17, at
  // 192 44 and 23; 96 -> 32 at 15 tiles 23 and 20, at 120 34 and 23, at 384 37
  // and 34, at 512 38 and 53; 32 -> 96 at 120 tiles 24 and 14, at 256 31 and 22
  // (two blocks; 25 with six), at 600 41 and 45.
  constexpr unsigned RESIDENT = 768;
#define PYRO_CONV(CA_, CB_, CO_, R_)                                                                        \
  if (ca == CA_ && cb == CB_ && cout == CO_ && relu == R_) {                                                \
    constexpr int S1 = CO_ / 16, S2 = CO_ == 64 || CO_ == 96 ? 2 : 1;                                       \
    if (nb * S1 <= RESIDENT) k_conv3<CA_, CB_, CO_, R_, S1><<<dim3(nb, S1), 256, 0, s>>>(p);                \
    else if (nb * S2 <= RESIDENT) k_conv3<CA_, CB_, CO_, R_, S2><<<dim3(nb, S2), 256, 0, s>>>(p);           \
    else k_conv3<CA_, CB_, CO_, R_, 1><<<nb, 256, 0, s>>>(p);                                               \
    return true;                                                                                            \
  }
#define PYRO_CONV16(CA_, R_)                                      \
  if (ca == CA_ && cb == 16 && cout == 16 && relu == R_) {        \
    k_conv3_16<CA_, R_><<<nb16, 256, 0, s>>>(p);                  \
    return true;                                                  \
  }
  // Small grids: the small tiles give four times the workgroups, and while
  // all of them are resident at once (two to a compute unit) a launch lasts as
  // long as one of them.  The forward pass with either kernel for these
  // layers: 24x40x24 (120 small tiles) 110 us against 118, 40x64x40 (480) 123
  // against 127; 48x80x48 (720) 151 against 152.5, 64x64x64 (1024) 166 against 157.
  if (nb <= 512) {
    PYRO_CONV(0, 16, 16, true)
    PYRO_CONV(32, 16, 16, true)
    PYRO_CONV(0, 16, 16, false)
  }
  PYRO_CONV16(0, true)
  PYRO_CONV16(32, true)
  PYRO_CONV16(0, false)
#undef PYRO_CONV16
  PYRO_CONV(0, 16, 32, true)
  PYRO_CONV(0, 32, 32, true)
  PYRO_CONV(0, 32, 64, true)
  PYRO_CONV(0, 64, 64, true)
  PYRO_CONV(64, 32, 32, true)
  PYRO_CONV(0, 32, 16, false)
  PYRO_CONV(0, 32, 32, false)
  PYRO_CONV(0, 64, 32, false)
  PYRO_CONV(0, 64, 64, false)
  PYRO_CONV(0, 32, 96, false)
  PYRO_CONV(0, 16, 48, false)
#undef PYRO_CONV
  return false;
}

// ------------------------------------------------------------ first layer, head, pool
// First layer on MFMA: 27 taps x 2 channels = 54 of the K = 64 of two K32
// groups (group g holds taps 16g .. 16g+15, channel-minor; taps past 26 have
// zero weights).  Lane group j of a B fragment holds 4 taps x 2 channels, one
// 4-byte LDS word per tap.  Packed weights: [2][16][32].
__global__ __launch_bounds__(256) void k_pack_conv_in(const float *__restrict__ W, bf16 *__restrict__ wp) {
  const int e = threadIdx.x + 256 * blockIdx.x;
  if (e >= 2 * 16 * 32) return;
  const int kk = e % 32, co = (e / 32) % 16, g = e / 512;
  const int tap = 16 * g + kk / 2, ci = kk % 2;
  wp[e] = tobf(tap < 27 ? W[(co * 2 + ci) * 27 + tap] : 0.0f);
}
void launch_pack_conv_in(const float *W, bf16 *wp, hipStream_t s) { k_pack_conv_in<<<4, 256, 0, s>>>(W, wp); }

__global__ __launch_bounds__(256) void k_conv_in(int nx, int ny, int nz, const bf16 *__restrict__ x0,
                                                 const bf16 *__restrict__ wp, const float *__restrict__ bias,
                                                 bf16 *__restrict__ out) {
  __shared__ uint32_t lds[CV_FN];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = lane >> 4, col = lane & 15;
  const int ntx = (nx + CV_TX - 1) / CV_TX, nty = (ny + CV_TY - 1) / CV_TY;
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0v = tx * CV_TX, y0 = ty * CV_TY, z0 = tz * CV_TZ;
  const uint32_t *src = reinterpret_cast<const uint32_t *>(x0);
  for (int s = threadIdx.x; s < CV_FN; s += 256) {
    const int fx = s % CV_FX, r2 = s / CV_FX, fy = r2 % CV_FY, fz = r2 / CV_FY;
    const int gx = x0v + fx - 1, gy = y0 + fy - 1, gz = z0 + fz - 1;
    uint32_t v = 0u;
    if (gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz)
      v = src[(size_t)gx + (size_t)nx * ((size_t)gy + (size_t)ny * (size_t)gz)];
    lds[s] = v;
  }
  bf16x8 A[2];
#pragma unroll
  for (int g = 0; g < 2; g++) A[g] = *reinterpret_cast<const bf16x8 *>(wp + (g * 16 + col) * 32 + 8 * j);
  __syncthreads();
  f32x4 acc[4];
#pragma unroll
  for (int nb = 0; nb < 4; nb++) acc[nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int base = w * CV_FX + col;
#pragma unroll
  for (int g = 0; g < 2; g++) {
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      uint4 u;
      uint32_t t4[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        int t = 16 * g + 4 * j + i;
        t = t > 26 ? 26 : t;  // zero weights beyond the 27 taps
        t4[i] = lds[base + nb * (CV_FX * CV_FY) + tap_off(t)];
      }
      u.x = t4[0]; u.y = t4[1]; u.z = t4[2]; u.w = t4[3];
      acc[nb] = mfma16x16x32(A[g], __builtin_bit_cast(bf16x8, u), acc[nb]);
    }
  }
  const int gx = x0v + col, gy = y0 + w;
  if (gx >= nx || gy >= ny) return;
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
    const int gz = z0 + nb;
    if (gz >= nz) continue;
    const size_t v = (size_t)gx + (size_t)nx * ((size_t)gy + (size_t)ny * (size_t)gz);
    const int co = 4 * j;
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float t = acc[nb][i] + bias[co + i];
      o[i] = tobf(t > 0.0f ? t : 0.0f);
    }
    *reinterpret_cast<bf16x4 *>(out + v * 16 + co) = o;
  }
}
void launch_conv_in(const G3 &g, const bf16 *x0, const bf16 *wp, const float *bias, bf16 *out, hipStream_t s) {
  const unsigned nb = (unsigned)(((g.nx + CV_TX - 1) / CV_TX) * ((g.ny + CV_TY - 1) / CV_TY) *
                                 ((g.nz + CV_TZ - 1) / CV_TZ));
  k_conv_in<<<nb, 256, 0, s>>>(g.nx, g.ny, g.nz, x0, wp, bias, out);
}

__global__ __launch_bounds__(256) void k_head(uint32_t n, const bf16 *__restrict__ d0, const float *__restrict__ wh,
                                              const float *__restrict__ bh, float *__restrict__ y) {
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  if (v >= n) return;
  const bf16x8 a = *reinterpret_cast<const bf16x8 *>(d0 + 16 * (size_t)v);
  const bf16x8 b = *reinterpret_cast<const bf16x8 *>(d0 + 16 * (size_t)v + 8);
  float t = bh[0];
#pragma unroll
  for (int c = 0; c < 8; c++) t += wh[c] * bf(a[c]);
#pragma unroll
  for (int c = 0; c < 8; c++) t += wh[8 + c] * bf(b[c]);
  y[v] = t;
}
void launch_head(const G3 &g, const bf16 *d0, const float *wh, const float *bh, float *y, hipStream_t s) {
  k_head<<<nblk(g.n()), 256, 0, s>>>(g.n(), d0, wh, bh, y);
}

// children of coarse voxel (ux, uy, uz) in the fine grid, in z, y, x order
__global__ __launch_bounds__(256) void k_pool(int nx, int ny, int nz, int c, const bf16 *__restrict__ in,
                                              bf16 *__restrict__ out) {
  const int cnx = (nx + 1) / 2, cny = (ny + 1) / 2, cnz = (nz + 1) / 2;
  const int ng = c / 8;
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  const uint32_t total = (uint32_t)cnx * cny * cnz * ng;
  if (t >= total) return;
  const int cg = (int)(t % (uint32_t)ng);
  const uint32_t u = t / (uint32_t)ng;
  const int ux = (int)(u % (uint32_t)cnx), r = (int)(u / (uint32_t)cnx), uy = r % cny, uz = r / cny;
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int cnt = 0;
  for (int dz = 0; dz < 2; dz++)
    for (int dy = 0; dy < 2; dy++)
      for (int dx = 0; dx < 2; dx++) {
        const int x = 2 * ux + dx, y = 2 * uy + dy, z = 2 * uz + dz;
        if (x >= nx || y >= ny || z >= nz) continue;
        const size_t v = (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * (size_t)z);
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(in + v * c + 8 * cg);
#pragma unroll
        for (int i = 0; i < 8; i++) s[i] += bf(a[i]);
        cnt++;
      }
  const float inv = 1.0f / (float)cnt;
  bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = tobf(s[i] * inv);
  *reinterpret_cast<bf16x8 *>(out + (size_t)u * c + 8 * cg) = o;
}
void launch_pool(const G3 &g, const bf16 *in, int c, bf16 *out, hipStream_t s) {
  const G3 h = half_of(g);
  k_pool<<<nblk((uint64_t)h.n() * (c / 8)), 256, 0, s>>>(g.nx, g.ny, g.nz, c, in, out);
}

// ------------------------------------------------------------ backward glue
__global__ __launch_bounds__(256) void k_unup_relu(int nx, int ny, int nz, const bf16 *__restrict__ gcat,
                                                   int ca, const bf16 *__restrict__ act, bf16 *__restrict__ gc) {
  const int cnx = (nx + 1) / 2, cny = (ny + 1) / 2, cnz = (nz + 1) / 2;
  const int ng = ca / 8;
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= (uint32_t)cnx * cny * cnz * ng) return;
  const int cg = (int)(t % (uint32_t)ng);
  const uint32_t u = t / (uint32_t)ng;
  const int ux = (int)(u % (uint32_t)cnx), r = (int)(u / (uint32_t)cnx), uy = r % cny, uz = r / cny;
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int dz = 0; dz < 2; dz++)
    for (int dy = 0; dy < 2; dy++)
      for (int dx = 0; dx < 2; dx++) {
        const int x = 2 * ux + dx, y = 2 * uy + dy, z = 2 * uz + dz;
        if (x >= nx || y >= ny || z >= nz) continue;
        const size_t v = (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * (size_t)z);
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(gcat + v * ca + 8 * cg);
#pragma unroll
        for (int i = 0; i < 8; i++) s[i] += bf(a[i]);
      }
  const bf16x8 a = *reinterpret_cast<const bf16x8 *>(act + (size_t)u * ca + 8 * cg);
  bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = tobf(bf(a[i]) > 0.0f ? s[i] : 0.0f);
  *reinterpret_cast<bf16x8 *>(gc + (size_t)u * ca + 8 * cg) = o;
}
void launch_unup_relu(const G3 &g, const bf16 *gcat, int ca, const G3 &gc, const bf16 *act, bf16 *gcoarse,
                      hipStream_t s) {
  k_unup_relu<<<nblk((uint64_t)gc.n() * (ca / 8)), 256, 0, s>>>(g.nx, g.ny, g.nz, gcat, ca, act, gcoarse);
}

__global__ __launch_bounds__(256) void k_skip_grad(int nx, int ny, int nz, const bf16 *__restrict__ gc,
                                                   const bf16 *__restrict__ gp, const bf16 *__restrict__ sa,
                                                   int c, bf16 *__restrict__ gs) {
  const int ng = c / 8;
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= (uint32_t)nx * ny * nz * ng) return;
  const int cg = (int)(t % (uint32_t)ng);
  const uint32_t v = t / (uint32_t)ng;
  const int x = (int)(v % (uint32_t)nx), r = (int)(v / (uint32_t)nx), y = r % ny, z = r / ny;
  const int cnx = (nx + 1) / 2, cny = (ny + 1) / 2;
  const int ux = x >> 1, uy = y >> 1, uz = z >> 1;
  // children of the parent inside the grid
  const int cnt = (2 * ux + 1 < nx ? 2 : 1) * (2 * uy + 1 < ny ? 2 : 1) * (2 * uz + 1 < nz ? 2 : 1);
  const float inv = 1.0f / (float)cnt;
  const size_t u = (size_t)ux + (size_t)cnx * ((size_t)uy + (size_t)cny * (size_t)uz);
  const bf16x8 a = *reinterpret_cast<const bf16x8 *>(gc + (size_t)v * c + 8 * cg);
  const bf16x8 b = *reinterpret_cast<const bf16x8 *>(gp + u * c + 8 * cg);
  const bf16x8 m = *reinterpret_cast<const bf16x8 *>(sa + (size_t)v * c + 8 * cg);
  bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = tobf(bf(m[i]) > 0.0f ? bf(a[i]) + bf(b[i]) * inv : 0.0f);
  *reinterpret_cast<bf16x8 *>(gs + (size_t)v * c + 8 * cg) = o;
}
void launch_skip_grad(const G3 &g, const bf16 *gc, const bf16 *gp, const bf16 *s, int c, bf16 *gs, hipStream_t st) {
  k_skip_grad<<<nblk((uint64_t)g.n() * (c / 8)), 256, 0, st>>>(g.nx, g.ny, g.nz, gc, gp, s, c, gs);
}

// head backward: gd0 and per-block partial sums of dwh (16) and dbh (1)
constexpr int HB_BLOCKS = 512;
static_assert(HB_BLOCKS * 17 == HEAD_PART);
__global__ __launch_bounds__(256) void k_head_bwd(uint32_t n, const bf16 *__restrict__ d0, const float *__restrict__ gy,
                                                  const float *__restrict__ wh, bf16 *__restrict__ gd0,
                                                  float *__restrict__ part) {
  float s[17];
#pragma unroll
  for (int c = 0; c < 17; c++) s[c] = 0.0f;
  for (uint32_t v = blockIdx.x * 256u + threadIdx.x; v < n; v += HB_BLOCKS * 256u) {
    const float g = gy[v];
    bf16x8 a = *reinterpret_cast<const bf16x8 *>(d0 + 16 * (size_t)v);
    bf16x8 b = *reinterpret_cast<const bf16x8 *>(d0 + 16 * (size_t)v + 8);
    bf16x8 oa, ob;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      s[c] += g * bf(a[c]);
      s[8 + c] += g * bf(b[c]);
      oa[c] = tobf(bf(a[c]) > 0.0f ? g * wh[c] : 0.0f);
      ob[c] = tobf(bf(b[c]) > 0.0f ? g * wh[8 + c] : 0.0f);
    }
    s[16] += g;
    *reinterpret_cast<bf16x8 *>(gd0 + 16 * (size_t)v) = oa;
    *reinterpret_cast<bf16x8 *>(gd0 + 16 * (size_t)v + 8) = ob;
  }
  __shared__ float sh[256];
  for (int c = 0; c < 17; c++) {
    sh[threadIdx.x] = s[c];
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
      if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
      __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x * 17 + c] = sh[0];
    __syncthreads();
  }
}
void launch_head_bwd(const G3 &g, const bf16 *d0, const float *gy, const float *wh, bf16 *gd0, float *part,
                     float *dwh, float *dbh, DwSums &sums, hipStream_t s) {
  k_head_bwd<<<HB_BLOCKS, 256, 0, s>>>(g.n(), d0, gy, wh, gd0, part);
  sums.hpart = part;
  sums.dwh = dwh;
  sums.dbh = dbh;
}

// ------------------------------------------------------------ weight gradients
// dW[co][ci][t] = sum_v g[v][co] * X[v + off(t)][ci].  The MFMA contracts over
// voxels, so both operands are first written channel-major: GT[co][z][y][x]
// (rows of P, a multiple of 32) and XT[ci][z + 1][y + 1][x + 8] (rows of
// P + 16, zero outside the grid).  A B fragment is eight consecutive x of one
// channel: the three x shifts of a row come from one aligned 16-byte load and
// the words beside it (in other lanes), by funnel shifts.
constexpr int DW_PAD = 8;  // elements before x = 0 and after x = P - 1
DwPlan dw_plan(const G3 &g, const ConvSpec &c) {
  DwPlan d;
  d.P = (g.nx + 31) / 32 * 32;
  d.rows_x = c.cin() < 16 ? 16 : c.cin();
  const int tasks = 27 * (d.rows_x / 16);
  int S = (2048 + tasks - 1) / tasks;
  const int rows = g.ny * g.nz;
  const int smax = rows / 4 > 0 ? rows / 4 : 1;
  d.S = S < 1 ? 1 : (S > smax ? smax : S);
  return d;
}
size_t dw_xt_elems(const G3 &g, const ConvSpec &c) {
  const DwPlan d = dw_plan(g, c);
  return (size_t)d.rows_x * (size_t)(g.nz + 2) * (size_t)(g.ny + 2) * (size_t)(d.P + 2 * DW_PAD);
}
size_t dw_gt_elems(const G3 &g, const ConvSpec &c) {
  const DwPlan d = dw_plan(g, c);
  return (size_t)c.cout * (size_t)g.nz * (size_t)g.ny * (size_t)d.P;
}
constexpr int BG_BLOCKS = 256;  // partials of the bias gradient
static size_t dw_bias_at(const DwPlan &d, int cout) { return (size_t)d.S * 27 * cout * d.rows_x; }
size_t dw_part_elems(const G3 &g, const ConvSpec &c) {
  return dw_bias_at(dw_plan(g, c), c.cout) + (size_t)BG_BLOCKS * c.cout;
}

// (Three shifted copies of XT, one per x tap, took three times the writes: 34
// + 10 us a layer against 22 us for both operands.)
// XT of the concatenated conv input [up(a) (ca ch), b (cb ch)] (cb = 2: the
// network input, rows 2..15 zero) in the first xgroups rows of blocks, GT in
// the rest: a row takes eight channels, a thread two x of them, one 4-byte
// store per channel.  The bias gradient's blocks come before them: a launch of
// its own, one block a CU, waits on its loads most of the time (eight layers at
// 80x160x80 182 + 72 us a step, together 198).
struct TransArgs {
  int nx, ny, nz, P, anx, any, ca, cb, xgroups;
  const bf16 *a, *b, *g;
  bf16 *xt, *gt;
  uint32_t x_items, g_items;  // per group of eight channels
  FastDiv dxp, dxy, dgp, dgy;  // (P + 16) / 2, ny + 2; P / 2, ny
  uint32_t n;                  // voxels
  float *bpart;
  FastDiv dnb;  // blocks a row
};
// bias gradient: partials of db[c] = sum_v g[v][c], sixteen loads in flight
template <int C>
__device__ __forceinline__ void bias_grad(uint32_t n, const bf16 *__restrict__ g, float *__restrict__ part) {
  constexpr uint32_t VL = 256 / C, STEP = BG_BLOCKS * VL, U = 16;
  const uint32_t c = threadIdx.x % C, vl = threadIdx.x / C;
  float s = 0.0f;
  uint32_t v = blockIdx.x * VL + vl;
  for (; (uint64_t)v + (U - 1) * STEP < n; v += U * STEP) {
    bf16 x[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) x[u] = g[(size_t)(v + u * STEP) * C + c];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) s += bf(x[u]);
  }
  for (; v < n; v += STEP) s += bf(g[(size_t)v * C + c]);
  __shared__ float sh[256];
  sh[threadIdx.x] = s;
  __syncthreads();
  if (vl == 0) {
    float t = 0.0f;
    for (uint32_t k = 0; k < VL; k++) t += sh[k * C + c];
    part[blockIdx.x * C + c] = t;
  }
}
__device__ __forceinline__ uint32_t pair_of(bf16 lo, bf16 hi) {
  return (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
}
template <int COUT>
__global__ __launch_bounds__(256) void k_to_t(TransArgs p) {
  if (blockIdx.x < BG_BLOCKS) {
    bias_grad<COUT>(p.n, p.g, p.bpart);
    return;
  }
  const uint32_t id = blockIdx.x - BG_BLOCKS, row = fdiv(id, p.dnb);
  const uint32_t t = (id - row * p.dnb.d) * 256u + threadIdx.x;
  bf16x8 v[2];
#pragma unroll
  for (int e = 0; e < 2; e++)
#pragma unroll
    for (int i = 0; i < 8; i++) v[e][i] = tobf(0.0f);
  if ((int)row < p.xgroups) {
    if (t >= p.x_items) return;
    const uint32_t hp = p.dxp.d, h2 = p.dxy.d, r = fdiv(t, p.dxp), zz = fdiv(r, p.dxy), yy = r - zz * h2;
    const int xp = 2 * (int)(t - r * hp);
    const int y = (int)yy - 1, z = (int)zz - 1, c = 8 * (int)row;
    if (y >= 0 && y < p.ny && z >= 0 && z < p.nz) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int x = xp + e - DW_PAD;
        if (x < 0 || x >= p.nx) continue;
        const size_t w = (size_t)x + (size_t)p.nx * ((size_t)y + (size_t)p.ny * (size_t)z);
        if (p.cb == 2) {
          if (c == 0) {
            v[e][0] = p.b[2 * w];
            v[e][1] = p.b[2 * w + 1];
          }
        } else if (c < p.ca) {
          const size_t u = (size_t)(x >> 1) + (size_t)p.anx * ((size_t)(y >> 1) + (size_t)p.any * (size_t)(z >> 1));
          v[e] = *reinterpret_cast<const bf16x8 *>(p.a + u * p.ca + c);
        } else {
          v[e] = *reinterpret_cast<const bf16x8 *>(p.b + w * p.cb + (c - p.ca));
        }
      }
    }
    const size_t plane = 2 * (size_t)p.x_items;
    const size_t base = (size_t)c * plane + 2 * (size_t)t;
#pragma unroll
    for (int i = 0; i < 8; i++)
      *reinterpret_cast<uint32_t *>(p.xt + base + (size_t)i * plane) = pair_of(v[0][i], v[1][i]);
    return;
  }
  if (t >= p.g_items) return;
  const uint32_t r = fdiv(t, p.dgp), z = fdiv(r, p.dgy), y = r - z * p.dgy.d;
  const int xp = 2 * (int)(t - r * p.dgp.d), c = 8 * ((int)row - p.xgroups);
#pragma unroll
  for (int e = 0; e < 2; e++) {
    if (xp + e >= p.nx) continue;
    const size_t w = (size_t)(xp + e) + (size_t)p.nx * ((size_t)y + (size_t)p.ny * (size_t)z);
    v[e] = *reinterpret_cast<const bf16x8 *>(p.g + w * COUT + c);
  }
  const size_t plane = 2 * (size_t)p.g_items;
  const size_t base = (size_t)c * plane + 2 * (size_t)t;
#pragma unroll
  for (int i = 0; i < 8; i++)
    *reinterpret_cast<uint32_t *>(p.gt + base + (size_t)i * plane) = pair_of(v[0][i], v[1][i]);
}

// One block per (z tap, 16-channel input block, row split); its 4 waves take
// interleaved quarters of the split's rows and are summed through LDS.  A
// wave keeps the sums of the nine (y, x) taps, so an A fragment (g) and the
// three rows of X are loaded once for nine products each; with one block per
// tap, every product loaded both of its fragments and the kernel ran at the
// L2's rate (the 16-channel layers at 80x160x80: 446 us on average).  One wave
// runs per SIMD, so the latency of its loads is hidden by fetching ahead: 133
// us, and 80 us with the rows kept (NC below); the products alone are 20 us.  Each tap's sum runs over the same
// rows in the same order whatever shares the loads.
//
// NC = P / 32 up to 3 (rows of 96): the three rows stay in registers and a
// step down y loads one new row, two rows ahead (the wave's rows exceed L1,
// so every row would come from L2 three times); NC = 0 loads the three rows
// of a step three steps ahead.
template <int COUT, int NC>
__global__ __launch_bounds__(256) void k_dw(int ny, int nz, int P, int rows_x, int S, const bf16 *__restrict__ gt,
                                            const bf16 *__restrict__ xt, float *__restrict__ part) {
  constexpr int MB = COUT / 16;
  const int ncib = rows_x / 16;
  const int task = blockIdx.x % (3 * ncib), split = blockIdx.x / (3 * ncib);
  const int dzi = task / ncib, cib = task % ncib;
  const int lane = threadIdx.x & 63, j = lane >> 4, col = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int rows = nz * ny;
  const int pid = split * 4 + w, np = S * 4;
  const int r0 = (int)((int64_t)rows * pid / np), r1 = (int)((int64_t)rows * (pid + 1) / np);
  const int PX = P + 2 * DW_PAD;
  const size_t xplane = (size_t)(nz + 2) * (ny + 2) * PX;
  const size_t gplane = (size_t)nz * ny * P;
  const bf16 *xb = xt + (size_t)(cib * 16 + col) * xplane + DW_PAD + 8 * j;
  const bf16 *gb = gt + (size_t)col * gplane + 8 * j;
  f32x4 acc[9][MB];
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int m = 0; m < MB; m++) acc[t][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // the words beside a lane's eight x lie in the lanes 16 away, for the first
  // and last of a step in the neighbouring step's fragment of the row (0
  // beyond the row: x = -1, and x = P, which meets zeros of g)
  const int from_lo = ((lane + 48) & 63) * 4, from_hi = ((lane + 16) & 63) * 4;
  // the nine products of one step: row d's fragment c, the last word bw of
  // the step before it and the first word aw of the step after it
  auto multiply = [&](const bf16x8 *A, int d, const uint4 &c, uint32_t bw, uint32_t aw)
      __attribute__((always_inline)) {
    const uint32_t p = (uint32_t)__builtin_amdgcn_ds_bpermute(from_lo, (int)(j == 3 ? bw : c.w));
    const uint32_t n = (uint32_t)__builtin_amdgcn_ds_bpermute(from_hi, (int)(j == 0 ? aw : c.x));
    const uint32_t s1 = __builtin_amdgcn_alignbit(c.y, c.x, 16), s2 = __builtin_amdgcn_alignbit(c.z, c.y, 16),
                   s3 = __builtin_amdgcn_alignbit(c.w, c.z, 16);
    const uint4 lo = make_uint4(__builtin_amdgcn_alignbit(c.x, p, 16), s1, s2, s3);  // x - 1
    const uint4 hi = make_uint4(s1, s2, s3, __builtin_amdgcn_alignbit(n, c.w, 16));  // x + 1
#pragma unroll
    for (int m = 0; m < MB; m++) {
      acc[3 * d][m] = mfma16x16x32(A[m], __builtin_bit_cast(bf16x8, lo), acc[3 * d][m]);
      acc[3 * d + 1][m] = mfma16x16x32(A[m], __builtin_bit_cast(bf16x8, c), acc[3 * d + 1][m]);
      acc[3 * d + 2][m] = mfma16x16x32(A[m], __builtin_bit_cast(bf16x8, hi), acc[3 * d + 2][m]);
    }
  };
  if constexpr (NC > 0) {
    struct Row {
      bf16x8 A[NC][MB];  // g of the row
      uint4 c[NC];       // X two rows below its first
    };
    auto load_x = [&](uint4 *c, int z, int yy) __attribute__((always_inline)) {
      const bf16 *xr = xb + ((size_t)(z + dzi) * (ny + 2) + yy) * PX;
#pragma unroll
      for (int q = 0; q < NC; q++) c[q] = *reinterpret_cast<const uint4 *>(xr + 32 * q);
    };
    constexpr int D = 2;  // rows ahead
    Row Q[D];
    int ar = r0, az = r0 / ny, ay = r0 - az * ny;  // the next row to fetch
    auto fetch = [&](Row &to) __attribute__((always_inline)) {
      if (ar >= r1) return;
      const bf16 *gr = gb + (size_t)ar * P;
#pragma unroll
      for (int q = 0; q < NC; q++)
#pragma unroll
        for (int m = 0; m < MB; m++)
          to.A[q][m] = *reinterpret_cast<const bf16x8 *>(gr + (size_t)m * 16 * gplane + 32 * q);
      load_x(to.c, az, ay + 2);
      ar++;
      if (++ay == ny) {
        ay = 0;
        az++;
      }
    };
    int z = az, y = ay;
    uint4 W[3][NC];
#pragma unroll
    for (int u = 0; u < D; u++) fetch(Q[u]);
    bool fresh = true;
    for (int r = r0; r < r1; r += D) {
#pragma unroll
      for (int u = 0; u < D; u++) {
        if (r + u < r1) {
          if (fresh) {  // the first row, or the first of a plane
            load_x(W[0], z, y);
            load_x(W[1], z, y + 1);
          }
#pragma unroll
          for (int q = 0; q < NC; q++) W[2][q] = Q[u].c[q];
#pragma unroll
          for (int q = 0; q < NC; q++)
#pragma unroll
            for (int d = 0; d < 3; d++)
              multiply(Q[u].A[q], d, W[d][q], q > 0 ? W[d][q > 0 ? q - 1 : 0].w : 0u,
                       q + 1 < NC ? W[d][q + 1 < NC ? q + 1 : 0].x : 0u);
          fetch(Q[u]);
#pragma unroll
          for (int q = 0; q < NC; q++) {
            W[0][q] = W[1][q];
            W[1][q] = W[2][q];
          }
          fresh = ++y == ny;
          if (fresh) {
            y = 0;
            z++;
          }
        }
      }
    }
  } else if (r0 < r1) {
    struct Frag {
      bf16x8 A[MB];
      uint4 c[3];
    };
    int r = r0, z = r0 / ny, y = r0 - z * ny, xc = 0;  // the next step to fetch
    constexpr int D = 4;  // fragments in flight: a load is issued three steps before its use
    const int steps = (r1 - r0) * (P / 32);
    Frag f[D];
    int ahead = 0, at = 0;  // steps fetched; x of the step that multiplies
    auto fetch = [&](Frag &to) __attribute__((always_inline)) {
      if (ahead >= steps) return;
      const bf16 *gr = gb + (size_t)r * P + xc;
#pragma unroll
      for (int m = 0; m < MB; m++) to.A[m] = *reinterpret_cast<const bf16x8 *>(gr + (size_t)m * 16 * gplane);
      const bf16 *xr = xb + ((size_t)(z + dzi) * (ny + 2) + y) * PX + xc;
#pragma unroll
      for (int d = 0; d < 3; d++) to.c[d] = *reinterpret_cast<const uint4 *>(xr + d * PX);
      ahead++;
      xc += 32;
      if (xc < P) return;
      xc = 0;
      r++;
      if (++y == ny) {
        y = 0;
        z++;
      }
    };
    uint32_t before[3] = {0u, 0u, 0u};  // last words of the step before
#pragma unroll
    for (int u = 0; u < D - 1; u++) fetch(f[u]);
    for (int k = 0; k < steps; k += D) {
#pragma unroll
      for (int u = 0; u < D; u++) {
        fetch(f[(u + D - 1) % D]);
        if (k + u < steps) {
          const bool first = at == 0, last = at == P - 32;
#pragma unroll
          for (int d = 0; d < 3; d++) {
            multiply(f[u].A, d, f[u].c[d], first ? 0u : before[d], last ? 0u : f[(u + 1) % D].c[d].x);
            before[d] = f[u].c[d].w;
          }
          at = last ? 0 : at + 32;
        }
      }
    }
  }
  __shared__ float red[4][COUT * 16];
#pragma unroll
  for (int t = 0; t < 9; t++) {
    if (t) __syncthreads();
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
      for (int i = 0; i < 4; i++) red[w][(m * 16 + 4 * j + i) * 16 + col] = acc[t][m][i];
    __syncthreads();
    for (int e = threadIdx.x; e < COUT * 16; e += 256) {
      const float s = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
      const int co = e / 16, c = e % 16;
      part[(((size_t)split * 27 + 9 * dzi + t) * COUT + co) * rows_x + cib * 16 + c] = s;
    }
  }
}
// a[first] + a[first + step] + ... (count terms) in that order, U loads in flight
typedef const float __attribute__((address_space(1))) *gf32c;
typedef float __attribute__((address_space(1))) *gf32;
template <int U>
__device__ __forceinline__ float seq_sum32(gf32c a, int count, size_t first, size_t step) {
  float s = 0.0f;
  for (int k0 = 0; k0 < count; k0 += U) {
    float x[U];
#pragma unroll
    for (int u = 0; u < U; u++) x[u] = k0 + u < count ? a[first + (size_t)(k0 + u) * step] : 0.0f;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + u < count) s += x[u];
  }
  return s;
}
// Every layer's dW from its row splits' partials (input channel fastest, as
// they lie), in a layer's last block the bias gradient from its partials, and
// in the launch's last the head's.  A launch a layer is bound by the round
// trips of one sum (6 us, and 10 for the head's): eight layers and the head
// 59 us a training step at 80x160x80, 17 in one launch.
__global__ __launch_bounds__(256) void k_dw_reduce(DwSums) {
  // indexed by block where the arguments lie
  const DwSums &a = *(const DwSums *)__builtin_amdgcn_kernarg_segment_ptr();
  if (a.hpart && blockIdx.x == a.blocks) {
    const int c = threadIdx.x;
    if (c >= 17) return;
    const float s = seq_sum32<32>((gf32c)a.hpart, HB_BLOCKS, (size_t)c, 17);
    *(c < 16 ? (gf32)a.dwh + c : (gf32)a.dbh) = s;
    return;
  }
  int k = 0;
  while (k + 1 < a.n && blockIdx.x >= a.e[k + 1].block0) k++;
  const DwSums::Entry &p = a.e[k];
  const int e = (int)(blockIdx.x - p.block0) * 256 + threadIdx.x, total = p.cout * p.cin * 27;
  const int nb = (total + 255) / 256;
  if ((int)(blockIdx.x - p.block0) == nb) {
    const int c = threadIdx.x;
    if (c >= p.cout) return;
    ((gf32)p.db)[c] = seq_sum32<32>((gf32c)p.bpart, BG_BLOCKS, (size_t)c, (size_t)p.cout);
    return;
  }
  if (e >= total) return;
  const int ci = e % p.cin, co = (e / p.cin) % p.cout, t = e / (p.cin * p.cout);
  const float s = seq_sum32<16>((gf32c)p.part, p.S, ((size_t)t * p.cout + co) * p.rows_x + ci,
                                (size_t)27 * p.cout * p.rows_x);
  ((gf32)p.dW)[((size_t)co * p.cin + ci) * 27 + t] = s;
}
void launch_dw_reduce(const DwSums &sums, hipStream_t s) {
  k_dw_reduce<<<sums.blocks + (sums.hpart ? 1 : 0), 256, 0, s>>>(sums);
}

template <int COUT>
static void launch_dw(unsigned nb, const G3 &g, const DwPlan &d, const bf16 *gt, const bf16 *xt, float *part,
                      hipStream_t s) {
  switch (d.P) {
    case 32: k_dw<COUT, 1><<<nb, 256, 0, s>>>(g.ny, g.nz, d.P, d.rows_x, d.S, gt, xt, part); break;
    case 64: k_dw<COUT, 2><<<nb, 256, 0, s>>>(g.ny, g.nz, d.P, d.rows_x, d.S, gt, xt, part); break;
    case 96:
      if constexpr (COUT < 64) {  // 64 channels and three steps do not fit the registers
        k_dw<COUT, 3><<<nb, 256, 0, s>>>(g.ny, g.nz, d.P, d.rows_x, d.S, gt, xt, part);
        break;
      }
      [[fallthrough]];
    default: k_dw<COUT, 0><<<nb, 256, 0, s>>>(g.ny, g.nz, d.P, d.rows_x, d.S, gt, xt, part); break;
  }
}
// weight and bias gradients of one layer (cb = 2: the first)
static void launch_dw_layer(const G3 &g, const ConvSpec &c, const bf16 *a, const G3 &ga, const bf16 *b,
                            const bf16 *gpre, bf16 *xt, bf16 *gt, float *part, float *dW, float *db, DwSums &sums,
                            hipStream_t s) {
  const DwPlan d = dw_plan(g, c);
  TransArgs p;
  p.nx = g.nx; p.ny = g.ny; p.nz = g.nz;
  p.P = d.P;
  p.anx = ga.nx; p.any = ga.ny;
  p.ca = c.ca; p.cb = c.cb;
  p.a = a; p.b = b; p.g = gpre;
  p.xt = xt; p.gt = gt;
  p.xgroups = d.rows_x / 8;
  p.dxp = make_fastdiv((uint32_t)(d.P + 2 * DW_PAD) / 2);
  p.dxy = make_fastdiv((uint32_t)g.ny + 2);
  p.dgp = make_fastdiv((uint32_t)d.P / 2);
  p.dgy = make_fastdiv((uint32_t)g.ny);
  p.x_items = (uint32_t)(g.nz + 2) * (uint32_t)(g.ny + 2) * p.dxp.d;
  p.g_items = (uint32_t)g.nz * (uint32_t)g.ny * p.dgp.d;
  p.n = g.n();
  p.bpart = part + dw_bias_at(d, c.cout);
  p.dnb = make_fastdiv(nblk(p.x_items > p.g_items ? p.x_items : p.g_items));
  const unsigned tb = BG_BLOCKS + p.dnb.d * (unsigned)(p.xgroups + c.cout / 8);
  const unsigned nb = (unsigned)(3 * (d.rows_x / 16) * d.S);
  if (c.cout == 16) {
    k_to_t<16><<<tb, 256, 0, s>>>(p);
    launch_dw<16>(nb, g, d, gt, xt, part, s);
  } else if (c.cout == 32) {
    k_to_t<32><<<tb, 256, 0, s>>>(p);
    launch_dw<32>(nb, g, d, gt, xt, part, s);
  } else {
    k_to_t<64><<<tb, 256, 0, s>>>(p);
    launch_dw<64>(nb, g, d, gt, xt, part, s);
  }
  DwSums::Entry &e = sums.e[sums.n++];
  e = {part, p.bpart, dW, db, c.cout, c.cin(), d.rows_x, d.S, sums.blocks};
  sums.blocks += (uint32_t)nblk((uint64_t)c.cout * c.cin() * 27) + 1;
}
void launch_conv_dw(const G3 &g, const ConvSpec &c, const bf16 *a, const G3 &ga, const bf16 *b, const bf16 *gpre,
                    bf16 *xt, bf16 *gt, float *part, float *dW, float *db, DwSums &sums, hipStream_t s) {
  launch_dw_layer(g, c, a, ga, b, gpre, xt, gt, part, dW, db, sums, s);
}
void launch_conv_in_dw(const G3 &g, const bf16 *x0, const bf16 *gpre, bf16 *xt, bf16 *gt, float *part, float *dW,
                       float *db, DwSums &sums, hipStream_t s) {
  launch_dw_layer(g, ConvSpec{0, 2, 16}, nullptr, g, x0, gpre, xt, gt, part, dW, db, sums, s);
}

// ------------------------------------------------------------ solver transforms
__global__ __launch_bounds__(256) void k_net_input64(uint32_t n, const double *__restrict__ r,
                                                     const uint8_t *__restrict__ f, double inv, bf16 *__restrict__ x0) {
  const uint32_t v = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
  if (v >= n) return;
  const bool fluid = f[v] != 1;
  x0[2 * (size_t)v] = tobf(fluid ? (float)(r[v] * inv) : 0.0f);
  x0[2 * (size_t)v + 1] = tobf(fluid ? 1.0f : 0.0f);
}
void launch_net_input64(const G3 &g, const double *r, const uint8_t *flags, double inv, bf16 *x0, hipStream_t s) {
  k_net_input64<<<nblk(g.n()), 256, 0, s>>>(g.n(), r, flags, inv, x0);
}
__global__ __launch_bounds__(256) void k_net_output64(uint32_t n, const float *__restrict__ y,
                                                      const uint8_t *__restrict__ f, double scale,
                                                      double *__restrict__ z) {
  const uint32_t v = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
  if (v >= n) return;
  z[v] = f[v] != 1 ? (double)y[v] * scale : 0.0;
}
void launch_net_output64(const G3 &g, const float *y, const uint8_t *flags, double scale, double *z, hipStream_t s) {
  k_net_output64<<<nblk(g.n()), 256, 0, s>>>(g.n(), y, flags, scale, z);
}

// training target of a solved pair: t[v] = fluid ? phi[v] * factor : 0
__global__ __launch_bounds__(256) void k_net_target64(uint32_t n, const double *__restrict__ phi,
                                                      const uint8_t *__restrict__ f, double factor,
                                                      float *__restrict__ t) {
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  if (v >= n) return;
  t[v] = f[v] != 1 ? (float)(phi[v] * factor) : 0.0f;
}
void launch_net_target64(const G3 &g, const double *phi, const uint8_t *flags, double factor, float *t,
                         hipStream_t s) {
  k_net_target64<<<nblk(g.n()), 256, 0, s>>>(g.n(), phi, flags, factor, t);
}
// host data: x0 (2 floats per voxel) -> bf16
__global__ __launch_bounds__(256) void k_f32_to_bf16(uint32_t n, const float *__restrict__ a, bf16 *__restrict__ b) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) b[i] = tobf(a[i]);
}
__global__ __launch_bounds__(256) void k_bf16_to_f32(uint32_t n, const bf16 *__restrict__ a, float *__restrict__ b) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) b[i] = bf(a[i]);
}
void launch_f32_to_bf16(uint32_t n, const float *a, bf16 *b, hipStream_t s) { k_f32_to_bf16<<<nblk(n), 256, 0, s>>>(n, a, b); }
void launch_bf16_to_f32(uint32_t n, const bf16 *a, float *b, hipStream_t s) { k_bf16_to_f32<<<nblk(n), 256, 0, s>>>(n, a, b); }

// ------------------------------------------------------------ loss, Adam
__global__ __launch_bounds__(256) void k_loss(uint32_t n, const float *__restrict__ y, const float *__restrict__ t,
                                              const bf16 *__restrict__ x0, double *__restrict__ part) {
  double e2 = 0.0, t2 = 0.0;
  for (uint32_t v = blockIdx.x * 256u + threadIdx.x; v < n; v += LOSS_BLOCKS * 256u) {
    if (bf(x0[2 * (size_t)v + 1]) > 0.5f) {
      const double d = (double)y[v] - (double)t[v];
      e2 += d * d;
      t2 += (double)t[v] * (double)t[v];
    }
  }
  __shared__ double sh[256 / 64];
  const double a = block_sum<256>(e2, sh);
  const double b = block_sum<256>(t2, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = a;
    part[LOSS_BLOCKS + blockIdx.x] = b;
  }
}
__global__ __launch_bounds__(256) void k_loss_final(double *__restrict__ part, float *__restrict__ rec) {
  // part[2*NB], part[2*NB+1] = totals (fixed order); rec (if not null) their ratio
  __shared__ double sh[256 / 64];
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < LOSS_BLOCKS; i += 256) {
    a += part[i];
    b += part[LOSS_BLOCKS + i];
  }
  a = block_sum<256>(a, sh);
  b = block_sum<256>(b, sh);
  if (threadIdx.x == 0) {
    part[2 * LOSS_BLOCKS] = a;
    part[2 * LOSS_BLOCKS + 1] = b;
    if (rec) rec[0] = (float)(b > 0.0 ? a / b : a);
  }
}
void launch_loss(const G3 &g, const float *y, const float *t, const bf16 *x0, double *part, float *rec,
                 hipStream_t s) {
  k_loss<<<LOSS_BLOCKS, 256, 0, s>>>(g.n(), y, t, x0, part);
  k_loss_final<<<1, 256, 0, s>>>(part, rec);
}
__global__ __launch_bounds__(256) void k_loss_grad(uint32_t n, const float *__restrict__ y, const float *__restrict__ t,
                                                   const bf16 *__restrict__ x0, const double *__restrict__ den,
                                                   float *__restrict__ gy) {
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  if (v >= n) return;
  const double d = den[0] > 0.0 ? den[0] : 1.0;
  gy[v] = bf(x0[2 * (size_t)v + 1]) > 0.5f ? (float)(2.0 * ((double)y[v] - (double)t[v]) / d) : 0.0f;
}
void launch_loss_grad(const G3 &g, const float *y, const float *t, const bf16 *x0, const double *den, float *gy,
                      hipStream_t s) {
  k_loss_grad<<<nblk(g.n()), 256, 0, s>>>(g.n(), y, t, x0, den, gy);
}

__global__ __launch_bounds__(256) void k_adam(uint32_t n, float *__restrict__ p, const float *__restrict__ gr,
                                              float *__restrict__ m, float *__restrict__ v, float lr, float b1,
                                              float b2, float eps, float c1, float c2, float gscale) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float g = gr[i] * gscale;
  const float mi = b1 * m[i] + (1.0f - b1) * g;
  const float vi = b2 * v[i] + (1.0f - b2) * (g * g);
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
void launch_adam(uint32_t n, float *p, const float *gr, float *m, float *v, float lr, float b1, float b2, float eps,
                 float c1, float c2, float gscale, hipStream_t s) {
  k_adam<<<nblk(n), 256, 0, s>>>(n, p, gr, m, v, lr, b1, b2, eps, c1, c2, gscale);
}

}  // namespace pyro
