// k_mg.hip -- geometric multigrid pressure solve on gfx950.
//
// Reference: mg.wgsl mg_smooth (:5-36), mg_restrict (:38-83), mg_prolong
// (:85-120), mg_resid (:122-158); V-cycle schedule sim.rs:451-491.
// Operator: (sum of fluid neighbours - cnt*phi)/h^2; ground (y<0) Neumann,
// side/top neighbours outside the box count with phi = 0, solid neighbours
// are skipped (Neumann).
//
// The reference dispatches the coarsest level's 80 red-black SOR iterations
// as 160 separate passes; here they run in one workgroup with phi, b and the
// solid mask on chip (160 KB of LDS per CU on gfx950), one barrier per colour
// pass, or, where a level is too large for that, as sweep launches: 40 of two
// sweeps each, or 80 single ones where two do not pay (sweep2_fits).
#include "kernels.hpp"

namespace pyro {

// Neighbour sum and count of cell (x,y,z) (mg.wgsl:25-33 / :56-64): fluid
// neighbours add phi and count 1, neighbours outside the box on a side or the
// top count wdir (1 in mg.wgsl), the ground and solids are skipped.  The
// count is formed as fluid + wdir * outside, which for wdir = 1 is the same
// small integer as the reference's running sum of 1.0.
__device__ __forceinline__ void nsum(const int d0, const int d1, const int d2, const float *__restrict__ p,
                                     const uint8_t *__restrict__ f, int x, int y, int z, uint32_t i, float wdir,
                                     float &sum, float &cnt) {
  const uint32_t sy = (uint32_t)d0, sz = (uint32_t)d0 * (uint32_t)d1;
  sum = 0.0f;
  int fl = 0, out = 0;
  if (x + 1 < d0) { if (f[i + 1] != 1) { sum += p[i + 1]; fl++; } } else out++;
  if (x - 1 >= 0) { if (f[i - 1] != 1) { sum += p[i - 1]; fl++; } } else out++;
  if (y + 1 < d1) { if (f[i + sy] != 1) { sum += p[i + sy]; fl++; } } else out++;
  if (y - 1 >= 0) { if (f[i - sy] != 1) { sum += p[i - sy]; fl++; } }  // ground: skipped
  if (z + 1 < d2) { if (f[i + sz] != 1) { sum += p[i + sz]; fl++; } } else out++;
  if (z - 1 >= 0) { if (f[i - sz] != 1) { sum += p[i - sz]; fl++; } } else out++;
  cnt = (float)fl + wdir * (float)out;
}

struct LvArgs {
  int d0, d1, d2;
  uint32_t n;
  float hh;
  float wdir;        // weight of a neighbour outside the box (1 = mg.wgsl)
  FastDiv dhx, dny;  // ceil(d0/2), d1
  uint32_t nhalf;    // ceil(d0/2)*d1*d2
};
static LvArgs lv_args(const MgLevel &L) {
  LvArgs a;
  a.d0 = L.d[0]; a.d1 = L.d[1]; a.d2 = L.d[2];
  a.n = L.n;
  a.hh = L.hh;
  a.wdir = L.wdir;
  uint32_t hx = (uint32_t)(L.d[0] + 1) / 2;
  a.dhx = make_fastdiv(hx);
  a.dny = make_fastdiv((uint32_t)L.d[1]);
  a.nhalf = hx * (uint32_t)L.d[1] * (uint32_t)L.d[2];
  return a;
}

// Fine residual at (x,y,z) (mg.wgsl:52-66).
__device__ __forceinline__ float resid_at(const LvArgs &F, const float *__restrict__ p, const float *__restrict__ b,
                                          const uint8_t *__restrict__ f, int x, int y, int z) {
  uint32_t i = (uint32_t)x + (uint32_t)F.d0 * ((uint32_t)y + (uint32_t)F.d1 * (uint32_t)z);
  if (f[i] == 1) return 0.0f;
  float pcen = p[i];
  float sum, cnt;
  nsum(F.d0, F.d1, F.d2, p, f, x, y, z, i, F.wdir, sum, cnt);
  return b[i] - (sum - cnt * pcen) / F.hh;
}

// Neighbour codes (setup pass below): bit 7 solid, bit 6 no counted
// neighbour, bits 0-2 fluid neighbours, bits 3-5 neighbours outside the box.
constexpr uint8_t NC_SOLID = 0x80, NC_NONE = 0x40;
__device__ __forceinline__ float nc_count(uint32_t code, float wdir) {
  return (float)(code & 7u) + wdir * (float)((code >> 3) & 7u);
}

// x / c for an integer count c in 1..6 given r = RN(1/c) and x != -0:
// q0 = x r, the remainder e = x - c q0 (exact through the FMA), q = q0 + e r
// (Markstein's correction).  Checked exhaustively over every finite float
// x != -0 for each c: q equals the IEEE quotient whenever q is not subnormal
// (the only mismatches are c = 6 with 0 < |x| < 2^-125), and a subnormal q
// takes the IEEE division.  In the sweep, x = (neighbour sum from +0) - h^2 b
// is never -0: a sum that starts at +0 never becomes -0, and s - t is -0
// only for s = -0.  For x = -0 the result is +0 (IEEE: -0), and with c = r =
// 0 it is +-0; the coarse solve uses q only in phi + (q - phi) omega, which
// is the same for q = +0 and q = -0 (+0 for phi = +-0, else q - phi = -phi).
__device__ __forceinline__ float div_count(float x, float c, float r) {
  const float q0 = x * r;
  const float e = __builtin_fmaf(-q0, c, x);
  float q = __builtin_fmaf(e, r, q0);
  if (__builtin_amdgcn_classf(q, 0x90)) {  // -subnormal | +subnormal
    float xs = x;
    asm volatile("" : "+v"(xs));  // a branch, not a select: the division runs only for these x
    q = xs / c;
  }
  return q;
}

// The same without the division: a subnormal quotient is noted in `redo`.
__device__ __forceinline__ float quot_count(float x, float c, float r, bool &redo) {
  const float q0 = x * r;
  const float e = __builtin_fmaf(-q0, c, x);
  const float q = __builtin_fmaf(e, r, q0);
  redo |= __builtin_amdgcn_classf(q, 0x90);  // -subnormal | +subnormal
  return q;
}

// The four elements from `over` on (0 beyond the fourth).
__device__ __forceinline__ float4 shift4(float4 v, int over) {
  if (over == 1) return make_float4(v.y, v.z, v.w, 0.0f);
  if (over == 2) return make_float4(v.z, v.w, 0.0f, 0.0f);
  if (over == 3) return make_float4(v.w, 0.0f, 0.0f, 0.0f);
  return v;
}

// Residual + average over fluid children, coarse phi = 0 (mg.wgsl:67-81).
// The coarse flags (mg.wgsl:82) are produced once per step by the setup pass.
// A block takes 16 x 4 x 4 coarse cells (one per thread); the fine φ and
// neighbour codes of their children plus a ring of 1 are staged in LDS, φ
// zeroed on solid and outside cells, so each child's neighbour sum adds the
// six LDS values in the order of nsum (x+1, x-1, y+1, y-1, z+1, z-1): a
// skipped neighbour contributes +0.0, which never changes the running sum.
constexpr int RS_TX = 16, RS_TY = 4, RS_TZ = 4;
constexpr int RS_FX = 2 * RS_TX + 2, RS_FY = 2 * RS_TY + 2, RS_FZ = 2 * RS_TZ + 2;
constexpr int RS_FN = RS_FX * RS_FY * RS_FZ;
// VEC (fine x-size a multiple of 4, arrays below 2 GiB): the footprint's x
// range is widened to 16-byte alignment, [2 x0 - 4, 2 x0 + 36), and staged
// as whole float4 / uchar4 groups: thread t < 250 loads group t % 10 of the
// rows t / 10 + 25 it, it = 0..3 (a group lies entirely inside or outside
// the level; outside reads 0 and codes 0x40).  ODD (any other x-size from four
// up): the same with the last group of a row loaded from where it ends with
// the row and shifted, and codes loaded as bytes; one element at a time the
// launch took 8.4 us on the levels of a 97x61x118 grid, 5.2 now.
constexpr int RS_VX = 2 * RS_TX + 8, RS_VQ = RS_VX / 4, RS_VN = RS_VX * RS_FY * RS_FZ;
static_assert(RS_VQ * 25 == 250 && RS_FY * RS_FZ == 100, "restriction staging map");
enum { ROWS_ANY = 0, ROWS_ODD = 1, ROWS_VEC = 2 };
template <int R>
__global__ __launch_bounds__(NT) void k_mg_restrict(LvArgs F, int ntx, int nty, const float *__restrict__ pf,
                                                     const float *__restrict__ bf, const uint8_t *__restrict__ ncf,
                                                     int c0, int c1, int c2, float *__restrict__ bc,
                                                     float *__restrict__ pc) {
  constexpr bool VEC = R != ROWS_ANY;
  constexpr int FX = VEC ? RS_VX : RS_FX;
  __shared__ __align__(16) float sp[VEC ? RS_VN : RS_FN];
  __shared__ __align__(16) uint8_t sc[VEC ? RS_VN : RS_FN];
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  // footprint origin
  const int fx0 = 2 * RS_TX * tx - (VEC ? 4 : 1), fy0 = 2 * RS_TY * ty - 1, fz0 = 2 * RS_TZ * tz - 1;
  const int sy = F.d0, sz = F.d0 * F.d1;
  const int lcx = threadIdx.x % RS_TX, lr = threadIdx.x / RS_TX, lcy = lr % RS_TY, lcz = lr / RS_TY;
  const int x = RS_TX * tx + lcx, y = RS_TY * ty + lcy, z = RS_TZ * tz + lcz;
  // the eight children's h^2 b, issued with the staging loads (a child
  // outside the level, also of a coarse cell outside it, reads element 0
  // and is skipped)
  float bv[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int a = 2 * x + (k & 1), bb = 2 * y + ((k >> 1) & 1), c = 2 * z + ((k >> 2) & 1);
    const bool in = a < F.d0 && bb < F.d1 && c < F.d2;
    bv[k] = bf[in ? a + sy * bb + sz * c : 0];
  }
  if (VEC) {
    const RB rp = rb_of(pf, F.n * 4u), rcd = rb_of(ncf, F.n);
    const int t = threadIdx.x, q = t % RS_VQ, r0 = t / RS_VQ;
    const int gx = fx0 + 4 * q;
    float4 pv[4];
    uint32_t cv[4];
#pragma unroll
    for (int it = 0; it < 4; it++) {
      const int r = r0 + 25 * it, lz = r / RS_FY, ly = r - RS_FY * lz;
      const int gy = fy0 + ly, gz = fz0 + lz;
      const bool ok = t < 250 && (uint32_t)gx < (uint32_t)F.d0 && (uint32_t)gy < (uint32_t)F.d1 &&
                      (uint32_t)gz < (uint32_t)F.d2;
      const uint32_t g = (uint32_t)gx + (uint32_t)sy * (uint32_t)gy + (uint32_t)sz * (uint32_t)gz;
      const int over = R == ROWS_ODD && gx + 4 > F.d0 ? gx + 4 - F.d0 : 0;  // elements past the row's end
      pv[it] = rb_ld4(rp, ok ? 4u * (g - (uint32_t)over) : RB_OOB);
      if (R == ROWS_VEC) {
        const uint32_t c = rb_ld32(rcd, ok ? g : RB_OOB);
        cv[it] = ok ? c : 0x40404040u;
      } else {
        cv[it] = 0u;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const bool okj = ok && gx + j < F.d0;
          const uint32_t cj = __builtin_amdgcn_raw_buffer_load_b8(rcd.r, okj ? g + j : RB_OOB, 0, 0);
          cv[it] |= (okj ? cj : (uint32_t)NC_NONE) << (8 * j);
        }
      }
    }
    if (t < 250) {
#pragma unroll
      for (int it = 0; it < 4; it++) {
        float4 v = R == ROWS_ODD ? shift4(pv[it], gx + 4 - F.d0) : pv[it];
        const uint32_t c = cv[it];
        if (c & 0x80808080u) {  // solids read 0 in the neighbour sums
          if (c & 0x80u) v.x = 0.0f;
          if (c & 0x8000u) v.y = 0.0f;
          if (c & 0x800000u) v.z = 0.0f;
          if (c & 0x80000000u) v.w = 0.0f;
        }
        const int e = 4 * (q + RS_VQ * (r0 + 25 * it));
        *reinterpret_cast<float4 *>(sp + e) = v;
        *reinterpret_cast<uint32_t *>(sc + e) = c;
      }
    }
  } else {
    // every load is unconditional (outside the level at element 0) and
    // selected afterwards, so all of a thread's loads are in flight at once
#pragma unroll
    for (int q = 0; q < (RS_FN + NT - 1) / NT; q++) {
      const int s = threadIdx.x + q * NT;
      const int se = s < RS_FN ? s : RS_FN - 1;
      const int lx = se % RS_FX, r2 = se / RS_FX, ly = r2 % RS_FY, lz = r2 / RS_FY;
      const int gx = fx0 + lx, gy = fy0 + ly, gz = fz0 + lz;
      const bool in = gx >= 0 && gx < F.d0 && gy >= 0 && gy < F.d1 && gz >= 0 && gz < F.d2;
      const int g = in ? gx + sy * gy + sz * gz : 0;
      const uint8_t c = ncf[g];
      const float p = pf[g];
      if (s < RS_FN) {
        sp[s] = (in && !(c & NC_SOLID)) ? p : 0.0f;
        sc[s] = in ? c : NC_NONE;
      }
    }
  }
  __syncthreads();
  if (x >= c0 || y >= c1 || z >= c2) return;
  float acc = 0.0f, nfl = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int a = 2 * x + (k & 1), bb = 2 * y + ((k >> 1) & 1), c = 2 * z + ((k >> 2) & 1);
    if (a >= F.d0 || bb >= F.d1 || c >= F.d2) continue;
    const int pi = ((c - fz0) * RS_FY + (bb - fy0)) * FX + (a - fx0);
    const uint8_t code = sc[pi];
    if (code & NC_SOLID) continue;
    nfl += 1.0f;
    float sum = 0.0f;
    sum += sp[pi + 1];
    sum += sp[pi - 1];
    sum += sp[pi + FX];
    sum += sp[pi - FX];
    sum += sp[pi + FX * RS_FY];
    sum += sp[pi - FX * RS_FY];
    const float cnt = nc_count(code, F.wdir);
    acc += bv[k] - (sum - cnt * sp[pi]) / F.hh;
  }
  const uint32_t i = (uint32_t)x + (uint32_t)c0 * ((uint32_t)y + (uint32_t)c1 * (uint32_t)z);
  bc[i] = nfl > 0.0f ? acc / fmax_(nfl, 1.0f) : 0.0f;
  pc[i] = 0.0f;
}
void launch_mg_restrict(const MgLevel &Fl, const MgLevel &C, hipStream_t s) {
  LvArgs F = lv_args(Fl);
  const int ntx = (C.d[0] + RS_TX - 1) / RS_TX, nty = (C.d[1] + RS_TY - 1) / RS_TY, ntz = (C.d[2] + RS_TZ - 1) / RS_TZ;
  const bool buf = (uint64_t)Fl.n * 4u < (1ull << 31);
#define PYRO_RESTRICT(R_)                                                                                       \
  k_mg_restrict<R_><<<ntx * nty * ntz, NT, 0, s>>>(F, ntx, nty, Fl.phi, Fl.b, Fl.nc, C.d[0], C.d[1], C.d[2], C.b, \
                                                   C.phi)
  if (buf && Fl.d[0] % 4 == 0) PYRO_RESTRICT(ROWS_VEC);
  else if (buf && Fl.d[0] > 4) PYRO_RESTRICT(ROWS_ODD);
  else PYRO_RESTRICT(ROWS_ANY);
#undef PYRO_RESTRICT
}

// Masked, renormalised trilinear correction (mg.wgsl:97-120).  A block takes
// 32 x 8 x 4 fine cells (4 per thread along y); the coarse φ and flags they
// interpolate from (18 x 6 x 4 cells, with the clamping of mg.wgsl applied
// while staging) sit in LDS.  Weights and the order of the sums are those of
// the per-cell formula.
constexpr int PL_TX = 32, PL_TY = 8, PL_TZ = 4;
constexpr int PL_CX = PL_TX / 2 + 2, PL_CY = PL_TY / 2 + 2, PL_CZ = PL_TZ / 2 + 2;
constexpr int PL_CN = PL_CX * PL_CY * PL_CZ;
__global__ __launch_bounds__(NT) void k_mg_prolong(int f0, int f1, int f2, int ntx, int nty,
                                                    const uint8_t *__restrict__ ff, float *__restrict__ pf, int c0,
                                                    int c1, int c2, const float *__restrict__ pc,
                                                    const uint8_t *__restrict__ fc) {
  __shared__ float sp[PL_CN];
  __shared__ uint8_t sf[PL_CN];
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0 = PL_TX * tx, y0 = PL_TY * ty, z0 = PL_TZ * tz;
  const int cx0 = x0 / 2 - 1, cy0 = y0 / 2 - 1, cz0 = z0 / 2 - 1;  // coarse footprint origin (unclamped)
  // a thread's cells: x = x0 + lx, y = y0 + ly, z = z0 + q for q < PL_TZ
  static_assert(NT / PL_TX == PL_TY && PL_TZ % 2 == 0, "one (x, y) column of PL_TZ cells per thread");
  constexpr int NQ = PL_TZ;
  const int lx = threadIdx.x % PL_TX, ly = threadIdx.x / PL_TX;
  const int x = x0 + lx, y = y0 + ly;
  // the thread's cells' flags and phi, issued with the staging loads (a
  // cell outside the level reads element 0 and is skipped)
  uint8_t fv[NQ];
  float pv[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int z = z0 + q;
    const uint32_t i =
        (x < f0 && y < f1 && z < f2) ? (uint32_t)x + (uint32_t)f0 * ((uint32_t)y + (uint32_t)f1 * (uint32_t)z) : 0u;
    fv[q] = ff[i];
    pv[q] = pf[i];
  }
  bool solid = false;
  for (int s = threadIdx.x; s < PL_CN; s += NT) {
    const int u = s % PL_CX, r2 = s / PL_CX, v = r2 % PL_CY, w = r2 / PL_CY;
    const int cx = clampi(cx0 + u, 0, c0 - 1), cy = clampi(cy0 + v, 0, c1 - 1), cz = clampi(cz0 + w, 0, c2 - 1);
    const uint32_t j = (uint32_t)cx + (uint32_t)c0 * ((uint32_t)cy + (uint32_t)c1 * (uint32_t)cz);
    sp[s] = pc[j];
    const uint8_t fl = fc[j];
    sf[s] = fl;
    solid |= fl == 1;
  }
  // whether any coarse cell of the footprint is solid (block-uniform)
  solid = __syncthreads_or(solid);
  if (x >= f0 || y >= f1) return;
  // A fine index's fraction is 0.75 (even) or 0.25 (odd), exactly, so the
  // weights are exact: wx wy is formed once per thread, and z = z0 + q (z0 a
  // multiple of 4) has the parity of q, so frz is a constant; the product
  // keeps the per-cell formula's order, (wx wy) wz.
  const float px = ((float)x + 0.5f) * 0.5f - 0.5f, py = ((float)y + 0.5f) * 0.5f - 0.5f;
  const int i0x = (int)floorf(px), i0y = (int)floorf(py);
  const float frx = px - (float)i0x, fry = py - (float)i0y;
  float wxy[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float wx = (k & 1) ? frx : 1.0f - frx, wy = (k >> 1) ? fry : 1.0f - fry;
    wxy[k] = wx * wy;
  }
  const int sxy = (i0y - cy0) * PL_CX + (i0x - cx0);
  if (!solid) {
    // No solid corner anywhere in the block: every weight is the plain
    // product and they sum to exactly 1 (multiples of 1/64 below 2, added
    // exactly), so the correction is acc itself; acc is formed with the
    // weights and in the order of the general loop below.
    float w8[2][8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      w8[0][k] = wxy[k & 3] * ((k >> 2) ? 0.75f : 1.0f - 0.75f);
      w8[1][k] = wxy[k & 3] * ((k >> 2) ? 0.25f : 1.0f - 0.25f);
    }
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const int z = z0 + q;
      if (z >= f2 || fv[q] == 1) continue;
      const uint32_t i = (uint32_t)x + (uint32_t)f0 * ((uint32_t)y + (uint32_t)f1 * (uint32_t)z);
      const int i0z = (int)floorf(((float)z + 0.5f) * 0.5f - 0.5f);
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int ox = k & 1, oy = (k >> 1) & 1, oz = (k >> 2) & 1;
        const int si = (i0z + oz - cz0) * (PL_CY * PL_CX) + sxy + oy * PL_CX + ox;
        acc += w8[q & 1][k] * sp[si];
      }
      pf[i] = pv[q] + acc;
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int z = z0 + q;
    if (z >= f2) continue;
    const uint32_t i = (uint32_t)x + (uint32_t)f0 * ((uint32_t)y + (uint32_t)f1 * (uint32_t)z);
    if (fv[q] == 1) continue;
    const float pz = ((float)z + 0.5f) * 0.5f - 0.5f;
    const int i0z = (int)floorf(pz);
    const float frz = (q & 1) ? 0.25f : 0.75f;  // = pz - i0z
    // a solid corner adds weight 0 (its coarse phi is 0, never updated):
    // +-0 added to these sums, which start at +0 and are never -0, leaves
    // them unchanged, so this is the per-cell loop that skips solid corners
    float acc = 0.0f, ws = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int ox = k & 1, oy = (k >> 1) & 1, oz = (k >> 2) & 1;
      const int si = (i0z + oz - cz0) * (PL_CY * PL_CX) + sxy + oy * PL_CX + ox;
      const float wgt = sf[si] == 1 ? 0.0f : wxy[k & 3] * (oz == 1 ? frz : 1.0f - frz);
      acc += wgt * sp[si];
      ws += wgt;
    }
    // with no solid corner the weights sum to exactly 1 and acc / 1 = acc:
    // the division runs (a branch, not a select) only for the other cells
    float corr = acc;
    if (ws != 1.0f) {
      float a = acc;
      asm volatile("" : "+v"(a));
      corr = a / ws;
    }
    if (ws > 1e-4f) pf[i] = pv[q] + corr;
  }
}
void launch_mg_prolong(const MgLevel &C, const MgLevel &F, hipStream_t s) {
  const int ntx = (F.d[0] + PL_TX - 1) / PL_TX, nty = (F.d[1] + PL_TY - 1) / PL_TY, ntz = (F.d[2] + PL_TZ - 1) / PL_TZ;
  k_mg_prolong<<<ntx * nty * ntz, NT, 0, s>>>(F.d[0], F.d[1], F.d[2], ntx, nty, F.f, F.phi, C.d[0], C.d[1], C.d[2],
                                              C.phi, C.f);
}

// ---------------------------------------------------------------- setup
// Per-level neighbour codes, computed once per step (flags are fixed during
// a step and restriction derives the same coarse flags in every cycle):
//   bit 7: solid (never updated, phi is Neumann for its neighbours)
//   bit 6: fluid cell without a counted neighbour (mg.wgsl:34 skips it)
//   bits 0-2: fluid neighbours; bits 3-5: neighbours outside the box on a side
//   or the top.  cnt of mg.wgsl:25-33 = fluid + wdir * outside; with
//   wdir = 1 it is the same small integer, exactly.

// All levels go in one launch, and the coarse flags of three levels in another:
// a launch a level and kind took 4 to 5 us each, seven of them in every step.
// The levels' blocks follow one another; the table is indexed where it lies,
// in the kernel arguments (a copy would be indexed in scratch memory).
typedef const __attribute__((address_space(1))) uint8_t *gcu8;
typedef __attribute__((address_space(1))) uint8_t *gu8;
struct SetupLevel {
  int d0, d1, d2;
  uint32_t n, block0;  // cells, first block
  FastDiv q0, q1;      // d0, d1
  gu8 f, nc, nm;
};
struct SetupArgs {
  int nl, first;  // levels, first level written (coarse flags)
  SetupLevel l[MG_MAX];
};

// The codes of a cell, or of four cells along x at once.
__device__ __forceinline__ void counts_cell(const SetupLevel &a, uint32_t i) {
  gcu8 f = a.f;
  const gu8 nc = a.nc, nm = a.nm;
  uint32_t r = fdiv(i, a.q0);
  int x = (int)(i - r * (uint32_t)a.d0);
  uint32_t zq = fdiv(r, a.q1);
  int y = (int)(r - zq * (uint32_t)a.d1), z = (int)zq;
  const uint32_t sy = (uint32_t)a.d0, sz = (uint32_t)a.d0 * (uint32_t)a.d1;
  const bool hxp = x + 1 < a.d0, hxm = x > 0, hyp = y + 1 < a.d1, hym = y > 0, hzp = z + 1 < a.d2, hzm = z > 0;
  // the cell's and its six neighbours' flags are loaded together (a
  // neighbour outside the level reads the cell itself and is not used)
  const uint8_t fc = f[i];
  const uint8_t fxp = f[hxp ? i + 1 : i], fxm = f[hxm ? i - 1 : i];
  const uint8_t fyp = f[hyp ? i + sy : i], fym = f[hym ? i - sy : i];
  const uint8_t fzp = f[hzp ? i + sz : i], fzm = f[hzm ? i - sz : i];
  if (fc == 1) {
    nc[i] = NC_SOLID;
    if (nm) nm[i] = 0;
    return;
  }
  const uint32_t m = (hxp && fxp != 1 ? 1u : 0u) | (hxm && fxm != 1 ? 2u : 0u) | (hyp && fyp != 1 ? 4u : 0u) |
                     (hym && fym != 1 ? 8u : 0u) | (hzp && fzp != 1 ? 16u : 0u) | (hzm && fzm != 1 ? 32u : 0u);
  // neighbours outside the box on a side or the top; the ground (y - 1) is not counted
  const int out = (hxp ? 0 : 1) + (hxm ? 0 : 1) + (hyp ? 0 : 1) + (hzp ? 0 : 1) + (hzm ? 0 : 1);
  const int fl = __builtin_popcount(m);
  nc[i] = (fl + out) == 0 ? NC_NONE : (uint8_t)(fl | (out << 3));
  if (nm) nm[i] = (uint8_t)m;
}

// The same codes four cells at a time along x (level x-size a multiple of
// 4): a thread reads the flag words of its cells and of their y and z
// neighbours and the two bytes beside them in x, and writes one code word.
__device__ __forceinline__ uint32_t byte_of(uint32_t w, int j) { return (w >> (8 * j)) & 0xffu; }
__device__ __forceinline__ void counts_cells4(const SetupLevel &a, uint32_t w) {  // w: word index
  typedef const __attribute__((address_space(1))) uint32_t *gcu32;
  typedef __attribute__((address_space(1))) uint32_t *gu32;
  gcu8 f = a.f;
  const uint32_t i = 4u * w;
  uint32_t r = fdiv(i, a.q0);
  const int x0 = (int)(i - r * (uint32_t)a.d0);
  uint32_t zq = fdiv(r, a.q1);
  const int y = (int)(r - zq * (uint32_t)a.d1), z = (int)zq;
  const uint32_t sy = (uint32_t)a.d0, sz = (uint32_t)a.d0 * (uint32_t)a.d1;
  const bool hyp = y + 1 < a.d1, hym = y > 0, hzp = z + 1 < a.d2, hzm = z > 0;
  const bool hx0 = x0 > 0, hx3 = x0 + 4 < a.d0;
  gcu32 f4 = (gcu32)f;
  // a neighbour outside the level reads the cell's own word or byte and is not used
  const uint32_t C = f4[w];
  const uint32_t YP = f4[hyp ? w + sy / 4u : w], YM = f4[hym ? w - sy / 4u : w];
  const uint32_t ZP = f4[hzp ? w + sz / 4u : w], ZM = f4[hzm ? w - sz / 4u : w];
  const uint32_t XM = f[hx0 ? i - 1u : i], XP = f[hx3 ? i + 4u : i];
  uint32_t codes = 0u, masks = 0u;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int x = x0 + j;
    const bool hxp = x + 1 < a.d0, hxm = x > 0;
    const uint32_t fc = byte_of(C, j);
    const uint32_t fxp = j < 3 ? byte_of(C, j + 1) : XP, fxm = j > 0 ? byte_of(C, j - 1) : XM;
    uint32_t code, m = 0u;
    if (fc == 1u) {
      code = NC_SOLID;
    } else {
      m = (hxp && fxp != 1u ? 1u : 0u) | (hxm && fxm != 1u ? 2u : 0u) | (hyp && byte_of(YP, j) != 1u ? 4u : 0u) |
          (hym && byte_of(YM, j) != 1u ? 8u : 0u) | (hzp && byte_of(ZP, j) != 1u ? 16u : 0u) |
          (hzm && byte_of(ZM, j) != 1u ? 32u : 0u);
      // neighbours outside the box on a side or the top; the ground (y - 1) is not counted
      const int out = (hxp ? 0 : 1) + (hxm ? 0 : 1) + (hyp ? 0 : 1) + (hzp ? 0 : 1) + (hzm ? 0 : 1);
      const int fl = __builtin_popcount(m);
      code = (fl + out) == 0 ? NC_NONE : (uint32_t)(fl | (out << 3));
    }
    codes |= code << (8 * j);
    masks |= m << (8 * j);
  }
  ((gu32)a.nc)[w] = codes;
  if (a.nm) ((gu32)a.nm)[w] = masks;
}

__global__ __launch_bounds__(NT) void k_mg_counts(SetupArgs) {
  const SetupArgs &a = *(const SetupArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t blk = (uint32_t)xcd_tile(blockIdx.x, gridDim.x);
  int l = 0;
  while (l + 1 < a.nl && blk >= a.l[l + 1].block0) l++;
  const SetupLevel &L = a.l[l];
  const uint32_t i = (blk - L.block0) * NT + threadIdx.x;
  if (L.d0 % 4 == 0) {
    if (i < L.n / 4u) counts_cells4(L, i);
  } else if (i < L.n) {
    counts_cell(L, i);
  }
}

// Coarse cell is solid iff every child inside the fine box is solid
// (mg.wgsl:74-82), so iff every cell of a finer level is that lies in it.  A
// thread takes a cell of the level K above the one read, a plane of its 8^K
// cells at a time (one beyond the box is read as the last inside it), and
// stops at the first plane that is not solid: nearly always the first.
template <int K>
__device__ __forceinline__ uint8_t all_solid(const SetupLevel &F, int x, int y, int z) {
  constexpr int S = 1 << K;
  for (int zz = 0; zz < S; zz++) {
    const int c = (z << K) + zz;
    if (c >= F.d2) break;
    bool solid = true;
#pragma unroll
    for (int k = 0; k < S * S; k++) {
      const int a = min((x << K) + k % S, F.d0 - 1), b = min((y << K) + k / S, F.d1 - 1);
      solid &= F.f[(uint32_t)a + (uint32_t)F.d0 * ((uint32_t)b + (uint32_t)F.d1 * (uint32_t)c)] == 1;
    }
    if (!solid) return 0;
  }
  return 1;
}
__global__ __launch_bounds__(NT) void k_mg_coarse_flags(SetupArgs) {
  const SetupArgs &a = *(const SetupArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t blk = blockIdx.x;
  int l = a.first;
  while (l + 1 < a.nl && blk >= a.l[l + 1].block0) l++;
  const SetupLevel &C = a.l[l], &F = a.l[a.first - 1];
  const uint32_t i = (blk - C.block0) * NT + threadIdx.x;
  if (i >= C.n) return;
  const uint32_t r = fdiv(i, C.q0), zq = fdiv(r, C.q1);
  const int x = (int)(i - r * (uint32_t)C.d0), y = (int)(r - zq * (uint32_t)C.d1), z = (int)zq;
  const int k = l - a.first + 1;
  C.f[i] = k == 1 ? all_solid<1>(F, x, y, z) : k == 2 ? all_solid<2>(F, x, y, z) : all_solid<3>(F, x, y, z);
}

void launch_mg_setup(const MgLevel *L, int nl, hipStream_t s) {
  SetupArgs a = {};
  a.nl = nl;
  for (int l = 0; l < nl; l++) {
    SetupLevel &S = a.l[l];
    S.d0 = L[l].d[0]; S.d1 = L[l].d[1]; S.d2 = L[l].d[2];
    S.n = L[l].n;
    S.q0 = make_fastdiv((uint32_t)L[l].d[0]);
    S.q1 = make_fastdiv((uint32_t)L[l].d[1]);
    S.f = (gu8)L[l].f; S.nc = (gu8)L[l].nc; S.nm = (gu8)L[l].nm;
  }
  SetupArgs c = a;
  for (int f = 1; f < nl; f += 3) {
    uint32_t blocks = 0;
    c.first = f;
    c.nl = f + 3 < nl ? f + 3 : nl;
    for (int l = f; l < c.nl; l++) {
      c.l[l].block0 = blocks;
      blocks += (uint32_t)nblocks(L[l].n);
    }
    k_mg_coarse_flags<<<blocks, NT, 0, s>>>(c);
  }
  uint32_t blocks = 0;
  for (int l = 0; l < nl; l++) {
    a.l[l].block0 = blocks;
    blocks += (uint32_t)nblocks(L[l].d[0] % 4 == 0 ? L[l].n / 4u : L[l].n);
  }
  k_mg_counts<<<blocks, NT, 0, s>>>(a);
}

// ---------------------------------------------------------------- sweep
// One full red-black sweep (colour 0 then colour 1, sim.rs:444-448) of a
// 32x8x4 tile per workgroup, staged in LDS.  The LDS footprint is x in
// [x0-4, x0+36) (16-byte aligned rows of 10 float4) by y, z with a halo of 2:
// phi and neighbour codes on the whole footprint, h^2 b on the ring-1 box.
// Colour-0 cells are updated on the tile plus a ring of 1 (the values the
// tile's colour-1 cells read), then colour-1 cells on the tile.  phi is read
// from `pin` and written to `pout` (ping-pong), so a tile never sees a
// neighbour's already-swept values.
// Solid and outside cells hold 0 in the LDS copy of phi, so the neighbour
// sum needs no mask: a skipped neighbour adds +0.0, which cannot change the
// running sum (it starts at +0.0 and never becomes -0.0).  The per-cell
// arithmetic is that of mg.wgsl:25-35, so the result equals two colour passes.
// VEC (level x-size a multiple of 4): whole float4/uchar4 rows; otherwise
// one element at a time.
constexpr int SW_TX = 32, SW_TY = 8, SW_TZ = 4, SW_NT = 256;
constexpr int SW_PX = SW_TX + 8, SW_PY = SW_TY + 4, SW_PZ = SW_TZ + 4;  // footprint
constexpr int SW_BY = SW_TY + 2, SW_BZ = SW_TZ + 2;                      // ring-1 rows for b
constexpr int SW_PN = SW_PX * SW_PY * SW_PZ;
constexpr int SW_Q = SW_PX / 4;  // float4 per footprint row

// The N cells of one colour that a thread updates in a pass (mg.wgsl:25-35
// per cell).  ICNT (outside weight 1): the count is the integer fluid +
// outside and ct[code & 63] holds (count, RN(1/count)) for div_count (code
// 0x40 / 0x80 reads (0, 0): a finite, discarded result).  The cells of a
// colour are independent (their neighbours are of the other colour, which
// the pass does not write), so all of the pass's LDS reads are issued
// first, the quotients are formed branch-free with one branch per pass for a
// subnormal quotient (div_count's IEEE fallback), and every cell is stored:
// one that is not updated (solid, or no counted neighbour) gets its own
// value back.  act[q] = false: slot q is not this thread's (no read, no
// store).
template <bool ICNT, int N>
__device__ __forceinline__ void sweep_cells(float *sp, const uint8_t *sc, const float *hb, const float2 *ct,
                                            const int *pi, const bool *act, float omega, float wdir) {
  uint32_t code[N];
  float nb[N][6], cen[N];
#pragma unroll
  for (int q = 0; q < N; q++) {
    const int p = act[q] ? pi[q] : SW_PX * SW_PY + SW_PX + 1;  // any interior entry
    code[q] = sc[p];
    nb[q][0] = sp[p + 1];
    nb[q][1] = sp[p - 1];
    nb[q][2] = sp[p + SW_PX];
    nb[q][3] = sp[p - SW_PX];
    nb[q][4] = sp[p + SW_PX * SW_PY];
    nb[q][5] = sp[p - SW_PX * SW_PY];
    cen[q] = sp[p];
  }
  float xs[N], qs[N];
  bool redo = false;
#pragma unroll
  for (int q = 0; q < N; q++) {
    // the sum starts with its first term: it then differs from +0 + ... only
    // in the sign of a zero sum (all six terms -0), and the update maps a
    // quotient of either sign of zero to the same value (cen + (q - cen) w)
    float sum = nb[q][0];
#pragma unroll
    for (int k = 1; k < 6; k++) sum += nb[q][k];
    xs[q] = sum - hb[q];
    if (ICNT) {
      const float2 cr = ct[code[q] & 63u];
      const float q0 = xs[q] * cr.y;
      const float e = __builtin_fmaf(-q0, cr.x, xs[q]);
      qs[q] = __builtin_fmaf(e, cr.y, q0);
      redo |= __builtin_amdgcn_classf(qs[q], 0x90);  // -subnormal | +subnormal
    } else {
      qs[q] = xs[q] / nc_count(code[q], wdir);
    }
  }
  if (ICNT && redo) {
#pragma unroll
    for (int q = 0; q < N; q++)
      if (__builtin_amdgcn_classf(qs[q], 0x90)) {
        float x = xs[q];
        asm volatile("" : "+v"(x));
        qs[q] = x / ct[code[q] & 63u].x;
      }
  }
#pragma unroll
  for (int q = 0; q < N; q++) {
    const float nv = mixf_(cen[q], qs[q], omega);
    if (act[q]) sp[pi[q]] = (code[q] & (NC_SOLID | NC_NONE)) ? cen[q] : nv;
  }
}

// h^2 b of the cell at grid (gx, gy, gz), read from global memory (0 outside
// the grid: the cell is then never updated).  Not staged in LDS, which
// keeps a block at 19.7 KB (8 blocks per CU).  VEC: through the buffer
// resource (arrays below 2 GiB); otherwise a bounds-checked load.
template <bool VEC>
__device__ __forceinline__ float sweep_hb(const LvArgs &a, const RB &rbb, const float *__restrict__ b, int gx, int gy,
                                          int gz) {
  const bool ok = (uint32_t)gx < (uint32_t)a.d0 && (uint32_t)gy < (uint32_t)a.d1 && (uint32_t)gz < (uint32_t)a.d2;
  if (VEC) {
    // 24-bit multiplies (full rate): d0, d1, z and the row index y + d1 z of
    // a cell inside the level are below 2^24 (launch_mg_sweep takes VEC only
    // for d1 d2 <= 2^24); the offset of a cell outside is replaced by the
    // out-of-range one
    const uint32_t g = (uint32_t)gx + __umul24((uint32_t)a.d0, (uint32_t)gy + __umul24((uint32_t)a.d1, (uint32_t)gz));
    return a.hh * __builtin_bit_cast(float, rb_ld32(rbb, ok ? 4u * g : RB_OOB));
  }
  const uint32_t g = (uint32_t)gx + (uint32_t)a.d0 * ((uint32_t)gy + (uint32_t)a.d1 * (uint32_t)gz);
  return ok ? a.hh * b[g] : 0.0f;
}

// Staging of the VEC path: thread t < 240 loads x-group q = t % 10 of
// footprint row ly = (t / 10) % 12 in planes (t / 120) + 2 it, it = 0..3
// (LDS float4 index t + 240 it).  Loads outside the grid take the
// out-of-range offset and read 0 (codes: 0x40, never updated).  The VEC path
// needs the level's arrays below 2 GiB (launch_mg_sweep checks).
constexpr int SW_PT = SW_Q * SW_PY * 2;
static_assert(SW_PZ == 8 && SW_PT <= SW_NT, "staging map");

template <bool FINE, bool VEC, bool ICNT>
__global__ __launch_bounds__(SW_NT) void k_mg_sweep(LvArgs a, int ntx, int nty, const float *__restrict__ b,
                                                     const uint8_t *__restrict__ nc, const float *__restrict__ pin,
                                                     float *__restrict__ pout, float omega) {
  __shared__ __align__(16) float sp[SW_PN];
  __shared__ __align__(16) uint8_t sc[SW_PN];
  __shared__ float2 ct[64];
  const int t = threadIdx.x;
  if (ICNT && t < 64) {
    const uint32_t cnt = (t & 7u) + ((t >> 3) & 7u);
    ct[t] = make_float2((float)cnt, cnt ? 1.0f / (float)cnt : 0.0f);
  }
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0 = tx * SW_TX - 4, y0 = ty * SW_TY - 2, z0 = tz * SW_TZ - 2;  // footprint origin, x0 % 4 == 0
  const int sy = a.d0, sz = a.d0 * a.d1;
  const RB rbb = rb_of(b, VEC ? a.n * 4u : 0u);
  if (VEC) {
    // pin null: phi is 0 (an empty resource reads 0)
    const RB rp = rb_of(pin, pin ? a.n * 4u : 0u), rcd = rb_of(nc, a.n);
    float4 pv[4];
    uint32_t cv[4];
    {
      const int q = t % SW_Q, r0 = t / SW_Q, ly = r0 % SW_PY, lz0 = r0 / SW_PY;
      const int gx = x0 + 4 * q, gy = y0 + ly;
      const bool okxy = t < SW_PT && (uint32_t)gx < (uint32_t)a.d0 && (uint32_t)gy < (uint32_t)a.d1;
      // offsets by 24-bit multiplies (the VEC bounds of sweep_hb)
#pragma unroll
      for (int it = 0; it < 4; it++) {
        const int gz = z0 + lz0 + 2 * it;
        const bool ok = okxy && (uint32_t)gz < (uint32_t)a.d2;
        const uint32_t g =
            (uint32_t)gx + __umul24((uint32_t)sy, (uint32_t)gy + __umul24((uint32_t)a.d1, (uint32_t)gz));
        pv[it] = rb_ld4(rp, ok ? 4u * g : RB_OOB);
        const uint32_t c = rb_ld32(rcd, ok ? g : RB_OOB);
        cv[it] = ok ? c : 0x40404040u;
      }
    }
    if (t < SW_PT) {
#pragma unroll
      for (int it = 0; it < 4; it++) {
        float4 v = pv[it];
        const uint32_t c = cv[it];
        if (c & 0x80808080u) {  // solids read 0 in the neighbour sums
          if (c & 0x80u) v.x = 0.0f;
          if (c & 0x8000u) v.y = 0.0f;
          if (c & 0x800000u) v.z = 0.0f;
          if (c & 0x80000000u) v.w = 0.0f;
        }
        *reinterpret_cast<float4 *>(sp + 4 * (t + SW_PT * it)) = v;
        *reinterpret_cast<uint32_t *>(sc + 4 * (t + SW_PT * it)) = c;
      }
    }
  } else {
    // every load unconditional (outside the level at element 0) and
    // selected, so a thread's loads are all in flight together
#pragma unroll
    for (int q = 0; q < (SW_PN + SW_NT - 1) / SW_NT; q++) {
      const int i = t + q * SW_NT;
      const int ie = i < SW_PN ? i : SW_PN - 1;
      const int lx = ie % SW_PX, row = ie / SW_PX, ly = row % SW_PY, lz = row / SW_PY;
      const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
      const bool in = gx >= 0 && gx < a.d0 && gy >= 0 && gy < a.d1 && gz >= 0 && gz < a.d2;
      const int g = in ? gx + sy * gy + sz * gz : 0;
      const uint8_t c = nc[g];
      const float p = pin ? pin[g] : 0.0f;
      if (i < SW_PN) {
        sp[i] = (in && !(c & NC_SOLID)) ? p : 0.0f;
        sc[i] = in ? c : NC_NONE;
      }
    }
  }
  // Colour of (gx, gy, gz) = (gx + gy + gz) & 1 with gx = x0 + lx etc.; x0 is
  // a multiple of 4, so the colour-c cell of an x-pair starting at an odd
  // lx is lx + ((K + ly + lz + c) & 1) with K = y0 + z0 + 1 (ly, lz counted
  // from the box the pass walks).
  const int K = y0 + z0 + 1;
  // h^2 b of the six cells this thread updates (maps below), loaded while
  // the tile is staged rather than inside the colour passes
  float hb0[4], hb1[2];
  {
    const int px = t % 17, r0 = t / 17;
#pragma unroll
    for (int it = 0; it < 4; it++) {
      const int r = r0 + 15 * it, lz = r / SW_BY, ly = r - SW_BY * lz;
      const int lx = 3 + 2 * px + ((K + ly + lz) & 1);
      hb0[it] = sweep_hb<VEC>(a, rbb, b, x0 + lx, y0 + 1 + ly, z0 + 1 + lz);
    }
  }
  {
    const int px = t % 16, r0 = t / 16;
#pragma unroll
    for (int it = 0; it < 2; it++) {
      const int r = r0 + 16 * it, ly = r % SW_TY, lz = r / SW_TY;
      const int lx = 4 + 2 * px + ((K + ly + lz) & 1);
      hb1[it] = sweep_hb<VEC>(a, rbb, b, x0 + lx, y0 + 2 + ly, z0 + 2 + lz);
    }
  }
  __syncthreads();
  // colour 0 on the tile + ring 1: x-pairs from lx = 3 (17 of them), rows
  // (ly, lz) of the 10 x 6 ring-1 box (LDS offset 1 in y and z); thread
  // t < 255 takes x-pair t % 17 of rows r0 + 15 it, r0 = t / 17, it = 0..3
  static_assert((SW_TX + 2) / 2 == 17 && SW_BY * SW_BZ == 60, "colour-0 map");
  {
    const int px = t % 17, r0 = t / 17;
    int pi[4];
    bool act[4];
#pragma unroll
    for (int it = 0; it < 4; it++) {
      const int r = r0 + 15 * it, lz = r / SW_BY, ly = r - SW_BY * lz;
      const int lx = 3 + 2 * px + ((K + ly + lz) & 1);
      pi[it] = (int)__umul24((uint32_t)((lz + 1) * SW_PY + (ly + 1)), (uint32_t)SW_PX) + lx;
      act[it] = t < 255;
    }
    sweep_cells<ICNT, 4>(sp, sc, hb0, ct, pi, act, omega, a.wdir);
  }
  __syncthreads();
  // colour 1 on the tile: x-pairs from lx = 4 (16), rows of the 8 x 4 tile
  // (LDS offset 2); thread t takes x-pair t % 16 of rows t / 16 and t / 16 + 16
  static_assert(SW_TX / 2 == 16 && SW_TY == 8 && SW_TZ == 4, "colour-1 map");
  {
    const int px = t % 16, r0 = t / 16;
    int pi[2];
    const bool act[2] = {true, true};
#pragma unroll
    for (int it = 0; it < 2; it++) {
      const int r = r0 + 16 * it, ly = r % SW_TY, lz = r / SW_TY;
      const int lx = 4 + 2 * px + ((K + ly + lz) & 1);
      pi[it] = (int)__umul24((uint32_t)((lz + 2) * SW_PY + (ly + 2)), (uint32_t)SW_PX) + lx;
    }
    sweep_cells<ICNT, 2>(sp, sc, hb1, ct, pi, act, omega, a.wdir);
  }
  __syncthreads();
  if (VEC) {
    constexpr int WN = (SW_TX / 4) * SW_TY * SW_TZ;
    static_assert(WN == SW_NT, "one float4 of the tile per thread");
    const int q = t % (SW_TX / 4), row = t / (SW_TX / 4), ly = row % SW_TY, lz = row / SW_TY;
    const int gx = x0 + 4 + 4 * q, gy = y0 + 2 + ly, gz = z0 + 2 + lz;
    if (gx < a.d0 && gy < a.d1 && gz < a.d2) {
      const uint32_t g = (uint32_t)gx + __umul24((uint32_t)sy, (uint32_t)gy + __umul24((uint32_t)a.d1, (uint32_t)gz));
      const int pi = ((lz + 2) * SW_PY + (ly + 2)) * SW_PX + 4 + 4 * q;
      float4 v = *reinterpret_cast<const float4 *>(sp + pi);
      const uint32_t cv = *reinterpret_cast<const uint32_t *>(sc + pi);
      if ((cv & 0x80808080u) && pin) {  // solid cells keep their phi (zeroed only in LDS)
        const float4 o = *reinterpret_cast<const float4 *>(pin + g);
        if (cv & 0x80u) v.x = o.x;
        if (cv & 0x8000u) v.y = o.y;
        if (cv & 0x800000u) v.z = o.z;
        if (cv & 0x80000000u) v.w = o.w;
      }
      *reinterpret_cast<float4 *>(pout + g) = v;
    }
  } else {
    constexpr int TN = SW_TX * SW_TY * SW_TZ;
    for (int i = t; i < TN; i += SW_NT) {
      const int lx = i % SW_TX, row = i / SW_TX, ly = row % SW_TY, lz = row / SW_TY;
      const int gx = x0 + 4 + lx, gy = y0 + 2 + ly, gz = z0 + 2 + lz;
      if (gx >= a.d0 || gy >= a.d1 || gz >= a.d2) continue;
      const int g = gx + sy * gy + sz * gz;
      const int pi = ((lz + 2) * SW_PY + (ly + 2)) * SW_PX + 4 + lx;
      pout[g] = (sc[pi] & NC_SOLID) && pin ? pin[g] : sp[pi];
    }
  }
}

// The same sweep in a walk along z, for levels of whole float4 rows: a block
// keeps a ring of twelve planes of its 40 x 12 footprint in LDS and moves four
// planes a step.  In step s wave w updates the colour-0 cells (tile and ring
// of 1) of plane 4 s + w, counted from the one below its first, and then the
// colour-1 cells of the tile in the plane below that, which have all their
// colour-0 neighbours by then; colour-1 values go straight to pout with their
// pair's colour-0 cell, since no other cell reads them in this sweep.  The
// next four planes are in registers meanwhile, loaded a whole step ahead.
// Against a tile at a time: 2.1 loads and 1.2 updates a cell instead of 3.75
// and 1.5, and the loads overlap the updates; 563 MB read from beyond the L2
// instead of 788 at 320x480x320 (443 are compulsory), and 41 M VALU
// instructions instead of 70.  Loads two steps ahead (95 registers) gave
// nothing more, chunks of 62 planes neither.  Outside weight 1.
constexpr int SZ_R = 12, SZ_PL = SW_PX * SW_PY, SZ_LEN = 30;  // ring, plane, planes a block
template <int N>
__device__ __forceinline__ void sweep_plane(const float *sp, const uint8_t *sc, const float2 *ct, int z0, int zm, int zp,
                                            const int *off, const float *hb, float omega, uint32_t *code,
                                            float *xp, float *xm, float *out) {
  float nb[N][6], cen[N];
#pragma unroll
  for (int q = 0; q < N; q++) {
    const int p = z0 + off[q];
    code[q] = sc[p];
    nb[q][0] = sp[p + 1];
    nb[q][1] = sp[p - 1];
    nb[q][2] = sp[p + SW_PX];
    nb[q][3] = sp[p - SW_PX];
    nb[q][4] = sp[zp + off[q]];
    nb[q][5] = sp[zm + off[q]];
    cen[q] = sp[p];
  }
  float xs[N], qs[N];
  bool redo = false;
#pragma unroll
  for (int q = 0; q < N; q++) {
    float sum = nb[q][0];
#pragma unroll
    for (int k = 1; k < 6; k++) sum += nb[q][k];
    xs[q] = sum - hb[q];
    xp[q] = nb[q][0];
    xm[q] = nb[q][1];
    const float2 cr = ct[code[q] & 63u];
    const float q0 = xs[q] * cr.y;
    const float e = __builtin_fmaf(-q0, cr.x, xs[q]);
    qs[q] = __builtin_fmaf(e, cr.y, q0);
    redo |= __builtin_amdgcn_classf(qs[q], 0x90);  // -subnormal | +subnormal
  }
  if (redo) {
#pragma unroll
    for (int q = 0; q < N; q++)
      if (__builtin_amdgcn_classf(qs[q], 0x90)) {
        float x = xs[q];
        asm volatile("" : "+v"(x));
        qs[q] = x / ct[code[q] & 63u].x;
      }
  }
#pragma unroll
  for (int q = 0; q < N; q++) {
    const float nv = mixf_(cen[q], qs[q], omega);
    out[q] = (code[q] & (NC_SOLID | NC_NONE)) ? cen[q] : nv;
  }
}

__global__ __launch_bounds__(SW_NT, 5) void k_mg_sweep_z(LvArgs a, int ntx, int nty,
                                                          const float *__restrict__ b, const uint8_t *__restrict__ nc,
                                                          const float *__restrict__ pin, float *__restrict__ pout,
                                                          float omega) {
  __shared__ __align__(16) float sp[SZ_R * SZ_PL];
  __shared__ __align__(16) uint8_t sc[SZ_R * SZ_PL];
  __shared__ float2 ct[64];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  if (t < 64) {
    const uint32_t cnt = (t & 7u) + ((t >> 3) & 7u);
    ct[t] = make_float2((float)cnt, cnt ? 1.0f / (float)cnt : 0.0f);
  }
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0 = tx * SW_TX - 4, y0 = ty * SW_TY - 2;
  const int zc = tz * SZ_LEN, zend = min(zc + SZ_LEN, a.d2), zr = zc - 1;  // outputs [zc, zend); zr: step 0's first plane
  const uint32_t sz = (uint32_t)a.d0 * (uint32_t)a.d1;
  const RB rp = rb_of(pin, pin ? a.n * 4u : 0u), rcd = rb_of(nc, a.n), rbb = rb_of(b, a.n * 4u);
  // staging: group k holds planes zr - 3 + 4 k .. + 3 in slots 4 (k % 3) .. + 3;
  // thread t < 240 loads float4 q of row sly in its planes half and half + 2
  const int q = t % SW_Q, sly = (t / SW_Q) % SW_PY, half = t / (SW_Q * SW_PY);
  const int sgx = x0 + 4 * q, sgy = y0 + sly;
  const bool okxy = t < SW_PT && (uint32_t)sgx < (uint32_t)a.d0 && (uint32_t)sgy < (uint32_t)a.d1;
  const uint32_t gxy = (uint32_t)sgx + (uint32_t)a.d0 * (uint32_t)sgy;
  const uint32_t zlim = (uint32_t)min(zend + 2, a.d2);  // planes from here on are not read
  float4 pv[2];
  uint32_t cv[2];
  auto load = [&](int k) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < 2; it++) {
      const uint32_t z = (uint32_t)(zr - 3 + 4 * k + half + 2 * it);
      const bool ok = okxy && z < zlim;
      const uint32_t g = gxy + sz * z;
      pv[it] = rb_ld4(rp, ok ? 4u * g : RB_OOB);
      cv[it] = rb_ld32(rcd, ok ? g : RB_OOB);
    }
  };
  // (the choice of the code for cells outside waits for the load: it is made
  // here, a step later, and not at the load)
  auto store = [&](int k, int slot) __attribute__((always_inline)) {
    if (t < SW_PT) {
#pragma unroll
      for (int it = 0; it < 2; it++) {
        float4 v = pv[it];
        const bool ok = okxy && (uint32_t)(zr - 3 + 4 * k + half + 2 * it) < zlim;
        const uint32_t c = ok ? cv[it] : 0x40404040u;
        if (c & 0x80808080u) {  // solids read 0 in the neighbour sums
          if (c & 0x80u) v.x = 0.0f;
          if (c & 0x8000u) v.y = 0.0f;
          if (c & 0x800000u) v.z = 0.0f;
          if (c & 0x80000000u) v.w = 0.0f;
        }
        const int e = (slot + half + 2 * it) * SZ_PL + sly * SW_PX + 4 * q;
        *reinterpret_cast<float4 *>(sp + e) = v;
        *reinterpret_cast<uint32_t *>(sc + e) = c;
      }
    }
  };
  // a wave's cells in its planes (the planes' parity is the same in every
  // step): colour 0, 17 x-pairs from lx = 3 in the rows 1 .. 10; colour 1, 16
  // from lx = 4 in the rows 2 .. 9
  int off0[3], off1[2];
  uint32_t vb0[3], vb1[2];  // byte offsets of b in plane 0
  bool act0[3];
#pragma unroll
  for (int it = 0; it < 3; it++) {
    const int i = lane + 64 * it, px = i % 17, ly = min(1 + i / 17, SW_PY - 2);
    const int lx = 3 + 2 * px + ((y0 + ly + zr + w + 1) & 1);  // (x0 + lx + gy + gz) even
    act0[it] = i < 170;
    off0[it] = ly * SW_PX + lx;
    const int gx = x0 + lx, gy = y0 + ly;
    const bool ok = (uint32_t)gx < (uint32_t)a.d0 && (uint32_t)gy < (uint32_t)a.d1;
    vb0[it] = ok ? 4u * ((uint32_t)gx + (uint32_t)a.d0 * (uint32_t)gy) : RB_OOB;
  }
#pragma unroll
  for (int it = 0; it < 2; it++) {
    const int px = lane % 16, ly = 2 + lane / 16 + 4 * it;
    const int lx = 4 + 2 * px + ((y0 + ly + zr - 1 + w + 1) & 1);  // (x0 + lx + gy + gz) odd
    off1[it] = ly * SW_PX + lx;
    const int gx = x0 + lx, gy = y0 + ly;
    const bool ok = (uint32_t)gx < (uint32_t)a.d0 && (uint32_t)gy < (uint32_t)a.d1;
    vb1[it] = ok ? 4u * ((uint32_t)gx + (uint32_t)a.d0 * (uint32_t)gy) : RB_OOB;
  }
  float hb0[3], hb1[2];  // of planes outside the level: not used, any plane's
  auto load_hb0 = [&](int z) __attribute__((always_inline)) {
    const int so = (int)(4u * sz * (uint32_t)min(max(z, 0), a.d2 - 1));
#pragma unroll
    for (int it = 0; it < 3; it++)
      hb0[it] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rbb.r, vb0[it], so, 0));
  };
  auto load_hb1 = [&](int z) __attribute__((always_inline)) {
    const int so = (int)(4u * sz * (uint32_t)min(max(z, 0), a.d2 - 1));
#pragma unroll
    for (int it = 0; it < 2; it++)
      hb1[it] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rbb.r, vb1[it], so, 0));
  };
  load(0);
  store(0, 0);
  load(1);
  store(1, 4);
  load(2);
  load_hb0(zr + w);
  load_hb1(zr - 1 + w);
  __syncthreads();
  const int nstep = (zend - zc + 1) / 4 + 1;
  int base = 0;  // (4 s) % 12
  for (int s = 0; s < nstep; s++) {
    auto slot = [&](int k) __attribute__((always_inline)) {
      const int i = base + k + w;
      return (i >= SZ_R ? i - SZ_R : i) * SZ_PL;
    };
    const int z = zr + 4 * s + w;
    if (z >= 0 && z < a.d2 && z <= zend) {
      uint32_t code[3];
      float h[3], xp[3], xm[3], o[3];
#pragma unroll
      for (int it = 0; it < 3; it++) h[it] = a.hh * hb0[it];
      const int z0 = slot(3);
      sweep_plane<3>(sp, sc, ct, z0, slot(2), slot(4), off0, h, omega, code, xp, xm, o);
#pragma unroll
      for (int it = 0; it < 3; it++)
        if (act0[it]) sp[z0 + off0[it]] = o[it];
    }
    load_hb0(z + 4);
    __syncthreads();
    store(s + 2, base >= 4 ? base - 4 : 8);  // slot (4 s + 8) % 12
    load(s + 3);
    const int y = z - 1;
    if (y >= zc && y < zend) {
      uint32_t code[2];
      float h[2], xp[2], xm[2], o[2];
#pragma unroll
      for (int it = 0; it < 2; it++) h[it] = a.hh * hb1[it];
      const int z0 = slot(2);
      sweep_plane<2>(sp, sc, ct, z0, slot(1), slot(3), off1, h, omega, code, xp, xm, o);
#pragma unroll
      for (int it = 0; it < 2; it++) {
        if (vb1[it] == RB_OOB) continue;
        const int odd = off1[it] & 1;  // the colour-1 cell is the pair's odd one
        const uint32_t g = vb1[it] / 4u - (uint32_t)odd + sz * (uint32_t)y;
        float lo = odd ? xm[it] : o[it], hi = odd ? o[it] : xp[it];
        if (pin) {  // solid cells keep their phi (zeroed only in LDS)
          const uint32_t other = sc[z0 + (off1[it] ^ 1)];
          if ((odd ? other : code[it]) & NC_SOLID) lo = pin[g];
          if ((odd ? code[it] : other) & NC_SOLID) hi = pin[g + 1];
        }
        *reinterpret_cast<float2 *>(pout + g) = make_float2(lo, hi);
      }
    }
    load_hb1(y + 4);
    base = base == 8 ? 0 : base + 4;
    __syncthreads();
  }
}

void launch_mg_sweep(const MgLevel &L, const float *pin, float *pout, float omega, hipStream_t s, bool fine) {
  LvArgs a = lv_args(L);
  int ntx = (L.d[0] + SW_TX - 1) / SW_TX, nty = (L.d[1] + SW_TY - 1) / SW_TY, ntz = (L.d[2] + SW_TZ - 1) / SW_TZ;
  int nb = ntx * nty * ntz;
  // VEC: whole float4 rows, buffer loads with 32-bit byte offsets below 2 GiB,
  // row indices y + d1 z below 2^24 (sweep_hb's 24-bit multiplies)
  bool vec = (L.d[0] % 4) == 0 && (uint64_t)L.n * 4u < (1ull << 31) && (uint64_t)L.d[1] * L.d[2] <= (1ull << 24);
  // The walk along z where the arrays (13 bytes a cell and sweep) leave the
  // 256 MB cache beyond the L2s: 320x480x320 248 -> 207 us a sweep,
  // 272x400x272 151 -> 134, 224x336x224 58 -> 54, 208x304x208 (13 M cells)
  // 46 -> 44; below, the tiles' shorter chain wins: 160x320x160 28 against 29,
  // 80x160x80 7.0 against 8.8.
  if (vec && L.wdir == 1.0f && L.n >= 12000000u) {
    const int nbz = ntx * nty * ((L.d[2] + SZ_LEN - 1) / SZ_LEN);
    k_mg_sweep_z<<<nbz, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
    return;
  }
  if (L.wdir == 1.0f) {
    if (fine && vec)
      k_mg_sweep<true, true, true><<<nb, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
    else if (vec)
      k_mg_sweep<false, true, true><<<nb, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
    else
      k_mg_sweep<false, false, true><<<nb, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
  } else {
    if (fine && vec)
      k_mg_sweep<true, true, false><<<nb, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
    else if (vec)
      k_mg_sweep<false, true, false><<<nb, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
    else
      k_mg_sweep<false, false, false><<<nb, SW_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega);
  }
}

// ---------------------------------------------------------------- two sweeps
// Both red-black sweeps of a smoothing step in one launch, for levels where a
// sweep is bound by its launch and its load latency and not by its bytes.  A
// block of 512 threads takes 16 x 8 x 8 cells; phi, h^2 b and the codes of the
// tile and a ring of 4 sit in LDS, and the four colour passes run on rings of
// 3, 2, 1 and 0.  The arrays are split by colour: entry k of row (y, z) of
// colour c is the cell lx = 2 k + par, par = (c + ly + lz) & 1 (tile origins are
// multiples of four), so the lanes
// of a pass touch consecutive words, and the neighbours of an entry of one
// colour are entries of the other: k and k + 1 (par = 1) or k - 1 (par = 0) of
// its row, k of the rows y +- 1 and z +- 1.  Arithmetic and order are those of
// k_mg_sweep (the two x neighbours may change places in the first addition).
constexpr int S2_NT = 512, S2_TX = 16, S2_TY = 8, S2_TZ = 8;
constexpr int S2_K = (S2_TX + 8) / 2, S2_Y = S2_TY + 8, S2_Z = S2_TZ + 8, S2_E = S2_K * S2_Y * S2_Z;

struct S2Lds {
  float p[2][S2_E], hb[2][S2_E];
  uint8_t c[2][S2_E];
  float2 ct[64];
};

// One colour pass on the tile and a ring of R.  OUT: the pass's cells are not
// stored but returned in *v (one a thread, with its entry in *e).
template <int C, int R, bool ICNT, bool OUT>
__device__ __forceinline__ void s2_pass(S2Lds &L, float omega, float wdir, float *v, int *e) {
  constexpr int KN = S2_TX / 2 + R, RY = S2_TY + 2 * R, RZ = S2_TZ + 2 * R, PER = KN * RY, ZS = S2_NT / PER;
  constexpr int N = (RZ + ZS - 1) / ZS;
  static_assert(!OUT || (N == 1 && R == 0), "one output cell a thread");
  const int t = threadIdx.x, zi = t / PER, r = t - zi * PER, yy = r / KN, kk = r - yy * KN;
  const int ly = yy + 4 - R;
  float *own = L.p[C];
  const float *oth = L.p[1 - C];
  uint32_t code[N];
  float nb[N][6], cen[N], hb[N];
  int id[N];
  bool act[N];
#pragma unroll
  for (int q = 0; q < N; q++) {
    const int lz = zi + 4 - R + ZS * q;
    act[q] = zi < ZS && (RZ % ZS == 0 || lz < 4 + S2_TZ + R);
    const int par = (ly + lz + C) & 1;
    const int i = (lz * S2_Y + ly) * S2_K + kk + ((5 - R - par) >> 1);
    id[q] = act[q] ? i : S2_K * S2_Y + S2_K + 1;  // any interior entry
    const int p = id[q];
    code[q] = L.c[C][p];
    nb[q][0] = oth[p];
    nb[q][1] = oth[p + 2 * par - 1];
    nb[q][2] = oth[p + S2_K];
    nb[q][3] = oth[p - S2_K];
    nb[q][4] = oth[p + S2_K * S2_Y];
    nb[q][5] = oth[p - S2_K * S2_Y];
    cen[q] = own[p];
    hb[q] = L.hb[C][p];
  }
  float xs[N], qs[N];
  bool redo = false;
#pragma unroll
  for (int q = 0; q < N; q++) {
    float sum = nb[q][0];
#pragma unroll
    for (int k = 1; k < 6; k++) sum += nb[q][k];
    xs[q] = sum - hb[q];
    if (ICNT) {
      const float2 cr = L.ct[code[q] & 63u];
      const float q0 = xs[q] * cr.y;
      const float er = __builtin_fmaf(-q0, cr.x, xs[q]);
      qs[q] = __builtin_fmaf(er, cr.y, q0);
      redo |= __builtin_amdgcn_classf(qs[q], 0x90);  // -subnormal | +subnormal
    } else {
      qs[q] = xs[q] / nc_count(code[q], wdir);
    }
  }
  if (ICNT && redo) {
#pragma unroll
    for (int q = 0; q < N; q++)
      if (__builtin_amdgcn_classf(qs[q], 0x90)) {
        float x = xs[q];
        asm volatile("" : "+v"(x));
        qs[q] = x / L.ct[code[q] & 63u].x;
      }
  }
#pragma unroll
  for (int q = 0; q < N; q++) {
    const float nv = mixf_(cen[q], qs[q], omega);
    const float o = (code[q] & (NC_SOLID | NC_NONE)) ? cen[q] : nv;
    if (OUT) {
      *v = o;
      *e = id[q];
    } else if (act[q]) {
      own[id[q]] = o;
    }
  }
}

// The coarse level that a fused prolongation (PRO) reads: 14 x 10 x 10 cells
// around the footprint, indices clamped to the level as in k_mg_prolong.
constexpr int S2_CX = S2_K + 2, S2_CY = S2_Y / 2 + 2, S2_CZ = S2_Z / 2 + 2, S2_CN = S2_CX * S2_CY * S2_CZ;
struct S2Coarse {
  int c0, c1, c2;
  const float *p;
  const uint8_t *f;
};
template <bool PRO>
struct S2CLds {
  float p[S2_CN];
  uint8_t f[S2_CN];
};
template <>
struct S2CLds<false> {};

// v[0..3] plus the masked, renormalised trilinear correction of mg.wgsl:97-120
// (k_mg_prolong, whose weights and order of sums these are) for the four cells
// from footprint x = 4 q at (ly, lz).  keep: cells that take no correction.
__device__ __forceinline__ void s2_prolong(const S2CLds<true> &C, bool solid, int q, int ly, int lz, uint32_t keep,
                                           float *v) {
  // cells 2 m and 2 m + 1 lie between the coarse cells m - 1, m and m, m + 1
  // with fractions 0.75 and 0.25; footprint cell 0 is even, and its m - 1 is
  // entry 0 of the staged cells
  const int base = (((lz + 1) >> 1) * S2_CY + ((ly + 1) >> 1)) * S2_CX + 2 * q;
  const float fy = (ly & 1) ? 0.25f : 0.75f, fz = (lz & 1) ? 0.25f : 0.75f;
  float pc[4][4], wyz[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {  // j = y offset + 2 z offset
    const int e = base + ((j >> 1) * S2_CY + (j & 1)) * S2_CX;
    wyz[j] = ((j & 1) ? fy : 1.0f - fy) * ((j >> 1) ? fz : 1.0f - fz);
#pragma unroll
    for (int k = 0; k < 4; k++) pc[j][k] = C.p[e + k];
  }
  // all weights are multiples of 1/64, so their products are exact in any order
  if (!solid) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float fx = (i & 1) ? 0.25f : 0.75f;
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < 8; k++) acc += (((k & 1) ? fx : 1.0f - fx) * wyz[k >> 1]) * pc[k >> 1][(i + 1) / 2 + (k & 1)];
      if (!((keep >> i) & 1u)) v[i] = v[i] + acc;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float fx = (i & 1) ? 0.25f : 0.75f;
    float acc = 0.0f, ws = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int j = k >> 1, m = (i + 1) / 2 + (k & 1);
      const bool sol = C.f[base + ((j >> 1) * S2_CY + (j & 1)) * S2_CX + m] == 1;
      const float w = sol ? 0.0f : ((k & 1) ? fx : 1.0f - fx) * wyz[j];
      acc += w * pc[j][m];
      ws += w;
    }
    float corr = acc;
    if (ws != 1.0f) {
      float x = acc;
      asm volatile("" : "+v"(x));
      corr = x / ws;
    }
    if (!((keep >> i) & 1u) && ws > 1e-4f) v[i] = v[i] + corr;
  }
}

// ALN: the level's x-size is a multiple of 4 (whole float4 and code words);
// otherwise the last group of a row is loaded from where it ends with the row
// and shifted, its elements past the row are masked, and codes are loaded as
// bytes.  The level has at most S2_MAX_ODD cells (32-bit offsets) and rows of
// at least four (sweep2_fits).
template <bool ALN, bool ICNT, bool PRO>
__global__ __launch_bounds__(S2_NT) void k_mg_sweep2(LvArgs a, int ntx, int nty, const float *__restrict__ b,
                                                      const uint8_t *__restrict__ nc, const float *__restrict__ pin,
                                                      float *__restrict__ pout, float omega, S2Coarse co) {
  __shared__ __align__(16) S2Lds L;
  __shared__ S2CLds<PRO> LC;
  const int t = threadIdx.x;
  if (ICNT && t < 64) {
    const uint32_t cnt = (t & 7u) + ((t >> 3) & 7u);
    L.ct[t] = make_float2((float)cnt, cnt ? 1.0f / (float)cnt : 0.0f);
  }
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = bid % ntx, rr = bid / ntx, ty = rr % nty, tz = rr / nty;
  const int x0 = tx * S2_TX - 4, y0 = ty * S2_TY - 4, z0 = tz * S2_TZ - 4;
  const RB rp = rb_of(pin, pin ? a.n * 4u : 0u), rbb = rb_of(b, a.n * 4u), rcd = rb_of(nc, a.n);
  constexpr int Q = S2_K / 2, NG = Q * S2_Y * S2_Z / S2_NT;
  static_assert(Q * S2_Y * S2_Z == NG * S2_NT, "whole staging rounds");
  float4 pv[NG], bv[NG];
  uint32_t cv[NG];
#pragma unroll
  for (int i = 0; i < NG; i++) {
    const int g = t + S2_NT * i, q = g % Q, row = g / Q, ly = row % S2_Y, lz = row / S2_Y;
    const int gx = x0 + 4 * q, gy = y0 + ly, gz = z0 + lz;
    const bool ok = (uint32_t)gx < (uint32_t)a.d0 && (uint32_t)gy < (uint32_t)a.d1 && (uint32_t)gz < (uint32_t)a.d2;
    const uint32_t n = (uint32_t)gx + (uint32_t)a.d0 * ((uint32_t)gy + (uint32_t)a.d1 * (uint32_t)gz);
    const int over = !ALN && gx + 4 > a.d0 ? gx + 4 - a.d0 : 0;  // elements past the row's end
    pv[i] = rb_ld4(rp, ok ? 4u * (n - over) : RB_OOB);
    bv[i] = rb_ld4(rbb, ok ? 4u * (n - over) : RB_OOB);
    if (ALN) {
      const uint32_t c = rb_ld32(rcd, ok ? n : RB_OOB);
      cv[i] = ok ? c : 0x40404040u;
    } else {
      uint32_t c = 0u;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool okj = ok && gx + j < a.d0;
        const uint32_t cj = __builtin_amdgcn_raw_buffer_load_b8(rcd.r, okj ? n + j : RB_OOB, 0, 0);
        c |= (okj ? cj : (uint32_t)NC_NONE) << (8 * j);
      }
      cv[i] = c;
    }
  }
  bool solid = false;
  if constexpr (PRO) {
#pragma unroll
    for (int i = 0; i < (S2_CN + S2_NT - 1) / S2_NT; i++) {
      const int g = min(t + S2_NT * i, S2_CN - 1), u = g % S2_CX, r = g / S2_CX;
      const int cx = clampi(x0 / 2 - 1 + u, 0, co.c0 - 1), cy = clampi(y0 / 2 - 1 + r % S2_CY, 0, co.c1 - 1);
      const int cz = clampi(z0 / 2 - 1 + r / S2_CY, 0, co.c2 - 1);
      const uint32_t j = (uint32_t)cx + (uint32_t)co.c0 * ((uint32_t)cy + (uint32_t)co.c1 * (uint32_t)cz);
      LC.p[g] = co.p[j];
      const uint8_t fl = co.f[j];
      LC.f[g] = fl;
      solid |= fl == 1;
    }
    solid = __syncthreads_or(solid);
  }
#pragma unroll
  for (int i = 0; i < NG; i++) {
    const int g = t + S2_NT * i, q = g % Q, row = g / Q, ly = row % S2_Y, lz = row / S2_Y;
    float4 v = pv[i], w = bv[i];
    const uint32_t c = cv[i];
    if (!ALN) {
      const int over = x0 + 4 * q + 4 - a.d0;
      v = shift4(v, over);
      w = shift4(w, over);
    }
    if constexpr (PRO) {
      const int gx = x0 + 4 * q, gy = y0 + ly, gz = z0 + lz;
      if ((uint32_t)gx < (uint32_t)a.d0 && (uint32_t)gy < (uint32_t)a.d1 && (uint32_t)gz < (uint32_t)a.d2) {
        float vv[4] = {v.x, v.y, v.z, v.w};
        const uint32_t keep = ALN || gx + 4 <= a.d0 ? 0u : (0xfu << (a.d0 - gx));  // past the row's end
        s2_prolong(LC, solid, q, ly, lz, keep, vv);
        v = make_float4(vv[0], vv[1], vv[2], vv[3]);
      }
    }
    if (c & 0x80808080u) {  // solids read 0 in the neighbour sums
      if (c & 0x80u) v.x = 0.0f;
      if (c & 0x8000u) v.y = 0.0f;
      if (c & 0x800000u) v.z = 0.0f;
      if (c & 0x80000000u) v.w = 0.0f;
    }
    const int e = row * S2_K + 2 * q, o = (ly + lz) & 1;  // o: colour of the group's even cells
    *reinterpret_cast<float2 *>(L.p[o] + e) = make_float2(v.x, v.z);
    *reinterpret_cast<float2 *>(L.p[1 - o] + e) = make_float2(v.y, v.w);
    *reinterpret_cast<float2 *>(L.hb[o] + e) = make_float2(a.hh * w.x, a.hh * w.z);
    *reinterpret_cast<float2 *>(L.hb[1 - o] + e) = make_float2(a.hh * w.y, a.hh * w.w);
    *reinterpret_cast<uint16_t *>(L.c[o] + e) = (uint16_t)((c & 0xffu) | ((c >> 8) & 0xff00u));
    *reinterpret_cast<uint16_t *>(L.c[1 - o] + e) = (uint16_t)(((c >> 8) & 0xffu) | ((c >> 16) & 0xff00u));
  }
  __syncthreads();
  s2_pass<0, 3, ICNT, false>(L, omega, a.wdir, nullptr, nullptr);
  __syncthreads();
  s2_pass<1, 2, ICNT, false>(L, omega, a.wdir, nullptr, nullptr);
  __syncthreads();
  s2_pass<0, 1, ICNT, false>(L, omega, a.wdir, nullptr, nullptr);
  __syncthreads();
  float v1;
  int e;
  s2_pass<1, 0, ICNT, true>(L, omega, a.wdir, &v1, &e);
  // the thread's colour-1 cell and its pair's colour-0 cell
  const int row = e / S2_K, k = e - row * S2_K, ly = row % S2_Y, lz = row / S2_Y;
  const int gx = x0 + 2 * k, gy = y0 + ly, gz = z0 + lz;
  if (gx >= a.d0 || gy >= a.d1 || gz >= a.d2) return;
  const int o = (ly + lz) & 1;  // colour of the pair's even cell
  const float v0 = L.p[0][e];
  float lo = o ? v1 : v0, hi = o ? v0 : v1;
  const uint32_t n = (uint32_t)gx + (uint32_t)a.d0 * ((uint32_t)gy + (uint32_t)a.d1 * (uint32_t)gz);
  const bool second = ALN || gx + 1 < a.d0;
  if (pin) {  // solid cells keep their phi (zeroed only in LDS)
    if (L.c[o][e] & NC_SOLID) lo = pin[n];
    if (second && (L.c[1 - o][e] & NC_SOLID)) hi = pin[n + 1];
  }
  if (ALN) {
    *reinterpret_cast<float2 *>(pout + n) = make_float2(lo, hi);
  } else {
    pout[n] = lo;
    if (second) pout[n + 1] = hi;
  }
}

// Levels that take both sweeps in one launch.  The tile's rings cost 2.4
// updates a cell and sweep against 1.5, so the launch saved (two, with the
// prolongation) has to be worth more than the work: four V-cycles with and
// without it for the level of n cells:
//   40x80x40 (128 k)   514 us before, 467 now     48x32x48 (74 k)  299, 278
//   80x120x80 (768 k)  1312 (its finer level apart), 1300
//   80x160x80 (1.02 M) 467 without, 479 with      160x320x160      1498, 1844
//   a solve at 96^3 (885 k)  2960 us without, 2893 with; 128^3 (2.1 M) 4453, 4727
// Rows that are no multiple of four cells take k_mg_sweep one element at a
// time, and there the line lies higher: a solve at 97x61x118 5594 us before,
// 4101 now; 129^3 (2.1 M) 9721 without, 9325 with; 193x121x235 (5.5 M) 17.45
// ms, 17.38 (no more than two runs differ); 255^3 30.8, 31.9.
constexpr uint32_t S2_MAX = 900000u, S2_MAX_ODD = 4000000u;
// The prolongation joins them up to here: every cell of the rings is prolonged
// too (6 times the tile).  A solve at 97x61x118 (its 698 k cells) 3.93 ms
// with it in the launch, 3.78 without; 129^3 9.07 and 8.44; 96^3 2.84 and
// 2.77; with a line of 50 k instead, four V-cycles at 80x160x80 (128 k) 465 us
// against 458.
constexpr uint32_t S2_PROLONG_MAX = 500000u;
static bool sweep2_fits(const MgLevel &L) { return L.d[0] >= 4 && L.n <= (L.d[0] % 4 ? S2_MAX_ODD : S2_MAX); }
// C: the level whose correction is added first, or null
static void launch_mg_sweep2(const MgLevel &L, const MgLevel *C, const float *pin, float *pout, float omega,
                             hipStream_t s) {
  const LvArgs a = lv_args(L);
  const int ntx = (L.d[0] + S2_TX - 1) / S2_TX, nty = (L.d[1] + S2_TY - 1) / S2_TY, ntz = (L.d[2] + S2_TZ - 1) / S2_TZ;
  const int nb = ntx * nty * ntz;
  const S2Coarse co = C ? S2Coarse{C->d[0], C->d[1], C->d[2], C->phi, C->f} : S2Coarse{};
#define PYRO_SWEEP2(A_, I_, P_) \
  k_mg_sweep2<A_, I_, P_><<<nb, S2_NT, 0, s>>>(a, ntx, nty, L.b, L.nc, pin, pout, omega, co)
  const int k = (L.d[0] % 4 == 0 ? 4 : 0) + (L.wdir == 1.0f ? 2 : 0) + (C ? 1 : 0);
  switch (k) {
    case 0: PYRO_SWEEP2(false, false, false); break;
    case 1: PYRO_SWEEP2(false, false, true); break;
    case 2: PYRO_SWEEP2(false, true, false); break;
    case 3: PYRO_SWEEP2(false, true, true); break;
    case 4: PYRO_SWEEP2(true, false, false); break;
    case 5: PYRO_SWEEP2(true, false, true); break;
    case 6: PYRO_SWEEP2(true, true, false); break;
    default: PYRO_SWEEP2(true, true, true); break;
  }
#undef PYRO_SWEEP2
}

// ---------------------------------------------------------------- coarse
// All red-black SOR iterations of the coarsest level (sim.rs:472-473: 80
// iterations, omega = 1.6): in the tail's workgroup (up to 16 k cells, by
// their shape), in one workgroup with a thread per column (below), or else as
// sweep launches (launch_mg_coarse has the rule).
constexpr int CO_NT = 1024;
constexpr int CO_PAD_MAX = 36000;  // floats of the column solve's LDS (144 KB)

// The solve with one thread per (x, y) column and the column's phi in
// registers, for an outside weight of 1 (integer counts 1..6, div_count).
// LDS holds phi plane-major: plane z + 1 (z = -1 .. ZJ - 1) of CZ_PLANE
// floats, the cell of column c = x + d0 * y at offset c.  CZ_PLANE is a
// multiple of 64, so a read or store of one slot by the 64 lanes of a wave
// (consecutive columns) touches 64 distinct banks.  Columns c >= d0 * d1 are
// zero; a lane on a side of the domain reads its missing x or y neighbour
// from the zero block at CZ_ZERO + (the neighbour's column mod 64), the bank
// the neighbour would have used, which gives the Dirichlet phi = 0 beyond the
// sides.  A cell reads its four x/y neighbours in LDS and its two z
// neighbours from registers.  Register slot j of a column holds
// z = j - ((x + y) & 1), so the cells of colour c are the slots j = c, c + 2,
// ... on every lane; slots outside the column hold phi = 0 and count 0 (each
// pass computes them like the others and they keep +0), which gives the
// Dirichlet phi = 0 above the top and below the bottom.
//
// EX (whole waves): the block has blockDim.x = 64 k < d0 d1 threads, one per
// column c < blockDim.x; the cells of the remaining columns (each SIMD issues
// its waves' VALU work in turn, so a wave of columns beyond a multiple of
// four adds a whole wave's slots to one SIMD) are taken one per thread and colour: extra
// index e = thread of colour c is leftover column blockDim.x + e % NL, cell
// z = ((c + parity) & 1) + 2 (e / NL), NL = d0 d1 - blockDim.x leftover
// columns (consecutive lanes, consecutive columns: distinct banks).  An extra cell
// reads all six neighbours in LDS (z +- 1: planes; the planes z = -1 and
// z = d2 hold +0) and keeps its phi in a register.
constexpr int CZ_ZERO = CO_NT, CZ_PLANE = CO_NT + 64, CZ_EX_NT = 768;

template <int ZJ, bool EX = false>
__global__ __launch_bounds__(EX ? CZ_EX_NT : CO_NT) void k_mg_coarse_z(LvArgs a, const float *__restrict__ b,
                                                                        const uint8_t *__restrict__ nc,
                                                                        float *__restrict__ p, int iters,
                                                                        float omega) {
  constexpr int PN = (ZJ + 1) * CZ_PLANE;  // planes z + 1 = j + 1 - par for slots j < ZJ
  static_assert(PN <= CO_PAD_MAX, "planes exceed the LDS budget");
  static_assert(!EX || ZJ > 12, "extra cells are taken by the long-column passes");
  __shared__ float sp[PN];
  const uint32_t sy = (uint32_t)a.d0, sz = (uint32_t)a.d0 * (uint32_t)a.d1;
  for (int i = threadIdx.x; i < PN; i += (int)blockDim.x) sp[i] = 0.0f;
  const int ncol = a.d0 * a.d1;  // <= CO_NT (host)
  const int col = threadIdx.x;
  const bool has = col < ncol;
  const int x = has ? col % a.d0 : 0, y = has ? col / a.d0 : 0;
  const int par = (x + y) & 1;
  // LDS index of slot j is B + j * CZ_PLANE.  A lane without a column
  // (ncol <= col < CO_NT) reads columns col +- 1 and the zero block, all
  // inside a plane, and never stores.
  const int B = (1 - par) * CZ_PLANE + col;
  const int cxp = !has || x < a.d0 - 1 ? col + 1 : CZ_ZERO + ((col + 1) & 63);
  const int cxm = !has || x > 0 ? col - 1 : CZ_ZERO + ((col - 1) & 63);
  const int cyp = has && y < a.d1 - 1 ? col + a.d0 : CZ_ZERO + ((col + a.d0) & 63);
  const int cym = has && y > 0 ? col - a.d0 : CZ_ZERO + ((col - a.d0) & 63);
  float ph[ZJ + 2], hb[ZJ], rc[ZJ];
  uint32_t cp[(ZJ + 3) / 4];
  ph[0] = 0.0f;
  ph[ZJ + 1] = 0.0f;
#pragma unroll
  for (int k = 0; k < (ZJ + 3) / 4; k++) cp[k] = 0u;
#pragma unroll
  for (int j = 0; j < ZJ; j++) {
    const int z = j - par;
    // a slot that is never updated (outside the column, solid, or a cell
    // with no fluid neighbour and no open face) holds phi = 0, count 0 and
    // reciprocal 0: its quotient is then +-0 and the update keeps +0, so the
    // passes need no per-slot select.  Such a cell's phi is read only by
    // solid neighbours, which are not updated, and is not written back.
    float v = 0.0f, h = 0.0f, r = 0.0f;
    uint32_t cnt = 0u;
    if (has && z >= 0 && z < a.d2) {
      const uint32_t g = (uint32_t)x + sy * (uint32_t)y + sz * (uint32_t)z;
      const uint8_t code = nc[g];
      if (!(code & (NC_SOLID | NC_NONE))) {
        v = p[g];
        cnt = (code & 7u) + ((code >> 3) & 7u);
        h = a.hh * b[g];
        r = 1.0f / (float)cnt;
      }
    }
    ph[j + 1] = v;
    hb[j] = h;
    rc[j] = r;
    cp[j >> 2] |= cnt << (8 * (j & 3));
  }
  // extra cell of each colour (EX): LDS index, neighbour indices, count,
  // reciprocal, h^2 b, phi; a cell that is never updated holds 0 as above
  bool ev[2] = {false, false};
  int ei[2] = {0, 0}, en[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  float ec[2] = {0.0f, 0.0f}, er[2] = {0.0f, 0.0f}, eh[2] = {0.0f, 0.0f}, ep[2] = {0.0f, 0.0f};
  if constexpr (EX) {
    const int nl = ncol - (int)blockDim.x;  // 1 .. 63 leftover columns (the host launches EX only then)
    const int k = col / nl;
    const int cl = (int)blockDim.x + (col - k * nl);  // leftover column
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const int xl = cl % a.d0, yl = cl / a.d0;
      const int z = ((c + xl + yl) & 1) + 2 * k;
      if (z >= a.d2) continue;
      const int pl = (z + 1) * CZ_PLANE;
      ev[c] = true;
      ei[c] = pl + cl;
      en[c][0] = pl + (xl < a.d0 - 1 ? cl + 1 : CZ_ZERO + ((cl + 1) & 63));
      en[c][1] = pl + (xl > 0 ? cl - 1 : CZ_ZERO + ((cl - 1) & 63));
      en[c][2] = pl + (yl < a.d1 - 1 ? cl + a.d0 : CZ_ZERO + ((cl + a.d0) & 63));
      en[c][3] = pl + (yl > 0 ? cl - a.d0 : CZ_ZERO + ((cl - a.d0) & 63));
      const uint32_t g = (uint32_t)xl + sy * (uint32_t)yl + sz * (uint32_t)z;
      const uint8_t code = nc[g];
      if (!(code & (NC_SOLID | NC_NONE))) {
        const uint32_t cnt = (code & 7u) + ((code >> 3) & 7u);
        ep[c] = p[g];
        ec[c] = (float)cnt;
        er[c] = 1.0f / (float)cnt;
        eh[c] = a.hh * b[g];
      }
    }
  }
  __syncthreads();  // the zero fill is complete
  if (has) {
#pragma unroll
    for (int j = 0; j < ZJ; j++) {
      const int z = j - par;
      if (z >= 0 && z < a.d2) sp[B + j * CZ_PLANE] = ph[j + 1];
    }
  }
  if constexpr (EX) {
#pragma unroll
    for (int c = 0; c < 2; c++)
      if (ev[c]) sp[ei[c]] = ep[c];
  }
  __syncthreads();
  const int pb = (1 - par) * CZ_PLANE;
  const float *sxp = sp + pb + cxp, *sxm = sp + pb + cxm, *syp = sp + pb + cyp, *sym = sp + pb + cym;
  for (int it = 0; it < iters; it++) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
      for (int k = 0; k < (ZJ + 3) / 4; k++) asm volatile("" : "+v"(cp[k]));  // conversions stay in the loop
      // every slot of the colour is computed and stored (reads and stores
      // stay inside sp: planes j + 1 - par <= ZJ, columns < CZ_PLANE; a slot
      // that is never updated stores its +0); the stores follow all reads of
      // the pass, so no read waits on them.  Each sum starts with its first
      // term rather than +0 + term: the two differ only in the sign of a
      // zero sum, and the update maps either to the same value.
      if constexpr (ZJ <= 12) {
        // Short columns (one wave per SIMD on small levels): the slots of a
        // colour are independent (red-black), so all of the pass's LDS reads
        // are issued first, the fast quotients of every slot are formed
        // branch-free, and one branch per pass redoes by IEEE division any
        // quotient that came out subnormal (div_count); the slots' latencies
        // overlap instead of queueing behind one another.
        constexpr int NS = ZJ / 2;
        float xs[NS], qs[NS], nb[4][NS];
        bool redo = false;
#pragma unroll
        for (int t = 0; t < NS; t++) {
          const int j = c + 2 * t;
          nb[0][t] = sxp[j * CZ_PLANE];
          nb[1][t] = sxm[j * CZ_PLANE];
          nb[2][t] = syp[j * CZ_PLANE];
          nb[3][t] = sym[j * CZ_PLANE];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NS; t++) {
          const int j = c + 2 * t;
          const float cn = (float)((cp[j >> 2] >> (8 * (j & 3))) & 0xffu);
          float sum = nb[0][t];
          sum += nb[1][t];
          sum += nb[2][t];
          sum += nb[3][t];
          sum += ph[j + 2];
          sum += ph[j];
          const float x = sum - hb[j];
          const float q0 = x * rc[j];
          const float e = __builtin_fmaf(-q0, cn, x);
          xs[t] = x;
          qs[t] = __builtin_fmaf(e, rc[j], q0);
          redo |= __builtin_amdgcn_classf(qs[t], 0x90);
        }
        if (redo) {
#pragma unroll
          for (int t = 0; t < NS; t++) {
            const int j = c + 2 * t;
            if (__builtin_amdgcn_classf(qs[t], 0x90)) {
              float x = xs[t];
              asm volatile("" : "+v"(x));
              qs[t] = x / (float)((cp[j >> 2] >> (8 * (j & 3))) & 0xffu);
            }
          }
        }
#pragma unroll
        for (int t = 0; t < NS; t++) {
          const int j = c + 2 * t;
          ph[j + 1] = mixf_(ph[j + 1], qs[t], omega);
        }
      } else {
        // Long columns: many waves share each SIMD and hide the latency;
        // registers are the limit (no per-pass arrays).  The next slot's
        // four reads are issued before this slot's arithmetic.  A quotient
        // that came out subnormal is only noted: LDS still holds the pass's
        // old values, from which the rare lane recomputes its slots with the
        // IEEE division.  The scheduling barriers keep the reads one slot
        // ahead: left to itself the compiler gathers all of a pass's reads,
        // and the waves then wait on the LDS together.  20x40x20: 165 us with
        // a branch a slot, 183 without the barriers, 155 now; 18x28x18 145,
        // 165 and 121; the counts kept as floats (21 more registers) 157.
        bool redo = false;
        float nb[4] = {sxp[c * CZ_PLANE], sxm[c * CZ_PLANE], syp[c * CZ_PLANE], sym[c * CZ_PLANE]};
#pragma unroll
        for (int j = c; j < ZJ; j += 2) {
          float nx[4] = {0.0f, 0.0f, 0.0f, 0.0f};
          if (j + 2 < ZJ) {
            nx[0] = sxp[(j + 2) * CZ_PLANE];
            nx[1] = sxm[(j + 2) * CZ_PLANE];
            nx[2] = syp[(j + 2) * CZ_PLANE];
            nx[3] = sym[(j + 2) * CZ_PLANE];
          }
          __builtin_amdgcn_sched_barrier(0);
          const float cn = (float)((cp[j >> 2] >> (8 * (j & 3))) & 0xffu);
          float sum = nb[0];
          sum += nb[1];
          sum += nb[2];
          sum += nb[3];
          sum += ph[j + 2];
          sum += ph[j];
          ph[j + 1] = mixf_(ph[j + 1], quot_count(sum - hb[j], cn, rc[j], redo), omega);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int k = 0; k < 4; k++) nb[k] = nx[k];
        }
        if (redo) {
#pragma unroll
          for (int j = c; j < ZJ; j += 2) {
            const float cn = (float)((cp[j >> 2] >> (8 * (j & 3))) & 0xffu);
            float sum = sxp[j * CZ_PLANE];
            sum += sxm[j * CZ_PLANE];
            sum += syp[j * CZ_PLANE];
            sum += sym[j * CZ_PLANE];
            sum += ph[j + 2];
            sum += ph[j];
            ph[j + 1] = mixf_(sp[B + j * CZ_PLANE], div_count(sum - hb[j], cn, rc[j]), omega);
          }
        }
      }
#pragma unroll
      for (int j = c; j < ZJ; j += 2) sp[B + j * CZ_PLANE] = ph[j + 1];
      if constexpr (EX) {
        if (ev[c]) {
          const int i = ei[c];
          float sum = sp[en[c][0]];
          sum += sp[en[c][1]];
          sum += sp[en[c][2]];
          sum += sp[en[c][3]];
          sum += sp[i + CZ_PLANE];
          sum += sp[i - CZ_PLANE];
          ep[c] = mixf_(ep[c], div_count(sum - eh[c], ec[c], er[c]), omega);
          sp[i] = ep[c];
        }
      }
      __syncthreads();
    }
  }
  if (has) {
#pragma unroll
    for (int j = 0; j < ZJ; j++) {
      const int z = j - par;
      if (z >= 0 && z < a.d2) {
        const uint32_t g = (uint32_t)x + sy * (uint32_t)y + sz * (uint32_t)z;
        if (!(nc[g] & (NC_SOLID | NC_NONE))) p[g] = ph[j + 1];
      }
    }
  }
  if constexpr (EX) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (!ev[c]) continue;
      const int z = ei[c] / CZ_PLANE - 1, cl = ei[c] - (z + 1) * CZ_PLANE;
      const uint32_t g = (uint32_t)cl + sz * (uint32_t)z;  // column index cl = x + d0 y
      if (!(nc[g] & (NC_SOLID | NC_NONE))) p[g] = ep[c];
    }
  }
}

// ---------------------------------------------------------------- tail
// The V-cycle from level `t` down and back up in one launch of one workgroup,
// for the levels that fit its LDS: two sweeps and the restriction on each
// level, all SOR iterations of the coarsest (sim.rs:472-473), then the
// prolongation and two sweeps on the way up -- the per-cell arithmetic and the
// order of every sum are those of the kernels above.  On these levels (8 k
// cells and fewer) a launch per sweep or transfer takes 4-5 us, all of it
// launch and load latency, and the coarsest solve is a chain of 160 dependent
// colour passes: both are bound by latency, which one workgroup with
// everything in LDS and registers shortens.  Per launch, before and after:
// levels 16x24x16 + 8x12x8 88 -> 47 us (two sweeps, restriction, solve,
// prolongation, two sweeps), 10x20x10 alone 71 -> 39 us, 14x30x14 142 -> 97 us.
//
// Layout: an x-pair (2g, 2g + 1) of a row holds one cell of each colour, and
// the two colours live in two LDS arrays indexed by pair (TL_CS floats apart,
// an immediate offset): a colour pass then reads and writes consecutive words
// in consecutive lanes (x with stride 2 would meet each bank twice).  For the
// cell of colour c in pair (g, y, z), at x = 2g + o with o = (y + z + c) & 1,
// the neighbours are in the other colour's array: x -+ 1 at pair g and at
// g + (o ? 1 : -1), y -+ 1 and z -+ 1 at the pairs of the same g.  (The two x
// terms open the sum, so their order does not matter.)  Rows have a pitch of
// hx + 1, planes of (d1 + 1) rows: one ghost column, row and plane between
// neighbours holds the phi = 0 beyond the box.
constexpr int TL_NT = 1024, TL_MAX = 5, TL_CS = 12288, TL_K = 8, TL_TOP = 4, TL_INNER = 4096;

struct TailLv {
  int d0, d1, d2, hx, py, pz;
  int off, np, n;  // LDS offset of the level's pairs, pairs, cells
  int io, bo;      // offsets of the level's codes and of an inner level's b in LDS
  float hh, wdir;
  FastDiv dhx, dd0, dd1;
  const __attribute__((address_space(1))) uint8_t *nc;  // global memory
  __attribute__((address_space(1))) float *phi, *b;
};
struct TailArgs {
  int nl, iters;
  float omega;
  TailLv l[TL_MAX];
};

// x / c for a count c = fluid + wdir * outside given r = RN(1/c): div_count's
// corrected product.  Over every float x with 2^-102 <= |x| < infinity and
// each c of the levels 1..11 (214 values) it equals the IEEE quotient; a
// smaller nonzero x (the remainder's low bits underflow) and an infinity (NaN
// product) take the division.  c = r = 0 gives 0.
template <bool ICNT>
__device__ __forceinline__ bool div_redo(float x, float q, float r) {
  if (ICNT) return __builtin_amdgcn_classf(q, 0x90);  // -subnormal | +subnormal
  return r != 0.0f && ((fabsf(x) < 0x1p-100f && x != 0.0f) || q != q);
}

// LDS of the tail: phi (colour 0, then colour 1 at + TL_CS); b of the inner
// levels and the neighbour codes of all, by cell; (count, RN(1/count)) of
// level k's codes at ctab + 64 k.
#define TAIL_SH float *sp, float *bl, uint8_t *cl, const float2 *ctab

__device__ __forceinline__ void tail_pair(const TailLv &L, int p, int &g, int &y, int &z) {
  const uint32_t r = fdiv((uint32_t)p, L.dhx), q = fdiv(r, L.dd1);
  g = p - (int)r * L.hx;
  z = (int)q;
  y = (int)r - z * L.d1;
}
__device__ __forceinline__ int tail_li(const TailLv &L, int g, int y, int z) {
  return L.off + (z + 1) * L.pz + (y + 1) * L.py + g + 1;
}

// The pairs t + 1024 j of thread t on one level: LDS index, cell 2g, codes of
// the two colours | o of colour 0 << 16 | cell 2g in the level << 17 | cell
// 2g + 1 << 18, h^2 b.
template <int K>
struct TailOwn {
  int li[K], gi[K];
  uint32_t cd[K];
  float hb[K][2];
};
template <int K, bool inner>
__device__ __forceinline__ void tail_own(const TailLv &L, TAIL_SH, TailOwn<K> &W) {
#pragma unroll
  for (int j = 0; j < K; j++) {
    const int p = (int)threadIdx.x + TL_NT * j;
    const bool act = p < L.np;
    int g, y, z;
    tail_pair(L, act ? p : 0, g, y, z);
    const int o = (y + z) & 1, gi = 2 * g + L.d0 * (y + L.d1 * z);
    const bool two = 2 * g + 1 < L.d0;
    const int i1 = two ? gi + 1 : gi;
    const uint32_t a0 = inner ? cl[L.io + gi] : L.nc[gi], a1 = inner ? cl[L.io + i1] : L.nc[i1];
    const float b0 = inner ? bl[L.bo + gi] : L.b[gi], b1 = inner ? bl[L.bo + i1] : L.b[i1];
    const uint32_t c0 = act ? a0 : (uint32_t)NC_NONE, c1 = act && two ? a1 : (uint32_t)NC_NONE;
    W.li[j] = tail_li(L, g, y, z);
    W.gi[j] = gi;
    W.cd[j] = (o ? c1 | (c0 << 8) : c0 | (c1 << 8)) | ((uint32_t)o << 16) | (act ? 1u << 17 : 0u) |
              (act && two ? 1u << 18 : 0u);
    const float h0 = L.hh * b0, h1 = L.hh * b1;
    W.hb[j][0] = o ? h1 : h0;
    W.hb[j][1] = o ? h0 : h1;
  }
}

// Red-black sweeps over the owned pairs.
template <int K, bool ICNT>
__device__ __forceinline__ void tail_sweeps(const TailLv &L, TAIL_SH, int k, const TailOwn<K> &W, int sweeps,
                                            float omega) {
  const float2 *ct = ctab + 64 * k;
  const int py = L.py, pz = L.pz;
  for (int s = 0; s < sweeps; s++) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      float *A = sp + c * TL_CS;
      const float *O = sp + (1 - c) * TL_CS;
      constexpr int KC = K < 2 ? K : 2;  // cells in flight (16 waves share the CU)
#pragma unroll
      for (int j0 = 0; j0 < K; j0 += KC) {
        if (TL_NT * j0 >= L.np) break;  // no thread owns a pair here (uniform)
        float nb[KC][6], cen[KC];
        float2 cr[KC];
#pragma unroll
        for (int q = 0; q < KC; q++) {
          const int j = j0 + q, i = W.li[j];
          const int o = (int)((W.cd[j] >> 16) & 1u) ^ c;
          nb[q][0] = O[i];
          nb[q][1] = O[i + 2 * o - 1];
          nb[q][2] = O[i + py];
          nb[q][3] = O[i - py];
          nb[q][4] = O[i + pz];
          nb[q][5] = O[i - pz];
          cen[q] = A[i];
          cr[q] = ct[(W.cd[j] >> (8 * c)) & 63u];
        }
        float xs[KC], qs[KC];
        bool redo = false;
#pragma unroll
        for (int q = 0; q < KC; q++) {
          float sum = nb[q][0];
#pragma unroll
          for (int m = 1; m < 6; m++) sum += nb[q][m];
          xs[q] = sum - W.hb[j0 + q][c];
          const float q0 = xs[q] * cr[q].y;
          const float e = __builtin_fmaf(-q0, cr[q].x, xs[q]);
          qs[q] = __builtin_fmaf(e, cr[q].y, q0);
          redo |= div_redo<ICNT>(xs[q], qs[q], cr[q].y);
        }
        if (redo) {
#pragma unroll
          for (int q = 0; q < KC; q++)
            if (div_redo<ICNT>(xs[q], qs[q], cr[q].y)) {
              float x = xs[q];
              asm volatile("" : "+v"(x));
              qs[q] = x / cr[q].x;
            }
        }
#pragma unroll
        for (int q = 0; q < KC; q++) {
          const float nv = mixf_(cen[q], qs[q], omega);
          if (!((W.cd[j0 + q] >> (8 * c)) & (uint32_t)(NC_SOLID | NC_NONE))) A[W.li[j0 + q]] = nv;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
    }
  }
}

// Residual of level F averaged over the fluid children of each cell of C
// (k_mg_restrict; phi of C is 0 from the fill): a coarse cell's x-children
// are one pair.
template <bool inner>
__device__ __forceinline__ void tail_restrict(const TailLv &F, const TailLv &C, TAIL_SH) {
  for (int i = threadIdx.x; i < C.n; i += TL_NT) {
    const uint32_t r = fdiv((uint32_t)i, C.dd0), zq = fdiv(r, C.dd1);
    const int x = i - (int)r * C.d0, z = (int)zq, y = (int)r - z * C.d1;
    const bool two = 2 * x + 1 < F.d0;
    const int f0 = 2 * x + F.d0 * (2 * y + F.d1 * 2 * z), q0 = tail_li(F, x, 2 * y, 2 * z);
    float bv[8];
    uint32_t cv[8];
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const int dy = m & 1, dz = m >> 1;
      const bool in = 2 * y + dy < F.d1 && 2 * z + dz < F.d2;
      const int f = in ? f0 + F.d0 * (dy + F.d1 * dz) : f0, f1 = two ? f + 1 : f;
      const uint32_t a0 = cl[F.io + f], a1 = cl[F.io + f1];
      bv[2 * m] = inner ? bl[F.bo + f] : F.b[f];
      bv[2 * m + 1] = inner ? bl[F.bo + f1] : F.b[f1];
      cv[2 * m] = in ? a0 : (uint32_t)NC_SOLID;
      cv[2 * m + 1] = in && two ? a1 : (uint32_t)NC_SOLID;
    }
    float acc = 0.0f, nfl = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (cv[k] & NC_SOLID) continue;  // solid or outside the level
      const int o = k & 1, dy = (k >> 1) & 1, dz = k >> 2;
      const int col = (o + dy + dz) & 1;  // colour of x = 2 g + o at even y and z plus dy, dz
      const float *A = sp + col * TL_CS, *O = sp + (1 - col) * TL_CS;
      const int q = q0 + dy * F.py + dz * F.pz;
      nfl += 1.0f;
      float sum = 0.0f;
      sum += O[q + o];      // x + 1
      sum += O[q + o - 1];  // x - 1
      sum += O[q + F.py];
      sum += O[q - F.py];
      sum += O[q + F.pz];
      sum += O[q - F.pz];
      acc += bv[k] - (sum - nc_count(cv[k], F.wdir) * A[q]) / F.hh;
    }
    const float bc = nfl > 0.0f ? acc / fmax_(nfl, 1.0f) : 0.0f;
    bl[C.bo + i] = bc;
    C.b[i] = bc;
  }
  __syncthreads();
}

// Masked, renormalised trilinear correction of level F from C (the general
// form of k_mg_prolong), one coarse cell's eight children per thread: they
// interpolate from its 27 neighbours, clamped at the level's sides.  A fine
// index's fraction is 0.75 (even) or 0.25 (odd), so the weights are exact
// products of constants, and without a solid coarse cell they sum to 1.
__device__ __forceinline__ void tail_prolong(const TailLv &C, const TailLv &F, TAIL_SH, bool solid) {
  for (int i = threadIdx.x; i < C.n; i += TL_NT) {
    const uint32_t r = fdiv((uint32_t)i, C.dd0), zq = fdiv(r, C.dd1);
    const int X = i - (int)r * C.d0, Z = (int)zq, Y = (int)r - Z * C.d1;
    const int xs[3] = {X > 0 ? X - 1 : 0, X, X + 1 < C.d0 ? X + 1 : X};
    float v[27];
    uint32_t sm = 0u;
#pragma unroll
    for (int m = 0; m < 9; m++) {
      const int cy = clampi(Y + m % 3 - 1, 0, C.d1 - 1), cz = clampi(Z + m / 3 - 1, 0, C.d2 - 1);
      const int row = tail_li(C, 0, cy, cz), par = cy + cz;
#pragma unroll
      for (int u = 0; u < 3; u++)
        v[3 * m + u] = sp[((xs[u] + par) & 1) * TL_CS + row + (xs[u] >> 1)];
      if (solid) {
        const int crow = C.io + C.d0 * (cy + C.d1 * cz);
#pragma unroll
        for (int u = 0; u < 3; u++) sm |= (cl[crow + xs[u]] & NC_SOLID) ? 1u << (3 * m + u) : 0u;
      }
    }
    const int q0 = tail_li(F, X, 2 * Y, 2 * Z), f0 = F.io + 2 * X + F.d0 * (2 * Y + F.d1 * 2 * Z);
#pragma unroll
    for (int ch = 0; ch < 8; ch++) {
      const int o = ch & 1, dy = (ch >> 1) & 1, dz = ch >> 2;
      if (2 * X + o >= F.d0 || 2 * Y + dy >= F.d1 || 2 * Z + dz >= F.d2) continue;
      if (cl[f0 + o + F.d0 * (dy + F.d1 * dz)] & NC_SOLID) continue;
      const float frx = o ? 0.25f : 0.75f, fry = dy ? 0.25f : 0.75f, frz = dz ? 0.25f : 0.75f;
      float acc = 0.0f, ws = 0.0f;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int ox = k & 1, oy = (k >> 1) & 1, oz = k >> 2;
        const int e = 3 * (3 * (oz + dz) + (oy + dy)) + ox + o;
        const float wx = ox ? frx : 1.0f - frx, wy = oy ? fry : 1.0f - fry, wz = oz ? frz : 1.0f - frz;
        float wgt = (wx * wy) * wz;
        if (solid) {
          wgt = (sm >> e) & 1u ? 0.0f : wgt;
          ws += wgt;
        }
        acc += wgt * v[e];
      }
      float corr = acc;
      if (solid && ws != 1.0f) {
        float a = acc;
        asm volatile("" : "+v"(a));
        corr = a / ws;
      }
      float *A = sp + ((o + dy + dz) & 1) * TL_CS + q0 + dy * F.py + dz * F.pz;
      if (!solid || ws > 1e-4f) *A = *A + corr;
    }
  }
  __syncthreads();
}

// The SOR iterations of the coarsest level: thread t owns K pairs of one
// (g, y) column, z = z0 .. z0 + K - 1, with phi, h^2 b, count and reciprocal
// of both colours in registers.  The pair's other cell and the z neighbours
// inside the segment are registers too, so a cell costs three LDS reads plus
// the segment's two ends.  A pass issues its reads first and stores the
// branch-free quotients; one branch per pass redoes those that need the IEEE
// division and stores them again.  K = 1 spreads a small level over the most
// lanes: the pass is then its latency chain (LDS read, 13 dependent
// operations, LDS write, barrier).  A slot that is never updated holds phi =
// count = reciprocal = 0 and keeps 0, as in k_mg_coarse_z.
template <int K, bool ICNT, bool inner>
__device__ __forceinline__ void tail_sor(const TailLv &L, TAIL_SH, int k, int iters, float omega) {
  const float2 *ct = ctab + 64 * k;
  const int cols = L.hx * L.d1;
  const int nseg = (L.d2 + K - 1) / K;
  const int t = threadIdx.x;
  if (__builtin_amdgcn_readfirstlane(t) >= cols * nseg) {  // a wave without columns only keeps the barriers
    for (int it = 0; it < 2 * iters; it++) __syncthreads();
    return;
  }
  const bool act = t < cols * nseg;
  const int seg = act ? t / cols : 0, cg = act ? t - seg * cols : 0;
  const int y = cg / L.hx, g = cg - y * L.hx, z0 = seg * K;
  int li[K];
  float ph[K][2], hb[K][2], cn[K][2], rc[K][2];
#pragma unroll
  for (int j = 0; j < K; j++) {
    const int z = z0 + j;
    const bool inz = act && z < L.d2;
    // a slot past the level or a thread without a column points at the first
    // pair: its reads stay in the level, it stores nothing
    li[j] = inz ? tail_li(L, g, y, z) : tail_li(L, 0, 0, 0);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const int x = 2 * g + ((y + z + c) & 1);
      const bool in = inz && x < L.d0;
      const int i = in ? x + L.d0 * (y + L.d1 * z) : 0;
      const uint32_t code = cl[L.io + i];
      const float b = inner ? bl[L.bo + i] : L.b[i];
      const bool up = in && !(code & (uint32_t)(NC_SOLID | NC_NONE));
      const float2 cr = ct[code & 63u];
      ph[j][c] = up ? sp[c * TL_CS + li[j]] : 0.0f;
      cn[j][c] = up ? cr.x : 0.0f;
      rc[j][c] = up ? cr.y : 0.0f;
      hb[j][c] = up ? L.hh * b : 0.0f;
    }
  }
  const int e = ((y + z0) & 1) ? 1 : -1;  // side of the LDS x neighbour of slot 0, colour 0
  const int nz = act ? (L.d2 - z0 < K ? L.d2 - z0 : K) : 0;  // slots inside the level
  const int zt = li[0] - L.pz, zb = nz == K ? li[K - 1] + L.pz : li[0] - L.pz;
  const int py = L.py;
  for (int it = 0; it < iters; it++) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const float *O = sp + (1 - c) * TL_CS;
      float nb[K][3];
#pragma unroll
      for (int j = 0; j < K; j++) {
        nb[j][0] = O[li[j] + (((j + c) & 1) ? -e : e)];
        nb[j][1] = O[li[j] + py];
        nb[j][2] = O[li[j] - py];
      }
      const float zlo = O[zt], zhi = O[zb];
      float xs[K], qs[K], old[K];
      bool redo = false;
#pragma unroll
      for (int j = 0; j < K; j++) {
        float sum = ph[j][1 - c] + nb[j][0];
        sum += nb[j][1];
        sum += nb[j][2];
        sum += j + 1 < K ? ph[j + 1][1 - c] : zhi;
        sum += j > 0 ? ph[j - 1][1 - c] : zlo;
        xs[j] = sum - hb[j][c];
        const float q0 = xs[j] * rc[j][c];
        const float er = __builtin_fmaf(-q0, cn[j][c], xs[j]);
        qs[j] = __builtin_fmaf(er, rc[j][c], q0);
        old[j] = ph[j][c];
        ph[j][c] = mixf_(old[j], qs[j], omega);
        if (j < nz) sp[c * TL_CS + li[j]] = ph[j][c];
        redo |= div_redo<ICNT>(xs[j], qs[j], rc[j][c]);
      }
      if (redo) {
#pragma unroll
        for (int j = 0; j < K; j++)
          if (div_redo<ICNT>(xs[j], qs[j], rc[j][c])) {
            float x = xs[j];
            asm volatile("" : "+v"(x));
            ph[j][c] = mixf_(old[j], x / cn[j][c], omega);
            if (j < nz) sp[c * TL_CS + li[j]] = ph[j][c];
          }
      }
      __syncthreads();
    }
  }
}

template <int KT, int KC, bool ICNT>
__global__ __launch_bounds__(TL_NT) void k_mg_tail(TailArgs) {
  // the levels are indexed at run time: read where they are (uniform scalar
  // loads from the kernel arguments), a copy of the argument would be indexed
  // in scratch memory
  const TailArgs &a = *(const TailArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  __shared__ __align__(16) float sp[2 * TL_CS];
  __shared__ float bl[TL_INNER];
  __shared__ uint8_t cl[2 * TL_NT * TL_K + TL_INNER];
  __shared__ float2 ct[64 * TL_MAX];
  const int t = threadIdx.x;
  if (t < 64 * a.nl) {
    const uint32_t code = (uint32_t)t & 63u;
    const float c = nc_count(code, a.l[t / 64].wdir);
    ct[t] = make_float2(c, c > 0.0f ? 1.0f / c : 0.0f);
  }
  for (int i = t; i < 2 * TL_CS / 4; i += TL_NT)
    reinterpret_cast<float4 *>(sp)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  uint32_t solid = 0u;  // bit l: level l has a solid cell
  for (int l = 1; l < a.nl; l++) {
    bool sl = false;
    for (int i = t; i < a.l[l].n; i += TL_NT) {
      const uint8_t code = a.l[l].nc[i];
      cl[a.l[l].io + i] = code;
      sl |= (code & NC_SOLID) != 0;
    }
    solid |= __syncthreads_or(sl) ? 1u << l : 0u;
  }
  TailOwn<KT> W;
  {
    // the top level's codes, h^2 b and phi (a solid reads 0 in the sums and keeps its phi in memory)
    const TailLv &T = a.l[0];
    tail_own<KT, false>(T, sp, bl, cl, ct, W);
    float p[KT][2];
#pragma unroll
    for (int j = 0; j < KT; j++) {
      p[j][0] = T.phi[W.gi[j]];
      p[j][1] = T.phi[W.gi[j] + ((W.cd[j] >> 18) & 1u)];
    }
    __syncthreads();  // the zero fill is complete
#pragma unroll
    for (int j = 0; j < KT; j++) {
      const uint32_t o = (W.cd[j] >> 16) & 1u;
      const uint32_t c0 = (W.cd[j] >> (8 * o)) & 0xffu, c1 = (W.cd[j] >> (8 * (o ^ 1u))) & 0xffu;
      if (W.cd[j] & (1u << 17)) {
        sp[(int)o * TL_CS + W.li[j]] = (c0 & NC_SOLID) ? 0.0f : p[j][0];
        cl[T.io + W.gi[j]] = (uint8_t)c0;
      }
      if (W.cd[j] & (1u << 18)) {
        sp[(int)(o ^ 1u) * TL_CS + W.li[j]] = (c1 & NC_SOLID) ? 0.0f : p[j][1];
        cl[T.io + W.gi[j] + 1] = (uint8_t)c1;
      }
    }
    __syncthreads();
  }
  auto smooth = [&](int l) __attribute__((always_inline)) {
    if (l == 0) {
      tail_sweeps<KT, ICNT>(a.l[0], sp, bl, cl, ct, 0, W, 2, 1.0f);
    } else {
      TailOwn<2> I;
      tail_own<2, true>(a.l[l], sp, bl, cl, ct, I);
      tail_sweeps<2, ICNT>(a.l[l], sp, bl, cl, ct, l, I, 2, 1.0f);
    }
  };
  for (int l = 0; l < a.nl - 1; l++) {
    smooth(l);
    if (l == 0) tail_restrict<false>(a.l[0], a.l[1], sp, bl, cl, ct);
    else tail_restrict<true>(a.l[l], a.l[l + 1], sp, bl, cl, ct);
  }
  if constexpr (KC == 0) tail_sweeps<KT, ICNT>(a.l[0], sp, bl, cl, ct, 0, W, a.iters, a.omega);
  else if (a.nl == 1) tail_sor<KC, ICNT, false>(a.l[0], sp, bl, cl, ct, 0, a.iters, a.omega);
  else tail_sor<KC, ICNT, true>(a.l[a.nl - 1], sp, bl, cl, ct, a.nl - 1, a.iters, a.omega);
  for (int l = a.nl - 2; l >= 0; l--) {
    tail_prolong(a.l[l + 1], a.l[l], sp, bl, cl, ct, (solid >> (l + 1)) & 1u);
    smooth(l);
  }
  // phi back to memory: the top level's from the owned pairs (solids and, of
  // a coarsest level alone, the cells its solve skips keep theirs)
  const uint32_t keep = a.nl == 1 ? NC_SOLID | NC_NONE : NC_SOLID;
#pragma unroll
  for (int j = 0; j < KT; j++) {
    const uint32_t o = (W.cd[j] >> 16) & 1u;
    const uint32_t c0 = (W.cd[j] >> (8 * o)) & 0xffu, c1 = (W.cd[j] >> (8 * (o ^ 1u))) & 0xffu;
    if ((W.cd[j] & (1u << 17)) && !(c0 & keep)) a.l[0].phi[W.gi[j]] = sp[(int)o * TL_CS + W.li[j]];
    if ((W.cd[j] & (1u << 18)) && !(c1 & keep)) a.l[0].phi[W.gi[j] + 1] = sp[(int)(o ^ 1u) * TL_CS + W.li[j]];
  }
  for (int l = 1; l < a.nl; l++) {
    const TailLv &L = a.l[l];
    for (int i = t; i < L.n; i += TL_NT) {
      const uint32_t r = fdiv((uint32_t)i, L.dd0), zq = fdiv(r, L.dd1);
      const int x = i - (int)r * L.d0, z = (int)zq, y = (int)r - z * L.d1;
      L.phi[i] = sp[((x + y + z) & 1) * TL_CS + tail_li(L, x >> 1, y, z)];
    }
  }
}

// Pairs per thread of the coarsest solve: the fewest with which the level's
// columns, cut into z segments, fit the workgroup (0: none do).  Fewer pairs
// on more lanes shorten the pass: 0.17 us at K = 1 (8x12x8), 0.35 at 2
// (12x20x12), 0.6 at 4 (14x30x14).  A coarsest level alone takes its sweeps
// over the owned pairs instead where no segments fit (KC = 0 of k_mg_tail).
static int tail_k(const MgLevel &L) {
  const int cols = ((L.d[0] + 1) / 2) * L.d[1];
  for (int k : {1, 2, 4, 8})
    if (cols * ((L.d[2] + k - 1) / k) <= TL_NT) return k;
  return 0;
}
static int tail_floats(const MgLevel &L) {  // LDS words of one colour's pairs with their ghosts
  const int py = (L.d[0] + 1) / 2 + 1, pz = py * (L.d[1] + 1);
  return (L.d[2] + 2) * pz + py + 2;
}
// Whether levels t .. nl - 1 run as one tail.  A level that is smoothed in it
// has at most 4 pairs per thread: each instruction per cell costs one CU what
// 256 share in a launch of its own, and with a 16 k-cell level on top (8 pairs
// per thread) the tail took 94 us against 39 us and six launches of 4.7 us.
static bool tail_fits(const MgLevel *lv, int t, int nl) {
  int64_t words = 0, inner = 0;
  if (nl - t > TL_MAX || (t < nl - 1 && !tail_k(lv[nl - 1]))) return false;
  for (int l = t; l < nl; l++) {
    const MgLevel &L = lv[l];
    if (L.n > 2u * TL_NT * TL_K) return false;
    const int np = ((L.d[0] + 1) / 2) * L.d[1] * L.d[2];
    if (np > TL_NT * (t == nl - 1 ? TL_K : l == t ? TL_TOP : 2)) return false;
    words += tail_floats(L);
    if (l > t) inner += L.n;
  }
  return words <= TL_CS && inner <= TL_INNER;
}
static TailArgs tail_args(const MgLevel *lv, int t, int nl, int iters, float omega) {
  TailArgs a;
  a.nl = nl - t;
  a.iters = iters;
  a.omega = omega;
  int off = 0, io = 0;
  for (int l = t; l < nl; l++) {
    const MgLevel &L = lv[l];
    TailLv &T = a.l[l - t];
    T.d0 = L.d[0]; T.d1 = L.d[1]; T.d2 = L.d[2];
    T.hx = (L.d[0] + 1) / 2;
    T.py = T.hx + 1;
    T.pz = T.py * (L.d[1] + 1);
    T.off = off;
    T.np = T.hx * L.d[1] * L.d[2];
    T.n = (int)L.n;
    T.io = io;
    T.bo = l > t ? io - a.l[0].n : 0;
    off += tail_floats(L);
    io += T.n;
    T.hh = L.hh;
    T.wdir = L.wdir;
    T.dhx = make_fastdiv((uint32_t)T.hx);
    T.dd0 = make_fastdiv((uint32_t)T.d0);
    T.dd1 = make_fastdiv((uint32_t)T.d1);
    T.nc = (const __attribute__((address_space(1))) uint8_t *)L.nc;
    T.phi = (__attribute__((address_space(1))) float *)L.phi;
    T.b = (__attribute__((address_space(1))) float *)L.b;
  }
  return a;
}

template <int KT, int KC>
static void launch_tail(const TailArgs &a, bool icnt, hipStream_t s) {
  if (icnt) k_mg_tail<KT, KC, true><<<1, TL_NT, 0, s>>>(a);
  else k_mg_tail<KT, KC, false><<<1, TL_NT, 0, s>>>(a);
}
static void launch_mg_tail(const MgLevel *lv, int t, int nl, int iters, float omega, hipStream_t s) {
  const TailArgs a = tail_args(lv, t, nl, iters, omega);
  bool icnt = true;
  for (int l = t; l < nl; l++) icnt = icnt && lv[l].wdir == 1.0f;
  const int kc = tail_k(lv[nl - 1]);
  const int kt = a.l[0].np <= 2 * TL_NT ? 2 : a.l[0].np <= 4 * TL_NT ? 4 : TL_K;
  switch (kc) {
    case 0:
      if (kt == 2) launch_tail<2, 0>(a, icnt, s);
      else if (kt == 4) launch_tail<TL_TOP, 0>(a, icnt, s);
      else launch_tail<TL_K, 0>(a, icnt, s);
      break;
    case 1:
      if (kt == 2) launch_tail<2, 1>(a, icnt, s);
      else launch_tail<TL_TOP, 1>(a, icnt, s);
      break;
    case 2:
      if (kt == 2) launch_tail<2, 2>(a, icnt, s);
      else launch_tail<TL_TOP, 2>(a, icnt, s);
      break;
    case 4:
      launch_tail<TL_TOP, 4>(a, icnt, s);
      break;
    default: launch_tail<TL_K, 8>(a, icnt, s); break;
  }
}

void launch_mg_coarse(const MgLevel &L, int iters, float omega, hipStream_t s) {
  LvArgs a = lv_args(L);
  const int ncol = L.d[0] * L.d[1];
  // the column solve takes integer counts, a thread a column and 22 slots
  const bool colz = L.wdir == 1.0f && ncol <= CO_NT && L.d[2] + 1 <= 22;
  // Eight pairs a thread lose to the column solve where there is one, and win
  // over sweep launches where the columns are too long for it: 48x8x24 224 us
  // in sweeps, 175 in the tail; 72x8x24 231, 207; 22x22x22 254, 198.  Too many
  // columns for the tail's solve (thin, wide levels) run its sweeps on the
  // owned pairs, which cost a pass per 2048 pairs: four V-cycles on 1100x2x2
  // 1118 us in sweep launches, 670 so; 200x12x3 1134, 743; 250x9x5 (5625
  // pairs) 1212, 1017; 120x18x6 (6480) 1144, 1287.  Rows below four cells have
  // only the single sweeps beside it: 3x700x2 2564, 840.
  const int tk = tail_k(L), np = ((L.d[0] + 1) / 2) * L.d[1] * L.d[2];
  const bool tail = tk ? !colz || tk < 8 : !colz && (np <= 6 * TL_NT || !sweep2_fits(L));
  if (tail && tail_fits(&L, 0, 1)) {
    launch_mg_tail(&L, 0, 1, iters, omega, s);
    return;
  }
  // one thread per column, whole waves only: a wave without columns would
  // still run every colour pass's arithmetic on the CU
  const int colt = ((ncol + 63) / 64) * 64;
  if (colz && L.d[2] + 1 <= 12) {
    k_mg_coarse_z<12><<<1, colt, 0, s>>>(a, L.b, L.nc, L.phi, iters, omega);
    return;
  }
  if (colz) {
    // waves run on SIMD w % 4.  Per iteration (both colours) a SIMD issues
    // ZJ slots for each of its column waves plus two for each of its waves
    // holding extra cells: take the extra-cell layout when its busiest SIMD
    // issues fewer slots.
    const int zj = L.d[2] + 1 <= 21 ? 21 : 22;
    const int full = (ncol / 64) * 64, zh = (L.d[2] + 1) / 2;
    const int wc = colt / 64, wf = full / 64, we = ((ncol - full) * zh + 63) / 64;
    const int load_col = zj * ((wc + 3) / 4);
    int load_ex = 0;
    for (int sm = 0; sm < 4; sm++) {
      int l = 0;
      for (int w = sm; w < wf; w += 4) l += zj + (w < we ? 2 : 0);
      load_ex = l > load_ex ? l : load_ex;
    }
    const bool ex = full >= 64 && full <= CZ_EX_NT && ncol > full && (ncol - full) * zh <= full && load_ex < load_col;
    if (zj == 21) {
      if (ex)
        k_mg_coarse_z<21, true><<<1, full, 0, s>>>(a, L.b, L.nc, L.phi, iters, omega);
      else
        k_mg_coarse_z<21><<<1, colt, 0, s>>>(a, L.b, L.nc, L.phi, iters, omega);
    } else {
      if (ex)
        k_mg_coarse_z<22, true><<<1, full, 0, s>>>(a, L.b, L.nc, L.phi, iters, omega);
      else
        k_mg_coarse_z<22><<<1, colt, 0, s>>>(a, L.b, L.nc, L.phi, iters, omega);
    }
    return;
  }
  // Two iterations a launch.  22x32x22 (15.5 k cells) 330 us in one workgroup
  // with phi in LDS, 259 now; at one iteration a launch 26x38x26 took 778 us
  // (rows that are no multiple of four), now 260, and 40x60x40 319, now 241.
  // The column solve above takes 165 us for 20x40x20.
  int it = 0;
  if (sweep2_fits(L))
    for (; it + 4 <= iters; it += 4) {
      launch_mg_sweep2(L, nullptr, L.phi, L.tmp, omega, s);
      launch_mg_sweep2(L, nullptr, L.tmp, L.phi, omega, s);
    }
  for (; it < iters; it += 2) {
    launch_mg_sweep(L, L.phi, L.tmp, omega, s, false);
    launch_mg_sweep(L, L.tmp, L.phi, omega, s, false);
  }
}

// ---------------------------------------------------------------- resid
// Per-block FP64 sums of r^2 and b^2 over fluid cells (mg.wgsl:134-158).
__global__ __launch_bounds__(NT) void k_mg_resid(LvArgs a, FastDiv d0, const float *__restrict__ p,
                                                  const float *__restrict__ b, const uint8_t *__restrict__ f,
                                                  double *__restrict__ part) {
  uint32_t i = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * NT + threadIdx.x;
  double r2 = 0.0, b2 = 0.0;
  if (i < a.n && f[i] != 1) {
    uint32_t r = fdiv(i, d0);
    int x = (int)(i - r * (uint32_t)a.d0);
    uint32_t zq = fdiv(r, a.dny);
    int y = (int)(r - zq * (uint32_t)a.d1), z = (int)zq;
    float rr = resid_at(a, p, b, f, x, y, z);
    float bb = b[i];
    r2 = (double)rr * (double)rr;
    b2 = (double)bb * (double)bb;
  }
  __shared__ double sh[NT / 64];
  double s1 = block_sum<NT>(r2, sh);
  double s2 = block_sum<NT>(b2, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x * 2] = s1;
    part[blockIdx.x * 2 + 1] = s2;
  }
}
int mg_resid_blocks(const MgLevel &L) { return nblocks(L.n); }
void launch_mg_resid(const MgLevel &L, StatParts *st, hipStream_t s) {
  LvArgs a = lv_args(L);
  k_mg_resid<<<nblocks(L.n), NT, 0, s>>>(a, make_fastdiv((uint32_t)L.d[0]), L.phi, L.b, L.f, st->resid);
}

// ---------------------------------------------------------------- V-cycle
void enqueue_vcycle(const MgLevel *lv, int nl, int coarse_iters, hipStream_t s, bool from_zero, VPart part) {
  // the levels from t on run in one launch where they fit
  int t = nl - 1;
  while (t > 0 && tail_fits(lv, t - 1, nl)) t--;
  if (from_zero && t == 0 && part != VPart::Rest) launch_zero32(lv[0].n, lv[0].phi, s);  // the tail reads phi
  // smoothing: two sweeps phi -> tmp -> phi, or both in one launch, phi ->
  // tmp before the coarser level and tmp -> phi after it
  for (int l = 0; l < t; l++) {
    MgLevel L = lv[l];
    const float *pin = (l > 0 || from_zero) ? nullptr : L.phi;  // a restricted level starts from 0
    const bool two = sweep2_fits(L);
    if (l > 0 || part != VPart::Rest) {
      if (two) {
        launch_mg_sweep2(L, nullptr, pin, L.tmp, 1.0f, s);
      } else {
        launch_mg_sweep(L, pin, L.tmp, 1.0f, s, l == 0);
        launch_mg_sweep(L, L.tmp, L.phi, 1.0f, s, l == 0);
      }
    }
    if (part == VPart::Head) return;
    if (two) L.phi = L.tmp;
    launch_mg_restrict(L, lv[l + 1], s);
  }
  if (part == VPart::Head) return;
  if (t < nl - 1) launch_mg_tail(lv, t, nl, coarse_iters, 1.6f, s);
  else launch_mg_coarse(lv[t], coarse_iters, 1.6f, s);
  for (int l = t - 1; l >= 0; l--) {
    MgLevel L = lv[l];
    if (sweep2_fits(L)) {
      const bool fuse = L.n <= S2_PROLONG_MAX;
      if (!fuse) {
        MgLevel T = L;
        T.phi = T.tmp;
        launch_mg_prolong(lv[l + 1], T, s);
      }
      launch_mg_sweep2(L, fuse ? &lv[l + 1] : nullptr, L.tmp, L.phi, 1.0f, s);
    } else {
      launch_mg_prolong(lv[l + 1], L, s);
      launch_mg_sweep(L, L.phi, L.tmp, 1.0f, s, l == 0);
      launch_mg_sweep(L, L.tmp, L.phi, 1.0f, s, l == 0);
    }
  }
}

}  // namespace pyro
